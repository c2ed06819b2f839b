"""FP8 with a scale for each row, around the lines where a list's rows change from 64 lanes to 256 and back."""

import pytest
import torch

from miles_amd import launch
from miles_amd.tools.convert_hf_to_fp8 import channel_fp8
from tests.test_gpu_any_alignment_kernels import _matrix, _one_nan
from tests.test_gpu_fp32_kernels import DEV, _assert_same, oracle  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows, units", [
    ((680, 684, 684), (128, 129, 200)),         # 2048 rows in one launch, the widest of 200 units
    ((680, 684, 685), (128, 129, 256)),         # 2049
    ((2048,), (129,)),
    ((2048,), (256,)),
    ((2049,), (129,)),
    ((2049,), (256,)),
    ((680, 684, 684), (1, 127, 128)),
    ((8, 7), (1, 128)),
    ((8, 7), (129, 256)),
    ((4001, 4190), (257, 384)),                 # 8191 rows of 257 to 384 units
    ((4001, 4191), (257, 384)),                 # 8192
    ((4001, 4192), (257, 320)),                 # 8193: a second round, of 16-bit rows up to 320 units
    ((4001, 4192), (257, 321)),
    ((4001, 4447), (257, 384)),                 # 8448
    ((4001, 4448), (257, 384)),
    ((4097, 4097), (257, 385)),
])
def test_lists_against_oracle(oracle, rows, units, dtype, offset):  # noqa: F811
    e = 4 if dtype == torch.float32 else 8
    hosts, views = [], []
    for i, (r, u) in enumerate(zip(rows, units)):
        cols = u * e - (offset if u > 1 else 0)
        wide = _matrix((r, cols + offset), dtype, 800 + i, r < 10)
        if r < 10:
            wide[0] = 0
        views.append(wide.to(DEV)[:, offset:])
        hosts.append(wide[:, offset:])
    with launch.deferred():
        outs = [channel_fp8(v) for v in views]
    for host, (q, s) in zip(hosts, outs):
        q_o, s_o = oracle.channel_fp8(host)
        _assert_same(s.nan_to_num(nan=77.0), s_o.nan_to_num(nan=77.0), f"scales {tuple(host.shape)}")
        _assert_same(_one_nan(q), _one_nan(q_o), f"codes {tuple(host.shape)}")
