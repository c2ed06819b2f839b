"""fp32 128x128 tiles, whose segments are four columns wide, against the oracle: widths around a segment and around a tile,
heights around the sixteen rows that a pass covers, rows of whole lines and rows at any element."""

import pytest
import torch

from miles_amd import launch
from tests.test_gpu_any_alignment_kernels import _matrix, _one_nan, _quantizers
from tests.test_gpu_fp32_kernels import DEV, _assert_same, oracle  # noqa: F401

pytestmark = pytest.mark.gpu
WIDTHS = [2, 3, 4, 5, 6, 8, 24, 124, 126, 128, 130, 131, 132, 133, 136, 152, 256, 264]


@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("specials", [False, True])
def test_fp32_tile_widths(oracle, specials, offset):  # noqa: F811
    hosts, views = [], []
    for i, cols in enumerate(WIDTHS):
        rows = (1, 15, 16, 17, 127, 129, 145)[i % 7]
        wide = _matrix((rows, (cols + 31) // 32 * 32 + 32), torch.float32, 300 + i, specials).to(DEV)
        views.append(wide[:, offset:offset + cols])
        hosts.append(views[-1].cpu().contiguous())
    for run, ref, name in _quantizers(oracle):
        with launch.deferred():
            outs = [run(v) for v in views]
        for host, (q, s) in zip(hosts, outs):
            q_o, s_o = ref(host)
            _assert_same(s, s_o, f"{name} scales {tuple(host.shape)}")
            _assert_same(_one_nan(q), _one_nan(q_o), f"{name} codes {tuple(host.shape)}")
