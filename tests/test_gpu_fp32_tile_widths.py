"""fp32 128x128 tiles, whose segments are four columns wide, against the oracle: widths around a segment and around a tile,
heights around the sixteen rows that a pass covers, rows of whole lines and rows at any element."""

import pytest
import torch

from miles_amd import launch
from miles_amd.kernels.quant.fp8_blockwise import fp8_blockwise_cast
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


# around the lists from which on the cast takes two or three workgroups per compute unit, unaligned rows and whole lines
@pytest.mark.parametrize("rows, cols, tensors", [
    (4095, 8191, 2), (3200, 8191, 1), (3072, 8191, 1), (65536, 515, 2), (65536, 509, 2), (8192, 32768, 1), (8064, 32768, 1),
    (32769, 131, 13), (32769, 131, 4), (32769, 131, 2), (16385, 195, 17), (65536, 129, 2), (262144, 125, 2)])
def test_long_lists_are_their_bands(rows, cols, tensors):
    """Each tile is by itself: a long list gives what its bands of 1024 rows give in calls of their own, infinities and NaN
    in some tiles included."""
    weights = []
    for i in range(tensors):
        g = torch.Generator(device=DEV).manual_seed(i)
        w = torch.randn(rows, cols, generator=g, device=DEV)
        w[5 + 128 * i, 7] = float("inf")
        w[rows - 1, cols - 1] = float("nan")
        w[640:768, 128:256] = 0.0
        weights.append(w)
    with launch.deferred():
        whole = [fp8_blockwise_cast(w) for w in weights]
    for w, (q, s) in zip(weights, whole):
        for r in range(0, rows, 1024):
            q1, s1 = fp8_blockwise_cast(w[r:r + 1024])
            assert torch.equal(q[r:r + 1024].view(torch.uint8), q1.view(torch.uint8)), f"codes from row {r}"
            assert torch.equal(s[r // 128:r // 128 + 8].view(torch.int32), s1.view(torch.int32)), f"scales from row {r}"
