"""128x128 FP8 tiles of aligned 16-bit matrices whose rows begin inside a 128-byte line, and of short lists: the any-alignment
kernel's share of them, around the lines where the fast kernel takes over."""

import pytest
import torch

from miles_amd import launch
from miles_amd.kernels.quant.fp8_blockwise import fp8_blockwise_cast
from tests.test_gpu_any_alignment_kernels import _matrix, _one_nan, _quantizers
from tests.test_gpu_fp32_kernels import DEV, _assert_same, oracle  # noqa: F401

pytestmark = pytest.mark.gpu


def _bytes_equal(got, want, what):
    for a, b in zip(got, want):
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), what


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("specials", [False, True])
@pytest.mark.parametrize("shapes", [
    [(1, 8), (127, 72), (129, 136), (128, 128), (300, 264)],
    [(1024, 1280)],                                  # 80 tiles: the last short list
    [(1152, 1152)],
    [(2048, 2048)],
    [(2049, 2048), (1, 8)],
    [(2049, 2056)],                                  # 289 tiles, rows that share lines
    [(16255, 1032)],                                 # 1143 of them
    [(16255, 1032), (127, 1032)],                    # 1152
    [(21759, 1056)],                                 # 1530, at half a line
    [(21760, 1056), (5, 1056)],                      # 1539
    [(1025, 1032)] * 4 + [(1024, 2048)] * 2,
    [(4000, 1032)] * 4 + [(1024, 2048)] * 8,         # mostly those, and mostly the others
    [(4000, 1032)] * 2 + [(1024, 2048)] * 8,
    [(4000, 1032)] * 2 + [(4000, 1056)] * 3,
])
def test_lists_against_oracle(oracle, shapes, dtype, specials):  # noqa: F811
    hosts = [_matrix(s, dtype, 700 + i, specials) for i, s in enumerate(shapes)]
    for run, ref, name in _quantizers(oracle):
        with launch.deferred():
            outs = [run(h.to(DEV)) for h in hosts]
        for host, (q, s) in zip(hosts, outs):
            q_o, s_o = ref(host)
            _assert_same(s.nan_to_num(nan=77.0), s_o.nan_to_num(nan=77.0), f"{name} scales {tuple(host.shape)}")
            _assert_same(_one_nan(q), _one_nan(q_o), f"{name} codes {tuple(host.shape)}")


def test_windows_and_nan_codes(oracle):  # noqa: F811
    """A window that starts eight elements into its lines gives what its copy gives, to the sign of a NaN's code and the
    payload of its scale (a list of one tile row and one of many: both kernels)."""
    wide = torch.randn(4096, 4096, device=DEV).bfloat16()
    wide[130, 300], wide[131, 301] = float("nan"), -float("nan")
    wide[3, 2000], wide[260, 2000], wide[4000, 9] = float("inf"), -float("inf"), float("nan")
    wide[256:384, 1024:1152] = 0
    for window in (wide[:, 8:2056], wide[:, 64:3000], wide[128:1000, 16:1040]):
        for run, _, name in _quantizers(oracle):
            whole = run(window)
            _bytes_equal(run(window.contiguous()), whole, name)
            for r in range(0, window.shape[0], 128):        # bands of a tile row: short lists
                q, s = run(window[r:r + 128])
                _bytes_equal((q, s), (whole[0][r:r + 128], whole[1][r // 128:r // 128 + 1]), f"{name} row {r}")


@pytest.mark.parametrize("n, rows, cols", [(70, 512, 1032), (70, 384, 776), (66, 130, 264)])
def test_long_lists_over_a_table(oracle, n, rows, cols):  # noqa: F811
    x = torch.randn(n, rows, cols, device=DEV).bfloat16()
    x[1, 0, 0] = float("nan")
    for run, _, name in _quantizers(oracle):
        with launch.recording() as batch:
            got = [run(t) for t in x]
        batch.freeze()
        batch.run()
        for i in (0, 1, n // 2, n - 1):
            _bytes_equal(run(x[i]), got[i], f"{name} {i}")


def test_row_blocks_with_rows_that_share_lines():
    x = torch.randn(3, 256, 72, device=DEV).bfloat16()
    view = torch.cat([x, x], 1)[:, :256]                    # blocks of 256 rows, 512 apart
    q, s = fp8_blockwise_cast(view)
    _bytes_equal((q.reshape(768, 72), s), fp8_blockwise_cast(x.reshape(768, 72)), "row blocks")
