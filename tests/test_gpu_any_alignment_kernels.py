"""The FP8 kernels for any row alignment and for fp32 against the oracle: widths around a segment and a tile, odd strides,
tensors off a 16-byte boundary, special values, grouped and recorded job lists."""

import pytest
import torch

from tests.test_gpu_fp32_kernels import DEV, _assert_same, fp32_case, oracle  # noqa: F401

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16, torch.float32]
# narrower than a segment, a segment and its neighbours, the same behind a whole tile, several tiles, one row, tall; no
# width a multiple of eight, which the kernel for aligned rows would take
TILE_SHAPES = [(3, 1), (130, 7), (5, 9), (129, 121), (128, 127), (127, 129), (200, 135), (257, 137), (1, 300), (1545, 515), (130, 263)]


def _matrix(shape, dtype, seed, specials):
    x = fp32_case(shape, seed, specials)
    if dtype == torch.float16:
        x = x * 2.0**-12       # keeps the plain values inside fp16's range
    x = x.to(dtype)
    if specials and shape[0] > 128 and shape[1] > 128:
        x[128:, 128:] = 0      # an all-zero tile, and one of subnormals
        x[:128, 128:] = torch.finfo(dtype).smallest_normal / 4
    return x


def _one_nan(codes):
    """The sign of a NaN product or quotient is nowhere specified (all-zero tiles, whose code 0xFF is, have tests elsewhere)."""
    c = codes.cpu().view(torch.uint8)
    return torch.where(c & 0x7F == 0x7F, torch.full_like(c, 0x7F), c)


def _quantizers(oracle):  # noqa: F811
    from miles_amd.kernels.quant.fp8_blockwise import fp8_blockwise_cast, per_block_cast_to_fp8
    from miles_amd.tools.convert_hf_to_fp8 import block_fp8

    return [(lambda w: block_fp8(w, [128, 128]), lambda w: oracle.block_fp8(w, (128, 128)), "block"),
            (fp8_blockwise_cast, oracle.fp8_blockwise_cast, "cast"), (per_block_cast_to_fp8, oracle.per_block_cast_to_fp8, "pow2")]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("specials", [False, True])
def test_tiles_of_any_width(oracle, dtype, specials):  # noqa: F811
    """One list per quantizer; every other matrix is a window of a wider one that starts at an odd element."""
    from miles_amd import launch

    hosts, views = [], []
    for i, shape in enumerate(TILE_SHAPES):
        wide = _matrix((shape[0], shape[1] + 5), dtype, 100 + i, specials).to(DEV)
        views.append(wide[:, 3:3 + shape[1]] if i % 2 else wide[:, 5:].contiguous())
        hosts.append(views[-1].cpu().contiguous())
    for quantize, reference, what in _quantizers(oracle):
        with launch.recording() as batch:
            outs = [quantize(v) for v in views]
        for rep in range(2):
            batch.run()
            torch.cuda.synchronize()
            for (q, s), h in zip(outs, hosts):
                q_o, s_o = reference(h)
                _assert_same(s, s_o, f"{what} scales {tuple(h.shape)}, run {rep}")
                _assert_same(_one_nan(q), _one_nan(q_o), f"{what} codes {tuple(h.shape)}, run {rep}")
                q.view(torch.uint8).fill_(0x5A), s.fill_(-1.0)


def test_tile_outputs_stay_inside_their_rows(oracle):  # noqa: F811
    """Codes written into the middle of a larger buffer leave what surrounds them alone."""
    from miles_amd import _lib, launch

    w = _matrix((131, 141), torch.bfloat16, 7, False)
    d, room = w.to(DEV), torch.full((64 + w.numel() + 64,), 0x5A, dtype=torch.uint8, device=DEV)
    s = torch.empty(2, 2, device=DEV)
    launch.submit(_lib.JOB_FP8_BLOCKWISE_CAST, d, room[61:], s, None, None, 131, 141, 141, 128, 128)
    q_o, _ = oracle.fp8_blockwise_cast(w)
    assert torch.equal(room[61:61 + w.numel()].cpu().view(131, 141), q_o.view(torch.uint8))
    assert (room[:61] == 0x5A).all() and (room[61 + w.numel():] == 0x5A).all()


def near_code_boundaries(rows, cols, amax, g):
    """fp32 values whose quotient by amax / 448 lies on a midpoint between two codes or a few ulp beside one."""
    code = torch.randint(0, 126, (rows, cols), generator=g).to(torch.uint8)
    mid = (code.view(torch.float8_e4m3fn).double() + (code + 1).view(torch.float8_e4m3fn).double()) / 2
    x = (mid * (float(amax) / 448)).float()
    x = (x.view(torch.int32) + torch.randint(-2, 3, x.shape, generator=g, dtype=torch.int32)).view(torch.float32).clamp(0.0, float(amax))
    x = torch.where(torch.rand(x.shape, generator=g) < 0.5, -x, x)
    x[0, 0] = amax
    return x


def test_division_sequence_of_fp32_tiles(oracle):  # noqa: F811
    """block_fp8 divides: a divisor of its own for every tile, quotients at the rounding boundaries of the codes."""
    from miles_amd.tools.convert_hf_to_fp8 import block_fp8

    g = torch.Generator().manual_seed(3)
    w = torch.empty(128 * 12, 128 * 12)
    for i in range(0, len(w), 128):
        for j in range(0, len(w), 128):
            amax = (torch.rand((), generator=g) + 0.5) * 2.0 ** float(torch.randint(-88, 90, (), generator=g))
            w[i:i + 128, j:j + 128] = near_code_boundaries(128, 128, amax, g)
    q, s = block_fp8(w.to(DEV), [128, 128])
    q_o, s_o = oracle.block_fp8(w, (128, 128))
    _assert_same(s, s_o, "scales")
    _assert_same(q, q_o, "codes")
