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


# shorter than a unit of either size, a unit and its neighbours, the register limits of the row kernels (256, 1024, 2048 and
# 4096 units of four or eight elements) and past them
ROW_WIDTHS = [1, 3, 4, 5, 7, 8, 9, 255, 1021, 1027, 2047, 2049, 4093, 4099, 8191, 8195, 16381, 16387, 32767, 32771]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("specials", [False, True])
@pytest.mark.parametrize("strategy", ["channel", "tensor"])
def test_scaled_rows_of_any_width(oracle, dtype, specials, strategy):  # noqa: F811
    from miles_amd.tools.convert_hf_to_fp8 import quant_fp8

    reference = oracle.channel_fp8 if strategy == "channel" else oracle.tensor_fp8
    for i, cols in enumerate(ROW_WIDTHS):
        wide = _matrix((5 + i % 3, cols + 3), dtype, 300 + i, specials).to(DEV)
        wide[1] = 0
        views = [wide[:, 3:].contiguous(), wide[:, 1:1 + cols]]      # contiguous rows; rows of a wider matrix off every boundary
        flat = torch.empty(views[0].numel() + 1, dtype=dtype, device=DEV)
        flat[1:] = views[0].reshape(-1)
        views.append(flat[1:].view(views[0].shape))                  # contiguous, one element off the allocation's start
        for v in views:
            q, s = quant_fp8(v, strategy)
            q_o, s_o = reference(v.cpu().contiguous())
            what = f"{strategy} {dtype} {tuple(v.shape)} stride {v.stride(0)}"
            _assert_same(_one_nan(s.view(torch.uint8)) if specials else s, _one_nan(s_o.view(torch.uint8)) if specials else s_o, what + " scales")
            _assert_same(_one_nan(q), _one_nan(q_o), what + " codes")


def test_tensor_scale_of_many_workgroups(oracle):  # noqa: F811
    """Several trips of the amax pass, and the maximum in the last, moved-back unit."""
    from miles_amd.tools.convert_hf_to_fp8 import tensor_fp8

    for dtype in DTYPES:
        w = _matrix((1021, 2053), dtype, 400, False)
        w[-1, -1] = w.abs().max() * 2
        q, s = tensor_fp8(w.to(DEV))
        q_o, s_o = oracle.tensor_fp8(w)
        _assert_same(s, s_o, f"{dtype} scale")
        _assert_same(q, q_o, f"{dtype} codes")


@pytest.mark.parametrize("shape,dtype", [((63, 1027), torch.float32), ((64, 1027), torch.float32), ((65, 515), torch.bfloat16),
                                         ((64, 1), torch.float16), ((4097, 16387), torch.bfloat16)])
def test_tensor_scale_of_many_partial_maxima(oracle, shape, dtype):  # noqa: F811
    """The rows from which the amax pass has 64 words, and the size from which it has 2048 workgroups; the maximum comes last."""
    from miles_amd.tools.convert_hf_to_fp8 import tensor_fp8

    w = torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(7), device=DEV).to(dtype)
    w[-1, -1] = -2 * w.abs().max()
    q, s = tensor_fp8(w)
    q_o, s_o = oracle.tensor_fp8(w.cpu())
    _assert_same(s, s_o, f"{shape} {dtype} scale")
    _assert_same(q, q_o, f"{shape} {dtype} codes")


@pytest.mark.parametrize("block", [8, 32, 128])
def test_dequantize_rows_of_any_width(oracle, block):  # noqa: F811
    """One list of matrices from one unit to several tiles wide, codes at any byte, NaN codes and non-finite scales."""
    from miles_amd import launch
    from miles_amd.tools.fp8_cast_bf16 import weight_dequant

    g = torch.Generator().manual_seed(block)
    cases = []
    for cols in [1, 7, 8, 9, 15, 17, 121, 127, 129, 135, 263, 1000, 2051]:
        rows = 3 * block // 2 + 1
        codes = torch.randint(0, 256, (rows, cols), generator=g, dtype=torch.uint8)
        if cols % 2:
            codes = torch.where(codes & 0x7F == 0x7F, codes & 0x3F, codes)
        s = torch.exp2(torch.randint(-30, 30, (-(-rows // block), -(-cols // block)), generator=g).float()) * 1.37
        if cols > 128:
            s[0, 0], s[-1, -1] = float("inf"), float("nan")
        flat = torch.zeros(codes.numel() + 3, dtype=torch.uint8, device=DEV)
        flat[3:] = codes.reshape(-1).to(DEV)
        cases.append((codes.view(torch.float8_e4m3fn), s, flat[3:].view(rows, cols).view(torch.float8_e4m3fn)))
    with launch.deferred():
        outs = [weight_dequant(x, s.to(DEV), block) for _codes, s, x in cases]
    for (codes, s, _x), y in zip(cases, outs):
        _assert_same(y, oracle.weight_dequant(codes, s, block), f"block {block} {tuple(codes.shape)}")


@pytest.mark.parametrize("per_channel", [1, 0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_scales_below_the_normal_range(oracle, dtype, per_channel):  # noqa: F811
    """With a floor of zero (the entry point takes any) a row of subnormals has a scale that is rounded to a few units in the
    last place, or to zero: quotients lie far above 448 and are clamped."""
    from miles_amd import _lib

    w = torch.zeros(8, 15, dtype=torch.float32)
    for r, units in enumerate([1, 223, 225, 300, 650, 671, 1000, 5000]):
        w[r] = torch.linspace(-1, 1, 15) * units * 2.0**-149
    if dtype == torch.bfloat16:
        w = w * 2.0**16
    w = w.to(dtype)
    for host in [w] if per_channel else [w[i:i + 1].contiguous() for i in range(8)]:
        d = host.to(DEV)
        q, s = torch.empty(host.shape, dtype=torch.uint8, device=DEV), torch.empty(len(host), device=DEV)
        ws = torch.empty(8, dtype=torch.int32, device=DEV)
        _lib.check(_lib.load().mq_fp8_scaled_quant(d.data_ptr(), _lib.DTYPE_CODE[dtype], 15, q.data_ptr(), s.data_ptr(), ws.data_ptr(),
                                                   len(host), 15, per_channel, 0.0, _lib.stream_ptr(d.device)))
        amax = host.float().abs().amax(1, keepdim=True)
        scale = amax / 448
        want = host.float() / scale
        want = want.to(dtype).float() if not per_channel else want
        want = want.clamp(-448, 448).to(torch.float8_e4m3fn)
        _assert_same(s, scale.reshape(-1), "scales")
        _assert_same(_one_nan(q.view(torch.float8_e4m3fn)), _one_nan(want), "codes")
