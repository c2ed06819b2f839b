"""fp32 instances of the tuned kernels against the oracle: sizes at the edges of a workgroup, special values, grouped
and recorded job lists."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def oracle():
    from oracle import mq_oracle as O

    return O


def _bits(t):
    t = t.cpu().contiguous()
    return t.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])


def _assert_same(got, want, what):
    g, w = _bits(got), _bits(want)
    assert g.shape == w.shape, f"{what}: shape {tuple(g.shape)} vs {tuple(w.shape)}"
    if not torch.equal(g, w):
        bad = (g != w).nonzero()
        i = tuple(bad[0].tolist())
        raise AssertionError(f"{what}: {bad.shape[0]} of {g.numel()} differ; first at {i}: got {g[i].item()} want {w[i].item()}")


def fp32_case(shape, seed, specials=False):
    """Values over forty binades with all 24 significant bits in use; optionally the format's extremes, subnormals,
    signed zeros, infinities and NaN strewn over them, and a row of zeros."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g) * torch.exp2(torch.randint(-20, 21, (shape[0], 1), generator=g).float())
    if specials:
        values = torch.tensor([0.0, -0.0, 1e-45, -1e-40, 1.1754944e-38, 3.4028235e38, -3.4028235e38, float("inf"),
                               -float("inf"), float("nan"), 448.0, 464.0, 2.0**-9, 6.0, 5.0000005, 2.5])
        at = torch.rand(shape, generator=g) < 0.004
        x = torch.where(at, values[torch.randint(0, len(values), shape, generator=g)], x)
        if shape[0] > 2:
            x[2] = 0
    return x


# one group, ragged last workgroups (a workgroup covers 2048 elements), several of them
FLAT_SHAPES = [(1, 32), (5, 96), (1, 2048), (1, 2080), (129, 2016), (3, 12288), (513, 1024)]


@pytest.mark.parametrize("shape", FLAT_SHAPES)
@pytest.mark.parametrize("specials", [False, True])
def test_mxfp8_fp32(oracle, shape, specials):
    from miles_amd.utils.mxfp8 import mxfp8_quantize

    w = fp32_case(shape, 10 + shape[1], specials)
    q, s = mxfp8_quantize(w.to(DEV))
    q_o, s_o = oracle.mxfp8_quantize(w)
    _assert_same(s, s_o, "scales")
    _assert_same(q, q_o, "codes")


def test_mxfp8_fp32_in_one_list_with_16_bit_tensors(oracle):
    """A recorded list of seventy tensors (more than the kernel arguments of a launch hold), run twice."""
    from miles_amd import launch
    from miles_amd.utils.mxfp8 import mxfp8_quantize

    tensors = [fp32_case((33, 160), 50 + i) for i in range(72)]
    tensors[5], tensors[6] = tensors[5].bfloat16(), tensors[6].half()
    dev = [t.to(DEV) for t in tensors]
    with launch.recording() as batch:
        outs = [mxfp8_quantize(t) for t in dev]
    batch.freeze()
    for rep in range(2):
        batch.run()
        torch.cuda.synchronize()
        for i, t in enumerate(tensors):
            for got, want, what in zip(outs[i], oracle.mxfp8_quantize(t), ("codes", "scales")):
                _assert_same(got, want, f"tensor {i} ({t.dtype}) {what}, run {rep}")
        for o in outs:
            for t in o:
                t.view(torch.uint8).fill_(0x5A)


# the largest magnitudes of a group decide how its codes are computed: near the top of the range, at the limit of the fused
# form (2^90), and an overflowing sevenfold scale
INT4_TOPS = [3.4028235e38, -3.4e38, 2.0**90, 2.0**90 * (1 + 2.0**-23), 1e-5, 7e-5, 2.0**-120]


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("shape", [(1, 128), (5, 384), (1, 2048), (3, 2176), (129, 2048), (513, 1024)])
@pytest.mark.parametrize("specials", [False, True])
def test_int4_pack_fp32(oracle, shape, group, specials):
    from miles_amd.kernels.quant.int4_fake import pack_layer

    w = fp32_case(shape, 20 + shape[1] + group)
    # quotients at and next to a half: multiples of half a scale of 1 (group maximum 7), and their neighbours
    w[0, :32] = torch.arange(-16, 16) * 0.5
    w[0, 0] = 7.0
    w[0, 1:32:3] = torch.nextafter(w[0, 1:32:3], torch.tensor(100.0))
    if specials:
        at = torch.rand(shape, generator=torch.Generator().manual_seed(shape[1])) < 0.002
        values = torch.tensor(INT4_TOPS + [0.0, -0.0, 1e-45, float("inf"), -float("inf")])
        w = torch.where(at, values[torch.randint(0, len(values), shape, generator=torch.Generator().manual_seed(group))], w)
        w[-1, -group:] = 0
    q, s, _ = pack_layer(w.to(DEV), group)
    q_o, s_o, _ = oracle.pack_layer(w, group)
    _assert_same(s, s_o, "scales")
    _assert_same(q, q_o, "codes")


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("shape", [(8, 128), (8, 384), (16, 4224), (136, 1024)])
@pytest.mark.parametrize("specials", [False, True])
def test_int4_pack_asym_fp32(oracle, shape, group, specials):
    from miles_amd.kernels.quant.int4_fake import pack_layer

    w = fp32_case(shape, 25 + shape[1] + group)
    # quotients at and next to a half: multiples of half a scale of 1 (extrema -7 and 8), and their neighbours
    w[0, :32] = torch.arange(-14, 18) * 0.5
    w[0, 1:31:3] = torch.nextafter(w[0, 1:31:3], torch.tensor(100.0))
    if specials:
        w[1] += 1e4 * w[1].abs().max()        # minima far above zero and far below it: the zero point is clamped, codes carry
        w[2] -= 1e4 * w[2].abs().max()
        at = torch.rand(shape, generator=torch.Generator().manual_seed(shape[1])) < 0.002
        values = torch.tensor(INT4_TOPS + [0.0, -0.0, 1e-45])
        w = torch.where(at, values[torch.randint(0, len(values), shape, generator=torch.Generator().manual_seed(group))], w)
        w[-1, -group:] = 0
        w[-2, -group:] = 3.25
    for got, want, what in zip(pack_layer(w.to(DEV), group, False), oracle.pack_layer(w, group, False), ("codes", "scales", "zero points")):
        _assert_same(got, want, what)


@pytest.mark.parametrize("shape", FLAT_SHAPES)
@pytest.mark.parametrize("specials", [False, True])
def test_mxfp4_fp32(oracle, shape, specials):
    from miles_amd.utils.mxfp4 import quantize_mxfp4

    w = fp32_case(shape, 30 + shape[1], specials).nan_to_num(nan=1.0, posinf=float("inf"), neginf=-float("inf"))
    # (the reference's scale byte for a NaN is an undefined float-to-integer conversion)
    # every bound between two codes at a scale of 1 (group maximum 6), and its neighbours on both sides
    bounds = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0])
    row = torch.cat([bounds, torch.nextafter(bounds, torch.tensor(9.0)), torch.nextafter(bounds, torch.tensor(0.0)), -bounds])
    w[0, :28], w[0, 28:32] = row, torch.tensor([6.0, -0.0, 0.0, -6.0])
    q, s = quantize_mxfp4(w.to(DEV), 32)
    q_o, s_o = oracle.quantize_mxfp4(w, 32)
    _assert_same(s, s_o, "scales")
    _assert_same(q, q_o, "codes")


@pytest.mark.parametrize("shape", [(1, 16), (5, 48), (1, 2048), (3, 4112), (129, 2032), (513, 1024)])
@pytest.mark.parametrize("mode", [None, "MAE", "MSE", "FP16"])
def test_nvfp4_fp32(oracle, monkeypatch, shape, mode):
    from miles_amd import _lib
    from miles_amd.utils.nvfp4 import nvfp4_quantize_1d

    e4m3_max, flags = 448, 0
    if mode is not None:
        monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights")
        monkeypatch.setenv("NVTE_NVFP4_4OVER6_ERR_MODE", "MSE" if mode == "MSE" else "MAE")
        monkeypatch.setenv("NVTE_NVFP4_4OVER6_ERR_USE_FAST_MATH", "1" if mode == "FP16" else "0")
        e4m3_max = 256
        flags = _lib.NVFP4_4OVER6 | (_lib.NVFP4_ERR_MSE if mode == "MSE" else 0) | (_lib.NVFP4_ERR_FP16 if mode == "FP16" else 0)
    for case in range(3):
        w = fp32_case(shape, 40 + shape[1] + case) * torch.logspace(0, -2, shape[1])
        if case == 1:
            w[:, : shape[1] // 16 // 2 * 16] = 0          # blocks of zeros
        if case == 2:
            w = torch.full(shape, 3e38) * torch.sign(w)   # an amax outside the range of the fast divisions
        q, s, g = nvfp4_quantize_1d(w.to(DEV))
        q_o, s_o, g_o = oracle.nvfp4_quantize_1d(w, e4m3_max=e4m3_max, flags=flags)
        _assert_same(g.reshape(1), torch.as_tensor(g_o).reshape(1).float(), "global scale")
        _assert_same(s, s_o, "scales")
        _assert_same(q, q_o, "codes")


@pytest.mark.parametrize("shape", [(1, 32), (5, 96), (1, 1024), (1, 1056), (129, 2016)])
@pytest.mark.parametrize("kind", ["fp8", "fp4", "kv"])
def test_fake_quant_fp32(oracle, shape, kind):
    """A workgroup covers 1024 elements, a lane four."""
    from miles_amd.kernels.quant import fake_quant as fq

    forward = {"fp8": fq.fake_quant_fp8_forward, "fp4": fq.fake_quant_fp4_forward, "kv": fq.fake_quant_compressed_kv_forward}[kind]
    w = fp32_case(shape, 70 + shape[1])
    w[0, :6] = torch.tensor([0.0, -0.0, 1e-45, -1e-45, 3e38, -1e-30])
    _assert_same(forward(w.to(DEV)), oracle.fake_quant(w, {"kv": "compressed_kv"}.get(kind, kind)), kind)


@pytest.mark.parametrize("shape", [(1, 128), (5, 384), (1, 1152), (129, 2048)])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("sym", [True, False])
def test_fake_int4_fp32(oracle, shape, group, sym):
    from miles_amd.kernels.quant.int4_fake import fake_int4_quant_cuda

    w = fp32_case(shape, 80 + shape[1] + group)
    w[-1, :group] = 0
    w[0, 1:5] = float("nan")           # a lane of NaNs, skipped by the extrema, in part of the groups
    if group > 32:
        w[0, 4:8] = float("nan")
    got, want = fake_int4_quant_cuda(w.to(DEV), (1, group), sym), oracle.fake_int4_quant(w, (1, group), sym)
    for a, b, what in list(zip(got, want, ("codes", "scales", "zero points")))[: 2 if sym else 3]:
        _assert_same(a.nan_to_num(nan=77.0), b.nan_to_num(nan=77.0), what)


@pytest.mark.parametrize("kind", ["int4", "int4_asym", "mxfp4", "nvfp4"])
def test_fp32_in_one_list_with_16_bit_tensors(oracle, kind):
    """A recorded list of seventy-odd tensors (more than the kernel arguments of a launch hold), run twice."""
    from miles_amd import launch
    from miles_amd.kernels.quant.int4_fake import pack_layer
    from miles_amd.utils.mxfp4 import quantize_mxfp4
    from miles_amd.utils.nvfp4 import nvfp4_quantize_1d

    here, there = {"int4": (lambda t: pack_layer(t, 32)[:2], lambda t: oracle.pack_layer(t, 32)[:2]),
                   "int4_asym": (lambda t: pack_layer(t, 32, False), lambda t: oracle.pack_layer(t, 32, False)),
                   "mxfp4": (lambda t: quantize_mxfp4(t, 32), lambda t: oracle.quantize_mxfp4(t, 32)),
                   "nvfp4": (lambda t: nvfp4_quantize_1d(t)[:2], lambda t: oracle.nvfp4_quantize_1d(t)[:2])}[kind]
    tensors = [fp32_case((40, 160), 60 + i) for i in range(72)]
    tensors[5], tensors[6] = tensors[5].bfloat16(), tensors[6].half()
    dev = [t.to(DEV) for t in tensors]
    with launch.recording() as batch:
        outs = [here(t) for t in dev]
    batch.freeze()
    for rep in range(2):
        batch.run()
        torch.cuda.synchronize()
        for i, t in enumerate(tensors):
            for got, want, what in zip(outs[i], there(t), ("codes", "scales")):
                _assert_same(got, want, f"tensor {i} ({t.dtype}) {what}, run {rep}")
        for o in outs:
            for t in o:
                t.view(torch.uint8).fill_(0x5A)
