"""Infinities and NaN of either sign, in fp32 tensors: the tuned kernels against the element-wise ones, which a tensor off a
16-byte boundary takes, byte for byte; where the reference defines the result, against the oracle as well."""

import pytest
import torch

from tests.test_gpu_fp32_kernels import DEV, _assert_same, fp32_case, oracle  # noqa: F401

pytestmark = pytest.mark.gpu

QUIET, SIGNED = 0x7FC00000, 0xFFC00001 - (1 << 32)


def _with_specials(shape, seed, nan=True):
    """Elements, whole groups and a whole row of infinities and NaN; most groups stay finite, or keep finite elements."""
    g = torch.Generator().manual_seed(seed)
    x = fp32_case(shape, seed)
    kinds = torch.tensor([float("inf"), -float("inf"), 3.4028235e38, -0.0])
    at = torch.rand(shape, generator=g) < 0.004
    x = torch.where(at, kinds[torch.randint(0, 4, shape, generator=g)], x)
    if nan:
        bits = x.view(torch.int32)
        bits[torch.rand(shape, generator=g) < 0.004] = QUIET
        bits[torch.rand(shape, generator=g) < 0.004] = SIGNED
        bits[0, :32] = QUIET
        bits[-1, -128:] = SIGNED
    x[0, -32:] = float("inf")
    return x


def _off_boundary(x):
    buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)
    buf[1:] = x.reshape(-1).to(DEV)
    out = buf[1:].view(x.shape)
    assert out.data_ptr() % 16 == 4
    return out


def _both(quantize, x, what):
    outs = quantize(x.to(DEV))
    for i, (a, b) in enumerate(zip(outs, quantize(_off_boundary(x)))):
        if isinstance(a, torch.Tensor) and a.numel():
            _assert_same(a.reshape(-1), b.reshape(-1), f"{what} output {i}")
    return outs


@pytest.mark.parametrize("shape", [(1, 128), (5, 384), (129, 2032), (40, 4112)])
@pytest.mark.parametrize("mode", [None, "MAE", "MSE", "FP16", "FP16 MSE"])
@pytest.mark.parametrize("nan", [False, True])
def test_nvfp4(oracle, monkeypatch, shape, mode, nan):  # noqa: F811
    from miles_amd import _lib
    from miles_amd.utils.nvfp4 import nvfp4_quantize_1d

    e4m3_max, flags = 448, 0
    if mode is not None:
        monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights")
        monkeypatch.setenv("NVTE_NVFP4_4OVER6_ERR_MODE", "MSE" if "MSE" in mode else "MAE")
        monkeypatch.setenv("NVTE_NVFP4_4OVER6_ERR_USE_FAST_MATH", "1" if "FP16" in mode else "0")
        e4m3_max = 256
        flags = _lib.NVFP4_4OVER6 | (_lib.NVFP4_ERR_MSE if "MSE" in mode else 0) | (_lib.NVFP4_ERR_FP16 if "FP16" in mode else 0)
    x = _with_specials(shape, 900 + shape[1], nan)
    q, s, g = _both(nvfp4_quantize_1d, x, f"{mode} {shape}")
    if not nan:         # (the oracle's amax passes a NaN over)
        q_o, s_o, g_o = oracle.nvfp4_quantize_1d(x, e4m3_max=e4m3_max, flags=flags)
        _assert_same(g.reshape(1), torch.as_tensor(g_o).reshape(1).float(), "global scale")
        _assert_same(s, s_o, "scales")
        _assert_same(q, q_o, "codes")


@pytest.mark.parametrize("shape", [(8, 128), (16, 4224), (136, 1024)])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("symmetric", [True, False])
def test_int4(oracle, shape, group, symmetric):  # noqa: F811
    """NaN (skipped by the extrema, code by code 8 or 0) and infinities send a wavefront through the chain as written, next
    to groups that keep the fused form."""
    from miles_amd.kernels.quant.int4_fake import pack_layer

    x = _with_specials(shape, 920 + shape[1] + group)
    outs = _both(lambda w: [t for t in pack_layer(w, group, symmetric) if t is not None], x, f"group {group}")
    # the oracle where a group is finite, or holds NaN but not only NaN, among which the reference's fmaxf picks the rest
    want = oracle.pack_layer(x, group, symmetric)
    grouped = x.view(shape[0], -1, group)
    finite = torch.isfinite(grouped).all(-1)
    _assert_same(outs[1].cpu()[finite], want[1][finite], "scales of finite groups")
    words = finite.repeat_interleave(group // 8, 1)
    _assert_same(outs[0].cpu()[words], want[0][words], "codes of finite groups")
    assert 0 < int(finite.sum()) < finite.numel()


@pytest.mark.parametrize("shape", [(1, 128), (5, 384), (129, 2016), (513, 1024)])
def test_mx_formats(shape):
    from miles_amd.utils.mxfp4 import quantize_mxfp4
    from miles_amd.utils.mxfp8 import mxfp8_quantize

    x = _with_specials(shape, 940 + shape[1])
    _both(lambda w: quantize_mxfp4(w, 32), x, "mxfp4")
    _both(mxfp8_quantize, x, "mxfp8")


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("symmetric", [True, False])
def test_fake_int4(group, symmetric):
    from miles_amd.kernels.quant.int4_fake import fake_int4_quant_cuda

    # (a NaN result carries the sign and payload its operands happen to give it)
    _both(lambda w: [t.nan_to_num(nan=77.0) for t in fake_int4_quant_cuda(w, (1, group), symmetric)[: 2 if symmetric else 3]],
          _with_specials((129, 2048), 960 + group), f"group {group}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("four_over_six", [False, True])
def test_lists_of_16_bit_weights(oracle, dtype, four_over_six):  # noqa: F811
    """NVFP4 fake quantization of lists: an infinite weight against the oracle, a NaN makes every result of its weight NaN and
    of no other."""
    from miles_amd import _lib
    from miles_amd.kernels.quant import nvfp4_qdq as m

    cfg = m.NVFP4QDQConfig(four_over_six, 256 if four_over_six else 448)
    weights = []
    for i, shape in enumerate([(3, 48), (129, 1040), (130, 1040), (1, 8208), (5, 2736)]):
        w = (fp32_case(shape, 980 + i) * 2.0**-12).to(dtype)
        if i % 2:
            w[0, 5], w[-1, -1] = float("inf"), -float("inf")
        if i == 2:
            w[-1, 3] = float("nan")
        weights.append(w)
    got = m.fake_nvfp4_quantization_ste_list([w.to(DEV) for w in weights], cfg)
    for i, (y, w) in enumerate(zip(got, weights)):
        if i == 2:
            assert torch.isnan(y).all()
            continue
        want = oracle.fused_nvfp4_qdq(w, e4m3_max=cfg.e4m3_max, flags=_lib.NVFP4_4OVER6 if four_over_six else 0)
        _assert_same(y.nan_to_num(nan=77.0), want.nan_to_num(nan=77.0), f"weight {i}")
