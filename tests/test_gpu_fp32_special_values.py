"""Infinities and NaN of either sign in fp32 weights: the tuned kernels against the element-wise ones, which a tensor off a
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
