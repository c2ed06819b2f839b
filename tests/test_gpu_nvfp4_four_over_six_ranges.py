"""Four Over Six where its shorter forms begin and end: the amax around 2^-60 and 2^-80, blocks far below it, and an amax of
the caller's that its elements exceed."""

import pytest
import torch

from tests.test_gpu_fp32_kernels import DEV, _assert_same, fp32_case, oracle  # noqa: F401

pytestmark = pytest.mark.gpu
MODES = [(448, "MAE", False), (256, "MSE", False), (256, "MAE", True)]


def _weight(shape, amax, seed):
    """Blocks of every size from the tensor's maximum down to denormal numbers and zero."""
    x = fp32_case(shape, seed).reshape(-1, 16)
    x = x / x.abs().amax(1, keepdim=True).clamp_min(1e-30) * amax
    x = x * torch.exp2(-(torch.arange(len(x)) % 41).float() * 1.5)[:, None] * torch.tensor([1.0, 1.0, 0.75])[torch.arange(len(x)) % 3][:, None]
    x[0] = 0.0
    x[1, 3] = -amax
    return x.reshape(shape).bfloat16()


@pytest.mark.parametrize("top, err, fast", MODES)
@pytest.mark.parametrize("exponent", [-81.0, -79.9, -60.1, -60.0, -59.9, -3.0, 76.5, 77.0])
@pytest.mark.parametrize("shape", [(2, 48), (33, 1040)])
def test_amax_ranges(oracle, monkeypatch, shape, exponent, top, err, fast):  # noqa: F811
    from miles_amd import _lib
    from miles_amd.kernels.quant import nvfp4_qdq as m
    from miles_amd.utils.nvfp4 import nvfp4_quantize_1d

    monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights")
    monkeypatch.setenv("NVTE_NVFP4_4OVER6_E4M3_USE_256", "all" if top == 256 else "none")
    monkeypatch.setenv("NVTE_NVFP4_4OVER6_ERR_MODE", err)
    monkeypatch.setenv("NVTE_NVFP4_4OVER6_ERR_USE_FAST_MATH", "1" if fast else "0")
    monkeypatch.delenv("NVTE_USE_FAST_MATH", raising=False)
    flags = _lib.NVFP4_4OVER6 | (_lib.NVFP4_ERR_MSE if err == "MSE" else 0) | (_lib.NVFP4_ERR_FP16 if fast else 0)
    w = _weight(shape, 2.0**exponent, 31 + shape[0])
    for a, b, what in zip(nvfp4_quantize_1d(w.to(DEV)), oracle.nvfp4_quantize_1d(w, e4m3_max=top, flags=flags), ("codes", "scales", "global scale")):
        _assert_same(a, b, what)
    cfg = m.NVFP4QDQConfig(True, top, m.NVFP4QDQErrorMode[err], fast)
    got = m.fake_nvfp4_quantization_ste_list([w.to(DEV).requires_grad_(True)], cfg)[0]
    _assert_same(got.detach(), oracle.fused_nvfp4_qdq(w, e4m3_max=top, flags=flags), "fake quantization")


@pytest.mark.parametrize("top, err, fast", MODES)
def test_amax_of_the_callers(oracle, top, err, fast):  # noqa: F811
    """An amax of few bits that is not the tensor's: below its elements, above them, and with a NaN and an infinity among them."""
    from miles_amd import _lib
    from miles_amd.kernels.quant import nvfp4_qdq as m

    cfg = m.NVFP4QDQConfig(True, top, m.NVFP4QDQErrorMode[err], fast)
    flags = _lib.NVFP4_4OVER6 | (_lib.NVFP4_ERR_MSE if err == "MSE" else 0) | (_lib.NVFP4_ERR_FP16 if fast else 0)
    w = _weight((33, 1040), 1.0, 77)
    for i in range(2):
        for amax in (0.125, 0.96875, 8.0):
            amax = torch.tensor(amax)
            got = m.fused_nvfp4_qdq(w.to(DEV), amax.to(DEV), cfg)
            want = oracle.fused_nvfp4_qdq(w, amax=amax, e4m3_max=top, flags=flags)
            number = ~w.isnan()             # (a NaN's own code is the conversion's)
            _assert_same(got.cpu()[number].nan_to_num(nan=77.0), want[number].nan_to_num(nan=77.0), f"amax {amax}, specials {i}")
        w[3, 100], w[20, 7] = float("nan"), float("inf")
