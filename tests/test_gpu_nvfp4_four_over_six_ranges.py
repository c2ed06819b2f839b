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


@pytest.mark.parametrize("copies", [1, 1000])       # (from 64 MiB on the record is finished in a launch of its own)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("top, err, fast", MODES)
def test_record_of_the_callers(oracle, top, err, fast, dtype, copies):  # noqa: F811
    """mq_nvfp4_quant with a record that the caller has written: an amax of few bits below the elements, above them, and without
    the NaN and the infinity among them."""
    from miles_amd import _lib
    from miles_amd.utils.nvfp4 import AMAX_RECORD_WORDS

    flags = _lib.NVFP4_4OVER6 | (_lib.NVFP4_ERR_MSE if err == "MSE" else 0) | (_lib.NVFP4_ERR_FP16 if fast else 0)
    w = _weight((33, 1040), 1.0, 78).to(dtype)
    record = torch.zeros(AMAX_RECORD_WORDS, dtype=torch.int32, device=DEV)
    rows, cols = w.shape
    q = torch.empty((copies * rows, cols // 2), dtype=torch.uint8, device=DEV)
    s = torch.empty((copies * rows, cols // 16), dtype=torch.uint8, device=DEV)
    g = torch.empty((), device=DEV)
    for i in range(2):
        dev = w.to(DEV).repeat(copies, 1)
        nan = w.isnan().view(rows, -1, 16).any(-1)      # blocks with a NaN: the largest scale, whose codes are the conversion's
        number = ~nan.repeat_interleave(16, dim=1)
        for amax in (0.125, 0.96875, 8.0):
            record[7] = int(torch.tensor(amax).view(torch.int32))
            _lib.check(_lib.load().mq_nvfp4_quant(dev.data_ptr(), _lib.DTYPE_CODE[dtype], record.data_ptr(), 1, q.data_ptr(), s.data_ptr(),
                                                  g.data_ptr(), copies * rows, cols, top, flags, _lib.stream_ptr()))
            q_o, s_o, g_o = oracle.nvfp4_quantize_1d(w, amax, top, flags)
            s_o = torch.where(nan, 0x7E, s_o.view(torch.uint8))
            nibbles = torch.stack((q & 15, q >> 4), -1).view(copies, rows, cols)
            nibbles_o = torch.stack((q_o & 15, q_o >> 4), -1).view(rows, cols)
            what = f"amax {amax}, specials {i}"
            assert torch.equal(s.view(copies, rows, -1), s_o.to(DEV).expand(copies, -1, -1)), f"scales, {what}"
            assert torch.equal(nibbles[:, number.to(DEV)], nibbles_o[number].to(DEV).expand(copies, -1)), f"codes, {what}"
            _assert_same(g, g_o, f"global scale, {what}")
        w[3, 100], w[20, 7] = float("nan"), float("inf")
