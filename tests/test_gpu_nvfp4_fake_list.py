"""NVFP4 fake quantization of lists of weights: one kernel for both forms of block scaling, amax folded where it is used."""

import pytest
import torch

from tests.test_gpu_fp32_kernels import DEV, _assert_same, fp32_case, oracle  # noqa: F401

pytestmark = pytest.mark.gpu

# one block, ragged ends of a workgroup (512 or 1024 units of eight elements), several workgroups, a ragged mix of sizes
SHAPES = [(1, 16), (1, 4096), (1, 4112), (3, 2736), (1, 8192), (1, 8208), (129, 1040), (130, 1040), (5, 48)]
MODES = [(False, 448, "MAE", False), (True, 448, "MAE", False), (True, 256, "MSE", False), (True, 256, "MAE", True), (True, 448, "MSE", True)]


def _weights(dtype, specials):
    out = []
    for i, shape in enumerate(SHAPES * 8):      # more than one launch holds
        x = fp32_case(shape, 500 + i, specials and i % 4 == 0) * (2.0**-12 if dtype == torch.float16 else 1.0)
        if i == 3:
            x = torch.zeros_like(x)
        out.append(x.to(dtype))
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("specials", [False, True])
def test_list_against_oracle(oracle, dtype, mode, specials):  # noqa: F811
    from miles_amd import _lib
    from miles_amd.kernels.quant import nvfp4_qdq as m

    fos, top, err, fast = mode
    cfg = m.NVFP4QDQConfig(fos, top, m.NVFP4QDQErrorMode[err], fast)
    flags = (_lib.NVFP4_4OVER6 if fos else 0) | (_lib.NVFP4_ERR_MSE if err == "MSE" else 0) | (_lib.NVFP4_ERR_FP16 if fast else 0)
    host = _weights(dtype, specials)
    dev = [w.to(DEV).requires_grad_(True) for w in host]
    got = m.fake_nvfp4_quantization_ste_list(dev, cfg)
    for i, (y, w, d) in enumerate(zip(got, host, dev)):
        if torch.isfinite(w).all():
            _assert_same(y.detach(), oracle.fused_nvfp4_qdq(w, e4m3_max=top, flags=flags), f"tensor {i} {tuple(w.shape)}")
        # alone, and with the amax as a scalar of the caller's
        _assert_same(m.fake_nvfp4_quantization_ste(d, cfg).detach(), y.detach(), f"tensor {i} alone")
        _assert_same(m.fused_nvfp4_qdq(d, m.compute_nvfp4_amax(d), cfg), y.detach(), f"tensor {i} with its amax")


def test_graph_nodes_of_a_list(monkeypatch):
    """Every weight keeps a node of its own: frozen weights, separate backward passes, gradients that never come."""
    from miles_amd.kernels.quant import nvfp4_qdq as m
    from miles_amd.utils import nvfp4_fake_qat as qat

    for name in ("NVTE_USE_FAST_MATH", "NVTE_NVFP4_4OVER6", "NVTE_NVFP4_4OVER6_E4M3_USE_256"):
        monkeypatch.delenv(name, raising=False)
    monkeypatch.setenv(qat.NVFP4_FAKE_QAT_FLAG, "1")
    ws = [torch.randn(16, 32, device=DEV, dtype=torch.bfloat16).requires_grad_(i != 1) for i in range(4)]
    ws[2].main_grad = torch.zeros(16, 32, device=DEV)
    ys = qat.maybe_fake_quantize_nvfp4_weight_tensors(ws)
    assert [y.requires_grad for y in ys] == [True, False, True, True] and ys[2].main_grad is ws[2].main_grad
    assert not any(y._is_view() for y in ys)
    ys[0].sum().backward()
    assert torch.equal(ws[0].grad, torch.ones_like(ws[0])) and ws[2].grad is None and ws[3].grad is None
    (2 * ys[2]).sum().backward()
    assert torch.equal(ws[2].grad, torch.full_like(ws[2], 2)) and ws[3].grad is None
    # several kinds in one list go weight by weight; what a weight is refused for is named as before
    mixed = qat.maybe_fake_quantize_nvfp4_weight_tensors([ws[0], ws[3].half()])
    assert [y.dtype for y in mixed] == [torch.bfloat16, torch.float16]
    with pytest.raises(TypeError, match="BF16 and FP16"):
        qat.maybe_fake_quantize_nvfp4_weight_tensors([ws[0], ws[3].float()])
    with pytest.raises(ValueError, match="empty"):
        m.fake_nvfp4_quantization_ste(ws[0][:0])


def test_list_in_a_graph(oracle):  # noqa: F811
    """Captured and replayed, with new weights and the program's own work between the replays."""
    from miles_amd.kernels.quant import nvfp4_qdq as m

    cfg = m.NVFP4QDQConfig()
    dev = [torch.randn(64, 128, device=DEV).bfloat16() for _ in range(3)]
    m.fake_nvfp4_quantization_ste_list(dev, cfg)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ys = m.fake_nvfp4_quantization_ste_list(dev, cfg)
    for rep in range(4):
        for d in dev:
            d.copy_(torch.randn(64, 128, device=DEV) * 10.0**rep)
        graph.replay()
        torch.cuda.synchronize()
        for y, d in zip(ys, dev):
            _assert_same(y, oracle.fused_nvfp4_qdq(d.cpu()), f"replay {rep}")
