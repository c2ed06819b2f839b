"""Quantizers that read a list twice, over lists of the lengths at which the first pass asks the memory-side cache for all, half
or none of it: the same bytes as each tensor alone, wherever the largest element lies."""

import pytest
import torch

from miles_amd import launch
from miles_amd.tools.convert_hf_to_fp8 import quant_fp8
from miles_amd.utils.nvfp4 import nvfp4_quantize_1d

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _weights(total, count, odd, dtype):
    """`count` matrices of together about `total` bytes; the largest element of each comes from another load of the amax pass."""
    numel = total // (count * (4 if dtype == torch.float32 else 2))
    cols = 4096 + 16 * odd
    g = torch.Generator(device="cuda").manual_seed(total % 1009 + odd)
    ws = [(torch.randn(numel // cols, cols, generator=g, device="cuda") * 0.02).to(dtype) for _ in range(count)]
    for i, w in enumerate(ws):
        w.view(-1)[(-1, 0, 2048, 5000, 7000)[i % 5]] = 4.0 + i
    return ws


def _same(got, want, what):
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.equal(a.contiguous().reshape(-1).view(torch.uint8), b.contiguous().reshape(-1).view(torch.uint8)), what


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("total", [200 * MIB, 300 * MIB, 800 * MIB])
@pytest.mark.parametrize("odd", [0, 1])
def test_long_lists(total, odd, dtype, monkeypatch):
    monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights" if dtype == torch.bfloat16 else "none")      # (in two passes)
    ws = _weights(total, 7, odd, dtype)
    with launch.deferred():
        fp4 = [nvfp4_quantize_1d(w) for w in ws]
    with launch.deferred():
        fp8 = [quant_fp8(w, "tensor") for w in ws]
    for i, w in enumerate(ws):
        _same(fp4[i], nvfp4_quantize_1d(w), f"NVFP4 {i}")
        _same(fp8[i], quant_fp8(w, "tensor"), f"FP8 {i}")
        assert fp8[i][1].item() == (torch.tensor(4.0 + i) / torch.tensor(448.0)).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("numels", [(8 * MIB // 4, 8 * MIB // 4 - 1, 8 * MIB // 4 + 9), (5 * 8192 - 1, 8192 * 900 + 7, 8192 * 900 - 4100)])
@pytest.mark.parametrize("at", [0, 1])
def test_fp8_tensor_four_units_a_lane(numels, at, dtype):
    """Lists at and above 8 MiB, with tails around the edges of a workgroup's piece."""
    from oracle import mq_oracle as oracle

    g = torch.Generator().manual_seed(len(numels) + at)
    cpu = [(torch.randn(1, n, generator=g) * 0.02).to(dtype) for n in numels]
    dev = []
    for w in cpu:
        flat = torch.empty(w.numel() + 1, dtype=dtype, device="cuda")
        flat[at:at + w.numel()] = w.reshape(-1).cuda()
        dev.append(flat[at:at + w.numel()].view(1, -1))
    with launch.deferred():
        got = [quant_fp8(d, "tensor") for d in dev]
    for w, result in zip(cpu, got):
        for have, ref in zip(result, oracle.tensor_fp8(w)):
            assert have.shape == ref.shape and torch.equal(have.cpu().reshape(-1).view(torch.uint8), ref.reshape(-1).view(torch.uint8)), tuple(w.shape)
