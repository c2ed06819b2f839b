"""NVFP4 in two passes: by which lists the records are finished in a launch of their own, around the sizes where that changes,
and that the results, the records and the counters are those of short lists, whose quantize pass does it."""

import ctypes

import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.utils.nvfp4 import nvfp4_quantize_1d, nvfp4_quantize_1d_pair

pytestmark = pytest.mark.gpu
MIB = 1 << 20
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _launches(batch):
    """Kernels of one run, counted in a capture of it."""
    nodes = _lib.load().hipGraphGetNodes        # (resolved in the HIP runtime that the library is linked against)
    nodes.restype, nodes.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        batch.run()
    count = ctypes.c_size_t()
    assert nodes(graph.raw_cuda_graph(), None, ctypes.byref(count)) == 0
    return count.value


def _quantize(weights, pairs):
    """The first 2 * pairs weights in pairs, the others by themselves."""
    out = [t for i in range(pairs) for t in nvfp4_quantize_1d_pair(weights[2 * i], weights[2 * i + 1])]
    return out + [nvfp4_quantize_1d(w) for w in weights[2 * pairs:]]


def _same(got, want, what):
    for i, (one, ref) in enumerate(zip(got, want, strict=True)):
        for j, (a, b) in enumerate(zip(one, ref, strict=True)):
            assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8)), f"{what}, tensor {i}, output {j}"


# dtype, Four Over Six, tensors, of them in pairs, bytes of a tensor, elements more or less in the last one, launches
CASES = [
    (BF16, False, 2, 2, 24 * MIB, 0, 2), (BF16, False, 4, 4, 24 * MIB, 0, 3), (F16, False, 4, 4, 24 * MIB, 0, 3),
    (BF16, False, 66, 66, 21 * MIB, 0, 3), (BF16, False, 2, 0, 48 * MIB, 0, 2),
    (F32, False, 16, 16, 4 * MIB, 0, 3), (F32, False, 16, 16, 4 * MIB, -16, 2), (F32, False, 16, 0, 4 * MIB, 0, 2),
    (F32, False, 16, 8, 4 * MIB, 0, 3), (F32, False, 16, 6, 4 * MIB, 0, 2), (F32, False, 72, 72, MIB, 0, 3), (F32, False, 72, 0, MIB, 0, 2),
    (BF16, True, 16, 0, 4 * MIB, 0, 3), (BF16, True, 16, 0, 4 * MIB, -16, 2), (F16, True, 16, 16, 4 * MIB, 0, 3),
    (F32, True, 16, 16, 4 * MIB, 0, 3), (F32, True, 16, 16, 4 * MIB, -16, 2), (F32, True, 32, 4, 4 * MIB, 0, 3),
    (F32, True, 32, 4, 4 * MIB, -16, 2), (F32, True, 32, 4, 8 * MIB, 0, 3), (F32, True, 32, 4, 8 * MIB, 16, 2),
]


@pytest.mark.parametrize("dtype, four_over_six, n, paired, size, more, launches", CASES)
def test_around_the_lines(dtype, four_over_six, n, paired, size, more, launches, monkeypatch):
    monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights" if four_over_six else "none")
    g = torch.Generator(device="cuda").manual_seed(n + paired)
    weights = []
    for i in range(n):
        w = torch.randn((size // dtype.itemsize + (more if i == n - 1 else 0)) // 16, 16, generator=g, device="cuda", dtype=dtype)
        w.view(-1)[-1 - i] = 20.0 + i           # the largest element, of each another one, in the last blocks
        weights.append(w)
    with launch.recording() as batch:
        got = _quantize(weights, paired // 2)
    records = batch.amax_records()
    for r in records:
        r.fill_(0x7F7F7F7F)                     # whatever the allocation held
    batch.freeze()
    torch.cuda.synchronize()
    assert _launches(batch) == launches
    counters = torch.zeros(2, dtype=torch.int32, device="cuda")
    table = batch._table.data_ptr() if batch._table is not None else None
    assert (table is not None) == (n > _lib.MAX_GROUP)
    for run in range(4):
        if run == 2:
            for w in weights:
                w.mul_(0.25)
        if run == 3 and dtype != F32:           # the single pass of a carried run over what the plain ones left
            batch.carry_amax(adaptive=False)
            for w in weights:
                w.mul_(0.5)
            batch.run()
        else:
            _lib.check(_lib.load().mq_run_jobs_feedback(batch.freeze(), len(batch), table, counters.data_ptr(), None, _lib.stream_ptr()))
            assert counters.tolist() == [(1, 1, 2, 2)[run] * n, (run + 1) * n]
        for i in range(0, n, 8):                # (a few at a time: lists whose quantize pass finishes the records)
            some = weights[i:i + 8] if i >= paired or i + 8 <= paired else None
            if some is not None and sum(w.nbytes for w in some) < 64 * MIB:
                _same(got[i:i + 8], _quantize(some, len(some) // 2 if i < paired else 0), f"run {run}, from {i}")
            else:
                pairs = range(i, min(i + 8, paired), 2)
                for k in pairs:
                    _same(got[k:k + 2], _quantize(weights[k:k + 2], 1), f"run {run}, pair {k}")
                for k in range(max(i, paired), min(i + 8, n)):
                    _same(got[k:k + 1], _quantize(weights[k:k + 1], 0), f"run {run}, tensor {k}")
        tops = torch.stack([w.abs().max().float() for w in weights])
        tops[:paired] = tops[:paired].view(-1, 2).max(dim=1).values.repeat_interleave(2)
        for r, top in zip(records, torch.unique_consecutive(tops) if len(records) < n else tops, strict=True):
            assert r[_lib.RECORD_AMAX_WORD].view(torch.float32).item() == top.item()
            if run < 3:
                assert r[_lib.RECORD_REDO_WORD].item() == 0 and r[_lib.RECORD_VOLATILE_WORD].item() == 0


@pytest.mark.parametrize("four_over_six", [False, True])
def test_an_empty_tensor_in_a_long_list(four_over_six, monkeypatch):
    monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights" if four_over_six else "none")
    g = torch.Generator(device="cuda").manual_seed(1)
    weights = [torch.randn(n, 2048, generator=g, device="cuda") for n in (*[1024] * 12, 0, 1024, 0, 0)]
    with launch.recording() as batch:
        got = _quantize(weights, len(weights) // 2)
    assert _launches(batch) == 3
    batch.run()
    for i in range(0, len(weights), 2):
        _same(got[i:i + 2], _quantize(weights[i:i + 2], 1), f"pair {i}")
