"""NVFP4 lists with Four Over Six that are read once, against the same tensors quantized one by one: every byte equal."""

import ctypes

import pytest
import torch

from miles_amd import _lib, _probes, launch
from miles_amd.utils.nvfp4 import nvfp4_quantize_1d, nvfp4_quantize_1d_pair

pytestmark = pytest.mark.gpu
FIRST_WORD, WORDS, STRIDE, PUBLISHED = 1056, 7, 32, 0x8000          # the words of a record that the waiting workgroups watch
MIB = 1 << 20


def _same(got, want, what):
    for a, b in zip(got, want):
        a, b = (t.contiguous().reshape(-1).view(torch.uint8) for t in (a, b))
        assert torch.equal(a, b), what


def _scribble(got):
    for one in got:
        for t in one:
            t.view(torch.uint8).fill_(0xA5) if t.dim() else t.fill_(-1.0)


@pytest.fixture
def four_over_six(monkeypatch):
    monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights")


def _tensors(n, rows, cols, dtype):
    g = torch.Generator(device="cuda").manual_seed(n + cols)
    x = torch.randn(n, rows, cols, generator=g, device="cuda") * 0.02
    # every third block of small whole numbers: its two errors are often the same, or both zero
    few = torch.randint(-6, 7, x.shape, generator=g, device="cuda") * 0.03125
    block = torch.arange(x[0].numel(), device="cuda").reshape(rows, cols) // 16 % 3 == 0
    x = torch.where(block, few, x).to(dtype)
    x[:, 0, :16] = x[:, 0, :16].abs() + 0.01
    if n > 4:
        x[0, 0, 3] = float("inf")                       # what the other code does: not a number, an empty range, a maximum
        x[1, rows - 1, cols - 1] = float("nan")         # below the range of the shared division
        x[2].zero_()
        if dtype == torch.bfloat16:
            x[3] *= 2.0 ** -65
    return x


@pytest.mark.parametrize("first_polls, patience", [(256, 1 << 16), (0, 0)])
@pytest.mark.parametrize("mse", [False, True])
@pytest.mark.parametrize("n, rows, cols", [
    (1, 2048, 8192),                    # every slot of a section
    (5, 512, 7216),                     # ragged last workgroup
    (6, 1, 16),                         # one block
    (9, 1, 256 * 16 * 8 + 16),          # one block in the second workgroup
    (64, 3, 16384),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_equals_single_calls(four_over_six, monkeypatch, n, rows, cols, mse, first_polls, patience, dtype):
    if mse:
        monkeypatch.setenv("NVTE_NVFP4_4OVER6_ERR_MODE", "MSE")
    x = _tensors(n, rows, cols, dtype)
    with launch.recording() as batch:
        got = [nvfp4_quantize_1d(t) for t in x]
    assert all(r[batch.P1] == _lib.NVFP4_4OVER6 | (_lib.NVFP4_ERR_MSE if mse else 0) for r in batch.records)
    _scribble(got)
    stream = torch.cuda.current_stream().cuda_stream
    _probes.check(_probes.load().mqp_nvfp4_one_pass(ctypes.byref(batch.freeze()), n, first_polls, patience, stream))
    for i in range(n):
        _same(got[i], nvfp4_quantize_1d(x[i]), f"tensor {i}")


@pytest.mark.parametrize("n, rows, cols, pairs, once", [
    (13, 1024, 8192, False, True),      # 208 MiB
    (12, 1024, 8192, False, False),     # 192 MiB
    (26, 509, 8208, True, True),
    (3, 5120, 8192, False, False),      # more workgroups than share a record on the chip
])
def test_which_lists_are_read_once(four_over_six, n, rows, cols, pairs, once):
    x = _tensors(n, rows, cols, torch.bfloat16)
    assert (n * rows * cols * 2 >= 200 * MIB) == (once or rows > 4096)
    with launch.recording() as batch:
        if pairs:
            got = [t for i in range(0, n, 2) for t in nvfp4_quantize_1d_pair(x[i], x[i + 1])]
        else:
            got = [nvfp4_quantize_1d(t) for t in x]
    for run in range(3):
        if run == 0:
            for record in batch.amax_records():
                record.zero_()
        if run == 1:
            batch.carry_amax(adaptive=False)            # the records serve a carried run
        if run == 2:
            x[4 % n, 0, 0] = 1e3
        _scribble(got)
        batch.run()
        if run == 0:
            words = torch.stack([r[FIRST_WORD:FIRST_WORD + WORDS * STRIDE:STRIDE] for r in batch.amax_records()]).cpu()
            assert bool((words & PUBLISHED).bool().all()) if once else not bool(words.any())
        for i in range(0, n, 2 if pairs else 1):
            if pairs:
                for one, ref in zip(got[i:i + 2], nvfp4_quantize_1d_pair(x[i], x[i + 1])):
                    _same(one, ref, f"run {run}, tensor {i}")
            else:
                _same(got[i], nvfp4_quantize_1d(x[i]), f"run {run}, tensor {i}")
