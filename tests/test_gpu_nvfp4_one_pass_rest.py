"""NVFP4 lists that are read once: the rows of workgroups behind the tensors', which quantize what was left, and workgroups that
do not wait for the word of a record's first one."""

import ctypes

import pytest
import torch

from miles_amd import _lib, _probes, launch
from miles_amd.megatron_to_hf.processors.quantizer_nvfp4 import quantize_nvfp4
from miles_amd.utils.nvfp4 import nvfp4_quantize_1d, nvfp4_quantize_1d_pair

pytestmark = pytest.mark.gpu


def _same(got, want, what):
    for a, b in zip(got, want):
        a, b = (t.contiguous().reshape(-1).view(torch.uint8) for t in (a, b))
        assert torch.equal(a, b), what


@pytest.mark.parametrize("flag", [0, _lib.NVFP4_NO_WAIT])
@pytest.mark.parametrize("n, rows, cols, pairs", [
    (3, 1024, 11184, False),            # few tensors: as many workers as a section has words
    (9, 512, 7216, False),              # ragged last workgroup
    (128, 16, 16384, False),            # over a device table, workers bounded by a tensor's blocks
    (140, 257, 1040, False),            # over a device table
    (24, 768, 2048, True),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_what_is_left_and_the_records_behind_it(n, rows, cols, pairs, dtype, flag):
    g = torch.Generator(device="cuda").manual_seed(n + cols)
    x = (torch.randn(n, rows, cols, generator=g, device="cuda") * 0.02).to(dtype)
    x[0, 0, 3] = float("inf")                           # left whatever the waits do, and the last one too
    x[n - 1, rows - 1, cols - 1] = float("nan")
    if n > 3:
        x[2].zero_()
    with launch.recording() as batch:
        if pairs:
            got = [t for i in range(0, n, 2) for t in nvfp4_quantize_1d_pair(x[i], x[i + 1])]
        else:
            got = [nvfp4_quantize_1d(t) for t in x]
    batch.replace_records([r[:batch.P1] + (r[batch.P1] | flag,) + r[batch.P1 + 1:] for r in batch.records])
    for record in batch.amax_records():
        record.fill_(-1)                                # whatever was in this memory
    for run in range(3):
        if run == 1:
            batch.carry_amax(adaptive=False)            # the records serve a carried run
        if run == 2:
            x[1, 0, 0] = 1e3
        for one in got:
            for t in one:
                t.view(torch.uint8).fill_(0xA5) if t.dim() else t.fill_(-1.0)
        batch.run()
        check = range(0, n, 2) if pairs else range(n) if n < 20 else [0, 1, 2, n // 2, n - 2, n - 1]
        for i in check:
            if pairs:
                for one, ref in zip(got[i:i + 2], nvfp4_quantize_1d_pair(x[i], x[i + 1])):
                    _same(one, ref, f"run {run}, tensor {i}")
            else:
                _same(got[i], nvfp4_quantize_1d(x[i]), f"run {run}, tensor {i}")


@pytest.mark.parametrize("first_polls", [0, 256])
@pytest.mark.parametrize("n, rows, cols", [(1, 2048, 8192), (5, 512, 7216), (64, 3, 16384)])
def test_workgroups_that_wait_for_nobody(n, rows, cols, first_polls):
    """Whoever finds no word yet takes the maximum from the tensor, those behind as well: every byte as in a single call."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x = (torch.randn(n, rows, cols, generator=g, device="cuda") * 0.02).bfloat16()
    x[n // 2, 0, 3] = float("inf")
    with launch.recording() as batch:
        got = [nvfp4_quantize_1d(t) for t in x]
    for one in got:
        for t in one:
            t.view(torch.uint8).fill_(0xA5) if t.dim() else t.fill_(-1.0)
    stream = torch.cuda.current_stream().cuda_stream
    _probes.check(_probes.load().mqp_nvfp4_one_pass(ctypes.byref(batch.freeze()), n, first_polls, 0, stream))
    for i in range(n):
        _same(got[i], nvfp4_quantize_1d(x[i]), f"tensor {i}")


@pytest.mark.parametrize("first_polls, patience", [(0, 0), (0, 256), (256, 0)])
@pytest.mark.parametrize("n, rows, cols", [(1, 2048, 8192), (5, 512, 7216), (64, 3, 16384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_records_serve_a_carried_run_however_the_waits_ended(dtype, n, rows, cols, first_polls, patience):
    """Nothing that waits in vain may leave in a record what a carried run takes for its own."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x = (torch.randn(n, rows, cols, generator=g, device="cuda") * 4.0).to(dtype)       # patterns with the exponent's top bit set
    with launch.recording() as batch:
        got = [nvfp4_quantize_1d(t) for t in x]
    records = batch.amax_records()
    for record in records:
        record.fill_(-1)
    stream = torch.cuda.current_stream().cuda_stream
    _probes.check(_probes.load().mqp_nvfp4_one_pass(ctypes.byref(batch.freeze()), n, first_polls, patience, stream))
    words = max(256, -(-rows * cols // (256 * 16 * 8)))
    assert all(bool((r[:words] >= 0).all()) for r in records), "marked as words of a carried run are"
    for r, t in zip(records, x):
        assert r[_lib.RECORD_AMAX_WORD].view(torch.float32).item() == t.abs().max().float().item()
    batch.carry_amax(adaptive=False)
    for run in range(2):
        for one in got:
            for t in one:
                t.view(torch.uint8).fill_(0xA5) if t.dim() else t.fill_(-1.0)
        batch.run()
        for i in {0, 1, n // 2, n - 1} & set(range(n)):
            _same(got[i], nvfp4_quantize_1d(x[i]), f"run {run}, tensor {i}")
            assert records[i][_lib.RECORD_REDO_WORD].item() == 0 or run > 0, "the amax has not moved"
        x.mul_(0.125)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_stack_cut_into_launches(dtype):
    """Without a device table a list is cut after 64 tensors, and each launch has the workers for its own number of them."""
    g = torch.Generator(device="cuda").manual_seed(70)
    x = (torch.randn(70, 1024, 2064, generator=g, device="cuda") * 0.02).to(dtype)      # 4 MiB and more: both launches read once
    x[5, 1, 3] = float("inf")
    x[69, 1023, 2063] = float("nan")
    codes, scales, published = quantize_nvfp4(x)
    for i in (0, 4, 5, 6, 63, 64, 65, 68, 69):
        _same((codes[i], scales[i], published[i]), nvfp4_quantize_1d(x[i]), f"tensor {i}")
