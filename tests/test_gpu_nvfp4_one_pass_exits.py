"""What an amax record says after a list was read once: which form its tensors took, and how the waiting ended."""

import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.utils.nvfp4 import nvfp4_quantize_1d, nvfp4_quantize_1d_pair

pytestmark = pytest.mark.gpu
FIRST_WORD, WORDS, STRIDE = 1056, 7, 32         # the words of a record that the waiting workgroups watch
PUBLISHED, GAVE_UP = 0x8000, 0x10000


def _run(tensors, pairs, flag=0):
    """Outputs, and of every record the words watched and the one that says it was left to the workgroups behind."""
    with launch.recording() as batch:
        if pairs:
            got = [t for i in range(0, len(tensors), 2) for t in nvfp4_quantize_1d_pair(tensors[i], tensors[i + 1])]
        else:
            got = [nvfp4_quantize_1d(t) for t in tensors]
    batch.replace_records([r[:batch.P1] + (r[batch.P1] | flag,) + r[batch.P1 + 1:] for r in batch.records])
    records = batch.amax_records()
    for r in records:
        r.zero_()
    batch.run()
    words = torch.stack([r[FIRST_WORD:FIRST_WORD + WORDS * STRIDE:STRIDE] for r in records]).cpu()
    redo = torch.stack([r[_lib.RECORD_REDO_WORD] for r in records]).cpu()
    return got, words, redo


def _tensors(n, rows, cols):
    g = torch.Generator(device="cuda").manual_seed(n)
    return list((torch.randn(n, rows, cols, generator=g, device="cuda") * 0.02).bfloat16())


@pytest.mark.parametrize("n, rows, cols, pairs", [(5, 1024, 7168, False), (70, 1031, 1040, False), (24, 768, 2048, True), (6, 1300, 7168, True)])
def test_a_first_workgroup_that_gives_up_says_so(n, rows, cols, pairs):
    """Every word that the other workgroups watch names the end of the wait, and the workgroups behind quantize the record."""
    x = _tensors(n, rows, cols)
    got, words, redo = _run(x, pairs, _lib.NVFP4_NO_WAIT)
    assert (words == words[:, :1]).all()
    gave_up = words[:, 0] == GAVE_UP
    assert (gave_up | ((words[:, 0] & PUBLISHED) != 0)).all()       # (a first workgroup may find all others done already)
    assert gave_up.any() and (redo[gave_up] == 1).all()
    want = [t for i in range(0, n, 2) for t in nvfp4_quantize_1d_pair(x[i], x[i + 1])] if pairs else [nvfp4_quantize_1d(t) for t in x]
    for one, ref in zip(got, want):
        for a, b in zip(one, ref):
            assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8))


@pytest.mark.parametrize("n, rows, cols, pairs, one_pass", [
    (5, 1024, 7168, False, True), (3, 2048, 8192, False, True), (2, 2048, 8208, False, False), (70, 1031, 1040, False, True),
    (1100, 1, 256 * 16 * 8 + 16, False, True), (2200, 1, 256 * 16 * 8, False, True),
    (24, 768, 2048, True, True), (6, 1300, 7168, True, True), (4, 2048, 7168, True, False)])
def test_lists_that_are_read_once(n, rows, cols, pairs, one_pass):
    """The lists that the comparison with single calls takes, and two that keep two passes: a tensor past a section's slots, a
    pair of more workgroups than may share a record.  With the chip to itself no workgroup waits in vain."""
    _got, words, redo = _run(_tensors(n, rows, cols), pairs)
    assert (((words & PUBLISHED) != 0) if one_pass else (words == 0)).all()
    assert (redo == 0).all()


def test_two_streams_at_once():
    """Two lists whose workgroups compete for the chip: whoever waits in vain leaves its record to the workgroups behind, and every
    byte is that of a single call."""
    lists = [_tensors(12, 2048, 7168), [t * 3 for t in _tensors(9, 2048, 8192)]]
    streams = [torch.cuda.Stream() for _ in lists]
    batches, outs = [], []
    for x in lists:
        with launch.recording() as batch:
            outs.append([nvfp4_quantize_1d(t) for t in x])
        batch.freeze()
        batches.append(batch)
    want = [[nvfp4_quantize_1d(t) for t in x] for x in lists]
    torch.cuda.synchronize()
    for rep in range(4):
        for batch, stream in zip(batches, streams):
            batch.run(stream.cuda_stream)
        torch.cuda.synchronize()
        for got, ref in zip(outs, want):
            for one, two in zip(got, ref):
                for a, b in zip(one, two):
                    assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8))
                    a.reshape(-1).view(torch.uint8).fill_(0xA5)
        torch.cuda.synchronize()


@pytest.mark.parametrize("n, kib, one_pass", [
    (66, 383, False), (66, 384, True),              # 24 MiB and more: 384 KiB a tensor
    (127, 383, False), (128, 384, True),            # around 48 MiB
    (160, 319, False), (160, 320, True),            # from 48 MiB on 320 KiB
    (800, 64, False), (1024, 64, True),             # from 64 MiB on any
])
@pytest.mark.parametrize("pairs", [False, True])
def test_lists_of_small_tensors(n, kib, one_pass, pairs):
    """Over a device table: two passes for lists of many small tensors."""
    if pairs and n % 2:
        n += 1
    x = _tensors(n, kib, 512)
    x[n - 1][kib - 1, 511] = 3.0
    got, words, redo = _run(x, pairs)
    assert (((words & PUBLISHED) != 0) if one_pass else (words == 0)).all()
    assert (redo == 0).all()
    for i in (0, 2, n // 2 & ~1, n - 2):
        want = nvfp4_quantize_1d_pair(x[i], x[i + 1]) if pairs else [nvfp4_quantize_1d(x[i]), nvfp4_quantize_1d(x[i + 1])]
        for one, ref in zip(got[i:i + 2], want):
            for a, b in zip(one, ref):
                assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8))


@pytest.mark.parametrize("n, rows, cols", [(1100, 4, 8192), (1100, 2, 16400), (140, 60, 8192), (140, 5, 98320)])
def test_few_workgroups_behind_small_tensors(n, rows, cols):
    """One, two, 15 and 16 of them behind each tensor, whose last piece is whole or of a few blocks: they quantize the tensors whose
    first workgroup gave up (a tensor of one workgroup has nothing to wait for)."""
    x = _tensors(n, rows, cols)
    got, words, redo = _run(x, False, _lib.NVFP4_NO_WAIT)
    assert (words != 0).all()
    for i in range(0, n, 7):
        for a, b in zip(got[i], nvfp4_quantize_1d(x[i])):
            assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8))
