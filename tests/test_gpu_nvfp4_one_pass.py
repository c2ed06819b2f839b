"""NVFP4 lists that are read once (the workgroups of a tensor hold it and wait for each other's maxima) against the same
tensors quantized one by one, which takes the two-pass kernels: every byte equal."""

import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.megatron_to_hf.processors.quantizer_nvfp4 import quantize_nvfp4
from miles_amd.utils.nvfp4 import nvfp4_quantize_1d, nvfp4_quantize_1d_pair

pytestmark = pytest.mark.gpu
WORKGROUP = 256 * 16 * 8        # elements a workgroup holds


def _stack(n, rows, cols, dtype):
    g = torch.Generator(device="cuda").manual_seed(n * rows + cols)
    x = torch.randn(n, rows, cols, generator=g, device="cuda")
    return (x * torch.logspace(-3, 2, n, device="cuda").reshape(-1, 1, 1)).to(dtype)


def _same(got, want):
    for a, b in zip(got, want):
        a, b = (t.contiguous().reshape(-1).view(torch.uint8) for t in (a, b))
        assert torch.equal(a, b)


@pytest.mark.parametrize("n, rows, cols", [
    (5, 1024, 7168),                      # whole workgroups
    (3, 2048, 8192),                      # the largest tensor: every slot of a section used
    (2, 2048, 8208),                      # one block row past it: two passes
    (70, 1031, 1040),                     # ragged end, odd slot count; more tensors than one launch takes
    (1100, 1, WORKGROUP + 16),            # one block in the second workgroup
    (2200, 1, WORKGROUP),                 # one workgroup a tensor
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_pass_equals_single_calls(n, rows, cols, dtype):
    x = _stack(n, rows, cols, dtype)
    x[0, 0, 5] = float("nan")
    x[1, -1, -1] = float("inf")
    x[n - 1].zero_()
    with launch.deferred():
        got = quantize_nvfp4(x)
    for i in (range(n) if n < 100 else [0, 1, 2, n // 2, n - 1]):
        _same([t[i] for t in got], nvfp4_quantize_1d(x[i]))


@pytest.mark.parametrize("no_wait", [False, True])
@pytest.mark.parametrize("pairs, rows, cols", [(12, 768, 2048), (40, 768, 2048), (3, 1300, 7168)])
def test_pairs_what_is_left_and_a_carried_run(pairs, rows, cols, no_wait):
    """A pair waits for both of its tensors; with no waiting at all the workgroups behind do what is left; either way the
    records serve a carried run.  (Pairs of [1300, 7168] are 570 workgroups, close to the most that share a record;
    40 pairs are submitted over a device table.)"""
    x = _stack(2 * pairs, rows, cols, torch.bfloat16)
    assert x.nbytes >= 24 << 20         # (shorter lists take two passes)
    with launch.recording() as batch:
        got = [t for i in range(pairs) for t in nvfp4_quantize_1d_pair(x[2 * i], x[2 * i + 1])]
    if no_wait:
        batch.replace_records([r[:batch.P1] + (r[batch.P1] | _lib.NVFP4_NO_WAIT,) + r[batch.P1 + 1:] for r in batch.records])
    want = [t for i in range(pairs) for t in nvfp4_quantize_1d_pair(x[2 * i], x[2 * i + 1])]
    for run in range(3):
        if run == 1:
            batch.carry_amax(adaptive=False)
        if run == 2:                      # one pair's amax moves
            x[2, 0, 0] = 1e4
            want[2:4] = nvfp4_quantize_1d_pair(x[2], x[3])
        for one in got:
            for t in one:
                t.view(torch.uint8).fill_(0xA5) if t.dim() else t.fill_(-1.0)
        batch.run()
        for one, ref in zip(got, want):
            _same(one, ref)
