"""NVFP4 in two passes: the quantize pass folds the partial maxima itself and publishes the record, around the sizes where
the amax pass gets another workgroup; and what a plain run leaves in the record does not reach the carried run behind it."""

import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.utils.nvfp4 import nvfp4_quantize_1d, nvfp4_quantize_1d_pair

pytestmark = pytest.mark.gpu
CHUNK = 256 * 4 * 8        # elements a workgroup of the amax pass reads at a time (16-bit inputs; half as many fp32 ones)


def _same(got, want, what):
    for j, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a.cpu().contiguous().reshape(-1).view(torch.uint8), b.contiguous().reshape(-1).view(torch.uint8)), f"{what}, output {j}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("four_over_six", [False, True])
@pytest.mark.parametrize("cols", [16, CHUNK // 2, CHUNK // 2 + 16, CHUNK, CHUNK + 16, 3 * CHUNK + 48, 256 * CHUNK + 16])
def test_plain_run_then_smaller_weights(cols, four_over_six, dtype, monkeypatch, oracle):
    monkeypatch.setenv("NVTE_NVFP4_4OVER6", "weights" if four_over_six else "none")
    options = {"e4m3_max": 256, "flags": 1} if four_over_six else {}
    g = torch.Generator().manual_seed(cols)
    cpu = [(torch.randn(1, cols, generator=g) * s).to(dtype) for s in (1.0, 0.02, 0.0, 30.0)]
    cpu[0][0, -1] = 50.0                                   # the largest element in the last block of 16
    dev = [w.cuda() for w in cpu]
    none = torch.empty(0, cols, dtype=dtype, device="cuda")
    with launch.recording() as batch:
        singles = [nvfp4_quantize_1d(dev[0]), nvfp4_quantize_1d(none), nvfp4_quantize_1d(dev[1])]
        pair = nvfp4_quantize_1d_pair(dev[2], dev[3])
    records = batch.amax_records()
    for r in records:
        r.fill_(0x7F7F7F7F)                                # whatever the allocation held
    for run in range(3):
        if run == 1:                                       # every partial maximum of the plain run is now too large
            batch.carry_amax(adaptive=False)
            for w in dev:
                w.mul_(0.25)
        batch.run()
        for i, k in ((0, 0), (1, 2)):
            _same(singles[k], oracle.nvfp4_quantize_1d(dev[i].cpu(), **options), f"run {run}, tensor {i}")
        _same([t for out in pair for t in out],
              [t for out in oracle.nvfp4_quantize_1d_pair(dev[2].cpu(), dev[3].cpu(), **options) for t in out], f"run {run}, pair")
        assert singles[1][2].item() == torch.tensor(torch.finfo(torch.float32).max).reciprocal().item(), "an empty tensor's scale"
        for r, top in zip(records, (dev[0].abs().max().item(), 0.0, dev[1].abs().max().item(), dev[3].abs().max().item())):
            assert r[_lib.RECORD_AMAX_WORD].view(torch.float32).item() == top


@pytest.mark.parametrize("no_wait", [False, True])
def test_read_once_then_smaller_weights(no_wait):
    g = torch.Generator(device="cuda").manual_seed(3)
    x = (torch.randn(6, 1024, 7168, generator=g, device="cuda") * 4.0).bfloat16()       # patterns with the exponent's top bit set
    with launch.recording() as batch:
        got = [nvfp4_quantize_1d(x[0]), nvfp4_quantize_1d(x[1]), *nvfp4_quantize_1d_pair(x[2], x[3]), nvfp4_quantize_1d(x[4]),
               nvfp4_quantize_1d(x[5])]
    if no_wait:
        batch.replace_records([r[:batch.P1] + (r[batch.P1] | _lib.NVFP4_NO_WAIT,) + r[batch.P1 + 1:] for r in batch.records])
    for run in range(3):
        if run == 1:
            batch.carry_amax(adaptive=False)
            x.mul_(0.125)
        batch.run()
        want = [nvfp4_quantize_1d(x[0]), nvfp4_quantize_1d(x[1]), *nvfp4_quantize_1d_pair(x[2], x[3]), nvfp4_quantize_1d(x[4]),
                nvfp4_quantize_1d(x[5])]
        for i, (one, ref) in enumerate(zip(got, want)):
            _same(one, [t.cpu() for t in ref], f"run {run}, tensor {i}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_read_once_with_extreme_tensors(dtype):
    """What the kernel that reads a tensor once leaves to the workgroups behind: scales at the ends of the fp32 range,
    infinities, NaN.  Its neighbours in the list stay where they are."""
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(8, 1024, 7168, generator=g, device="cuda").to(dtype)
    left = [2, 4]
    x[2, 17, 40] = float("inf")
    x[4, 1023, 7167] = float("nan")
    x[6].zero_()
    if dtype == torch.bfloat16:
        left += [1, 5, 7]
        x[1] = (x[1].float() * 1e-30).bfloat16()
        x[5] = (x[5].float() * 1e-40).bfloat16()           # subnormal elements
        x[7] = (x[7].float() * 5e37).bfloat16()
        x[7].clamp_(-3e38, 3e38)
    with launch.recording() as batch:
        got = [nvfp4_quantize_1d(w) for w in x]
    for run in range(2):
        if run == 1:
            batch.carry_amax(adaptive=False)
        batch.run()
        if run == 0:
            redo = [int(r[_lib.RECORD_REDO_WORD]) for r in batch.amax_records()]
            assert redo == [int(i in left) for i in range(8)]        # (1e-30, 1e-40 and 3e38, over 2688: outside 2^-82 .. 2^81)
        for i, one in enumerate(got):
            _same(one, [t.cpu() for t in nvfp4_quantize_1d(x[i])], f"run {run}, tensor {i}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows, cols", [(1037, 3680), (1024, 4096), (1, 16 * 262147)])
def test_read_once_with_empty_blocks(rows, cols, dtype):
    """Blocks of zeros and blocks whose scale rounds to zero have the largest factor; the last workgroup's piece is cut off at
    the first or the second of two units."""
    g = torch.Generator(device="cuda").manual_seed(6)
    x = (torch.randn(10, rows * cols // 16, 16, generator=g, device="cuda") * 0.02).to(dtype)
    x[:, 5::11] = 0.0
    x[:, 7::13] *= 2.0 ** -14
    x[:, ::17, 3] *= -0.0
    x[:, -1, 15] = torch.arange(1.0, 11.0, device="cuda").to(dtype)
    x = x.view(10, rows, cols)
    with launch.deferred():
        got = [nvfp4_quantize_1d(w) for w in x]
    for i, one in enumerate(got):
        _same(one, [t.cpu() for t in nvfp4_quantize_1d(x[i])], f"tensor {i}")
