"""Lists of per-channel and per-tensor FP8 conversions, which share launches: neighbours of other shapes, dtypes, alignments and
strategies, more tensors than a launch takes, the tail of a tensor that is no whole number of units, and recorded lists."""

import pytest
import torch

from miles_amd import launch
from miles_amd.tools.convert_hf_to_fp8 import quant_fp8
from miles_amd.workloads import gaussian_outliers

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
SHAPES = [(5, 12), (5, 12), (64, 256), (66, 250), (3, 3), (0, 16), (8, 2048), (9, 2050), (7, 8200), (130, 33), (1, 4), (513, 1027)]


def _same(got, want, what):
    for have, ref in zip(got, want):
        assert have.shape == ref.shape and torch.equal(have.cpu().view(torch.uint8), ref.view(torch.uint8)), what


@pytest.mark.parametrize("strategies", [("channel",), ("tensor",), ("channel", "tensor")])
def test_lists_of_many_kinds(strategies):
    from oracle import mq_oracle as oracle

    cases = []
    for i in range(3):
        for j, (rows, cols) in enumerate(SHAPES):
            strategy = strategies[(i + j) % len(strategies)]
            if rows == 0 and strategy == "tensor":
                continue
            dtype = [torch.bfloat16, torch.float32, torch.float16][(i * j + i) % 3]
            w = gaussian_outliers((rows, cols), std=0.02, p_outlier=0.01, gain=20.0, seed=100 * i + j, dtype=dtype)
            flat = torch.empty(w.numel() + 1, dtype=dtype, device=DEV)
            at = (i + j) % 2                    # on the allocation's boundary, or one element off it
            flat[at:at + w.numel()] = w.reshape(-1).to(DEV)
            cases.append((strategy, w, flat[at:at + w.numel()].view(rows, cols)))
    with launch.deferred() as batch:
        got = [quant_fp8(d, strategy) for strategy, _w, d in cases]
    assert batch.direct_calls == 0
    for (strategy, w, _d), result in zip(cases, got):
        _same(result, (oracle.channel_fp8 if strategy == "channel" else oracle.tensor_fp8)(w), f"{strategy} {tuple(w.shape)} {w.dtype}")


@pytest.mark.parametrize("strategy", ["channel", "tensor"])
@pytest.mark.parametrize("count", [2, 5, 70])
def test_equal_tensors_share_launches(strategy, count):
    """The number of partial maxima of a tensor depends on how many tensors there are; the largest element comes first or last."""
    from oracle import mq_oracle as oracle

    for rows, cols in [(33, 1024), (257, 4100)] if count < 70 else [(33, 1024)]:
        ws = [gaussian_outliers((rows, cols), std=0.02, p_outlier=0.0, gain=1.0, seed=i, dtype=torch.float32 if cols % 8 else torch.bfloat16)
              for i in range(count)]
        for i, w in enumerate(ws):
            w.view(-1)[-1 if i % 2 else 0] = 3.0 + i
        dev = [w.to(DEV) for w in ws]
        with launch.deferred():
            got = [quant_fp8(d, strategy) for d in dev]
        for w, result in zip(ws, got):
            _same(result, (oracle.channel_fp8 if strategy == "channel" else oracle.tensor_fp8)(w), f"{strategy} {rows} x {cols}")


def test_a_recorded_list_runs_them_at_once():
    """A list that is kept for later runs does not hold them: they run when they are called, and the list says so."""
    from oracle import mq_oracle as oracle

    w = gaussian_outliers((24, 100), std=0.02, p_outlier=0.01, gain=20.0, seed=5)
    d = w.to(DEV)
    with launch.recording() as batch:
        got = quant_fp8(d, "channel")
        _same(got, oracle.channel_fp8(w), "channel")
    assert len(batch) == 0 and batch.direct_calls == 1
