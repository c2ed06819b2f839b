"""Copy jobs in launches over a device table."""

import numpy as np
import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.utils.mxfp8 import mxfp8_quantize

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _copy(batch, src, dst, rows, cols, src_pitch=0, dst_pitch=0):
    batch.add(_lib.JOB_COPY, 0, src, dst, None, None, None, rows, cols, src_pitch, 0, 0, 0, dst_pitch)


@pytest.mark.parametrize("order", ["ascending", "scattered", "dependent"])
def test_copy_jobs_over_a_device_table(order):
    """More short copies than a launch's arguments hold, in a batch that has a table: byte counts around the 16-byte units and
    the 16 KiB chunks, any alignment, rows with a pitch; and jobs that read or overwrite what an earlier one touched."""
    sizes = [1, 7, 8, 15, 16, 17, 31, 255, 4095, 4096, 16383, 16384, 16385, 40000, 65536]
    rng = np.random.default_rng(3)
    memory = torch.from_numpy(rng.integers(0, 256, 8 << 20, dtype=np.uint8)).to(DEV)
    base, half = memory.data_ptr(), 4 << 20
    small = torch.randn(70, 32, 64, device=DEV).bfloat16()
    with launch.recording() as batch:
        for w in small:
            mxfp8_quantize(w)
    batch.device = memory.device
    jobs, at = [], 0                            # (source offset, destination offset, rows, cols, source pitch, destination pitch)
    for i in range(150):
        n = sizes[i % len(sizes)] if i % 7 else 24
        src = int(rng.integers(0, half - 70000))
        src += -src % 16 if i % 2 else 0
        if i % 11 == 10:                        # rows of a matrix
            jobs.append((src, half + at, 5, 24, 40, 32))
            at += 5 * 32
        else:
            jobs.append((src, half + at, 1, n, n, 0))
            at += n
        at += -at % 16 if i % 3 else 0
    if order == "scattered":
        jobs = [jobs[i] for i in rng.permutation(len(jobs))]
    if order == "dependent":
        jobs[40] = (jobs[12][1], jobs[40][1], 1, 16, 16, 0)            # reads what job 12 writes
        jobs[90] = (jobs[90][0], jobs[85][0], 1, 32, 32, 0)            # overwrites the source of job 85
        jobs[120] = (jobs[120][0], jobs[119][1] + 1, 1, 9, 9, 0)       # and the destination of job 119
    for src, dst, rows, cols, sp, dp in jobs:
        _copy(batch, base + src, base + dst, rows, cols, sp, dp)
    want = memory.cpu().numpy().copy()
    for _ in range(2):
        for src, dst, rows, cols, sp, dp in jobs:
            for r in range(rows):
                want[dst + r * dp:dst + r * dp + cols] = want[src + r * sp:src + r * sp + cols].copy()
        batch.run()
        assert batch._table is not None
        assert np.array_equal(memory.cpu().numpy(), want)
