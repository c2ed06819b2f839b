"""Jobs that the driver refuses before anything is launched: no GPU is needed to see the answer."""

import ctypes

import pytest

from miles_amd import _lib

MQ_ERR_ARG = -1
KINDS = [_lib.JOB_MXFP8, _lib.JOB_FP8_BLOCK, _lib.JOB_FP8_BLOCKWISE_CAST, _lib.JOB_FP8_BLOCK_POW2]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dtype", [-1, 3, 7])
def test_unknown_dtype(kind, dtype):
    block = 128 if kind != _lib.JOB_MXFP8 else 0
    # (addresses that are aligned for every kernel and never read)
    job = (_lib.Job * 1)(_lib.Job(kind, dtype, 1 << 20, 1 << 21, 1 << 22, None, None, 256, 256, 256, block, block, 0, 0))
    assert _lib.load().mq_run_jobs(ctypes.byref(job), 1, None) == MQ_ERR_ARG
