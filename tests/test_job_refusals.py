"""Jobs that the driver refuses before anything is launched: no GPU is needed to see the answer."""

import ctypes

import pytest
import torch

from miles_amd import _lib, launch

MQ_ERR_ARG = -1
KINDS = [_lib.JOB_MXFP8, _lib.JOB_FP8_BLOCK, _lib.JOB_FP8_BLOCKWISE_CAST, _lib.JOB_FP8_BLOCK_POW2]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dtype", [-1, 3, 7])
def test_unknown_dtype(kind, dtype):
    block = 128 if kind != _lib.JOB_MXFP8 else 0
    # (addresses that are aligned for every kernel and never read)
    job = (_lib.Job * 1)(_lib.Job(kind, dtype, 1 << 20, 1 << 21, 1 << 22, None, None, 256, 256, 256, block, block, 0, 0))
    assert _lib.load().mq_run_jobs(ctypes.byref(job), 1, None) == MQ_ERR_ARG


def _addresses(nbytes):
    """Three buffers of `nbytes` that a job may name: real ones where a GPU is visible, so that a job which is not refused
    shows as a wrong answer and not as a fault; elsewhere numbers (aligned for every kernel) that nothing can read."""
    if not torch.cuda.is_available():
        return [None, 1 << 20, 1 << 21, 1 << 22]
    keep = torch.zeros(3, nbytes, dtype=torch.uint8, device="cuda")
    return [keep, *(row.data_ptr() for row in keep)]


def _run(kind, dtype, rows, cols, p0, p1=0):
    keep, inp, out, scale = _addresses(max(1 << 16, rows * cols * 8))
    record = torch.zeros(1280, dtype=torch.int32, device="cuda" if keep is not None else "cpu")
    job = (_lib.Job * 1)(_lib.Job(kind, dtype, inp, out, scale, record.data_ptr(), None, rows, cols, cols, p0, p1, 0, 0))
    return _lib.load().mq_run_jobs(ctypes.byref(job), 1, None)


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("rows, cols, group", [(1, 40, 32), (3, 16, 32), (5, 72, 32), (1, 33, 33), (3, 32, 64), (2, 32, 0)])
def test_mxfp4_element_counts(dtype, rows, cols, group):
    """Elements that are no whole number of groups, or odd in number: refused as mq_mxfp4_quant refuses them, whatever the
    dtype and however the job would have been launched."""
    assert _run(_lib.JOB_MXFP4, dtype, rows, cols, group) == MQ_ERR_ARG


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("flag", [1 << 5, 1 << 28, 1 << 29, 1 << 30, -(1 << 31)])
def test_nvfp4_unknown_flags(dtype, flag):
    """Bits that mq_nvfp4_quant does not know: refused for jobs as well, never handed on to a kernel's launcher."""
    assert _run(_lib.JOB_NVFP4, dtype, 16, 32, 448, flag) == MQ_ERR_ARG
    assert _run(_lib.JOB_NVFP4, dtype, 16, 32, 448, flag | _lib.NVFP4_CARRY_AMAX | _lib.NVFP4_4OVER6) == MQ_ERR_ARG


def test_tensors_off_the_gpu():
    """A job that names host memory never reaches a stream: neither by itself nor from a batch."""
    host = torch.zeros(32, 32, dtype=torch.bfloat16)
    out, scale = torch.zeros(32, 32, dtype=torch.uint8), torch.zeros(32, 1, dtype=torch.uint8)
    with pytest.raises(ValueError, match="cuda device"):
        _lib.stream_ptr(host.device)
    with pytest.raises(ValueError, match="cuda device"):
        launch.submit(_lib.JOB_MXFP8, host, out, scale, None, None, 32, 32, 32)
    with pytest.raises(ValueError, match="cuda device"), launch.deferred():
        launch.submit(_lib.JOB_MXFP8, host, out, scale, None, None, 32, 32, 32)
