"""Jobs that the driver refuses before anything is launched: no GPU is needed to see the answer."""

import ctypes

import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.utils import nvfp4

MQ_ERR_ARG = -1
KINDS = [_lib.JOB_MXFP8, _lib.JOB_FP8_BLOCK, _lib.JOB_FP8_BLOCKWISE_CAST, _lib.JOB_FP8_BLOCK_POW2]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dtype", [-1, 3, 7])
def test_unknown_dtype(kind, dtype):
    block = 128 if kind != _lib.JOB_MXFP8 else 0
    assert _run(kind, dtype, 256, 256, block, block) == MQ_ERR_ARG


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


def _stacked(n, rows, cols):
    return (torch.zeros(n, rows, cols // 2, dtype=torch.uint8), torch.zeros(n, rows, cols // 16, dtype=torch.float8_e4m3fn), torch.zeros(n))


@pytest.mark.parametrize("wrong", range(4))
def test_outputs_of_a_stack(wrong):
    """Stacked outputs are checked like a single matrix's, and a slice of them serves its own matrix only."""
    stack, (codes, scales, top) = torch.zeros(3, 8, 32), _stacked(3, 8, 32)
    if wrong == 0:
        codes = codes[:, :4]
    elif wrong == 1:
        scales = scales[:, :, :1]
    elif wrong == 2:
        top = top[:2]
    else:
        codes = codes.transpose(0, 1).contiguous().transpose(0, 1)
    with pytest.raises(ValueError, match="shaped like the results"):
        next(nvfp4.stack_slices(stack, codes, scales, top))


@pytest.mark.gpu
def test_a_slice_of_a_stack_serves_its_own_matrix():
    stack = torch.zeros(3, 8, 32, device="cuda", dtype=torch.bfloat16)
    _matrix, out = next(nvfp4.stack_slices(stack, *(t.cuda() for t in _stacked(3, 8, 32))))
    with pytest.raises(ValueError, match="another matrix"):
        nvfp4.nvfp4_quantize_1d(torch.zeros(16, 32, device="cuda", dtype=torch.bfloat16), out=out)


@pytest.mark.gpu
@pytest.mark.parametrize("shape, error", [((16,), IndexError), ((2, 16, 32), ValueError), ((16, 24), ValueError)])
def test_nvfp4_weights_of_another_rank(shape, error):
    with pytest.raises(error):
        nvfp4.nvfp4_quantize_1d(torch.zeros(shape, device="cuda", dtype=torch.bfloat16))


@pytest.mark.parametrize("dtype, cols, p1, workspace, rows_per_block", [
    (3, 64, 1, True, 0), (-1, 64, 0, True, 0), (0, 64, 2, True, 0), (0, 64, 1, True, 128), (0, 64, 0, False, 0), (0, 7, 1, False, 0),
    (2, 3, 1, False, 0), (2, 16388, 1, False, 0)])
def test_scaled_fp8_jobs(dtype, cols, p1, workspace, rows_per_block):
    """An unknown dtype or flag, row blocks, and a missing workspace where a row is not held in registers."""
    keep, inp, out, scale = _addresses(1 << 16)
    aux = scale if workspace else None
    job = (_lib.Job * 1)(_lib.Job(_lib.JOB_FP8_SCALED, dtype, inp, out, scale, aux, None, 2, cols, cols, 0, p1, rows_per_block, 0))
    assert _lib.load().mq_run_jobs(ctypes.byref(job), 1, None) == MQ_ERR_ARG


def test_the_native_layer_leaves_host_tensors_to_python():
    """Not on the GPU: every entry of the native layer hands the call back."""
    from miles_amd._host import native

    x = torch.zeros(4, 32, dtype=torch.bfloat16)
    assert native.submit(_lib.JOB_MXFP8, None, x, x, x, None, None, 4, 32, 32, 0, 0, 0, 0) is False
    assert native.produce(_lib.JOB_MXFP8, None, x, None, 4, 32, 32, 0, 0, (torch.uint8, 4, 32), (torch.uint8, 4, 1), None, None) is None
    assert native.act_quant(x, 32, 0, torch.float32) is None and native.fake_quant(x, 0, 32) is None
    assert native.simulate(x, 32, 0) is None and native.nvfp4_images([x], 16, 256, 448, 0) is None
    assert native.nvfp4_images([None], 16, 256, 448, 0) is None and native.fake_quant(None, 0, 32) is None
    with launch.deferred() as batch:
        assert len(batch) == 0 and batch.records == []
