"""Whole quantizers of the native layer: the job, the outputs and their forms are those of the Python function that goes on where
the native one hands a call back."""

import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.kernels.quant import int4_fake
from miles_amd.megatron_to_hf.processors import quantizer_nvfp4
from miles_amd.tools import convert_hf_to_fp8, convert_kimi_int4_to_bf16, convert_mxfp4_to_fp8, fp8_cast_bf16
from miles_amd.utils import mxfp4, mxfp8

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
MODULES = (int4_fake, quantizer_nvfp4, convert_hf_to_fp8, convert_kimi_int4_to_bf16, convert_mxfp4_to_fp8, fp8_cast_bf16, mxfp4, mxfp8)
WHOLE = ("block_fp8", "scaled_fp8", "mxfp8", "mxfp4", "int4", "fp8_dequant", "mxfp4_dequant", "fp8_to_mxfp8", "mxfp4_to_fp8", "int4_unpack",
         "nvfp4_stack")


class _HandsBack:
    """The native layer with its whole quantizers handing every call back."""

    def __init__(self, native):
        self._native = native

    def __getattr__(self, name):
        return (lambda *a: None) if name in WHOLE else getattr(self._native, name)


class _Counts:
    def __init__(self, native, seen):
        self._native, self._seen = native, seen

    def __getattr__(self, name):
        f = getattr(self._native, name)
        if name not in WHOLE:
            return f

        def call(*a):
            out = f(*a)
            self._seen.append(out is not None)
            return out

        return call


def _w(*shape, dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV).to(dtype)


def _fp8(rows, cols):
    return convert_hf_to_fp8.quant_fp8(_w(rows, cols), "block", [128, 128])


def _fp4(rows, cols, as_int8=False):
    q, s = mxfp4.quantize_mxfp4(_w(rows, cols), 32)
    return (q.view(torch.int8) if as_int8 else q), s


def _int4(rows, cols, dtype=torch.bfloat16):
    q, s, _ = int4_fake.pack_layer(_w(rows, cols, dtype=dtype), 32)
    return q, s


BLOCK = lambda w: convert_hf_to_fp8.quant_fp8(w, "block", [128, 128])  # noqa: E731
# name -> (quantizer, its arguments, whether the native layer takes them)
CASES = {}
for _dtype in (torch.bfloat16, torch.float16, torch.float32):
    _n = str(_dtype)[6:]
    CASES.update({
        f"block_{_n}": (BLOCK, lambda d=_dtype: (_w(200, 300, dtype=d),), True),
        f"block_rows_apart_{_n}": (BLOCK, lambda d=_dtype: (_w(130, 520, dtype=d)[:, 3:260],), True),
        f"block_one_row_{_n}": (BLOCK, lambda d=_dtype: (_w(1, 77, dtype=d),), True),
        f"channel_{_n}": (lambda w: convert_hf_to_fp8.quant_fp8(w, "channel"), lambda d=_dtype: (_w(37, 264, dtype=d),), True),
        f"channel_short_{_n}": (lambda w: convert_hf_to_fp8.quant_fp8(w, "channel"), lambda d=_dtype: (_w(300, 3, dtype=d),), True),
        f"channel_wide_{_n}": (lambda w: convert_hf_to_fp8.quant_fp8(w, "channel"), lambda d=_dtype: (_w(3, 32776, dtype=d),), True),
        f"tensor_{_n}": (lambda w: convert_hf_to_fp8.quant_fp8(w, "tensor"), lambda d=_dtype: (_w(301, 129, dtype=d),), True),
        f"mxfp8_{_n}": (mxfp8.mxfp8_quantize, lambda d=_dtype: (_w(33, 96, dtype=d),), True),
        f"mxfp8_stack_{_n}": (mxfp8.mxfp8_quantize, lambda d=_dtype: (_w(2, 5, 64, dtype=d),), True),
        f"mxfp8_vector_{_n}": (mxfp8.mxfp8_quantize, lambda d=_dtype: (_w(64, dtype=d),), True),
        f"mxfp4_{_n}": (lambda w: mxfp4.quantize_mxfp4(w, 32), lambda d=_dtype: (_w(33, 96, dtype=d),), True),
        f"int4_{_n}": (lambda w: int4_fake.pack_layer(w, 32), lambda d=_dtype: (_w(33, 96, dtype=d),), True),
        f"int4_asym_{_n}": (lambda w: int4_fake.pack_layer(w, 32, False), lambda d=_dtype: (_w(16, 96, dtype=d),), True),
        f"int4_unpack_{_n}": (lambda q, s: convert_kimi_int4_to_bf16._dequantize_tensor(q, s, (24, 96), 32), lambda d=_dtype: _int4(24, 96, d), True),
        f"nvfp4_stack_{_n}": (quantizer_nvfp4.quantize_nvfp4, lambda d=_dtype: (_w(3, 17, 48, dtype=d),), True),
    })
CASES.update({
    "fp8_dequant": (fp8_cast_bf16.weight_dequant, lambda: _fp8(200, 300), True),
    "mxfp4_dequant": (lambda q, s: mxfp4.dequantize_mxfp4(q, s, 32), lambda: _fp4(7, 96), True),
    "mxfp4_dequant_stack": (lambda q, s: mxfp4.dequantize_mxfp4(q, s, 32), lambda: tuple(t.view(2, 3, -1) for t in _fp4(6, 96)), True),
    "fp8_to_mxfp8": (mxfp8.requantize_fp8_block_to_mxfp8, lambda: _fp8(130, 288), True),
    "mxfp4_to_fp8": (convert_mxfp4_to_fp8.cast_e2m1fn_to_e4m3fn, lambda: _fp4(256, 384, True), True),
    # forms that go back to Python
    "block_transposed": (BLOCK, lambda: (_w(300, 200).t(),), False),
    "mxfp8_rows_apart": (mxfp8.mxfp8_quantize, lambda: (_w(33, 192)[:, :96],), False),
    "int4_shape_tensor": (lambda q, s: convert_kimi_int4_to_bf16._dequantize_tensor(q, s, torch.tensor([24, 96]), 32), lambda: _int4(24, 96), False),
    "nvfp4_stack_apart": (quantizer_nvfp4.quantize_nvfp4, lambda: (_w(3, 17, 96)[:, :, :48],), False),
})


@pytest.mark.parametrize("name", sorted(CASES))
def test_the_same_job_and_outputs_as_the_python_path(name, monkeypatch):
    f, arguments, taken = CASES[name]
    args, native, seen = arguments(), launch.native, []
    results, records = [], []
    for layer in (_Counts(native, seen), _HandsBack(native)):
        for module in MODULES:
            monkeypatch.setattr(module, "native", layer)
        at_once = f(*args)
        with launch.deferred() as batch:
            got = f(*args)
            records.append([r[:batch.IN] + r[batch.ROWS:] + tuple(v is not None for v in r[batch.IN:batch.ROWS]) for r in batch.records])
        results.append([(at_once,) if torch.is_tensor(at_once) else at_once, (got,) if torch.is_tensor(got) else got])
    assert seen == [taken, taken]
    assert records[0] == records[1]
    for one, two in zip(*results):
        assert type(one) is type(two) and len(one) == len(two)
        for a, b in zip(one, two):
            assert (a is None) == (b is None)
            if a is not None:
                assert (a.shape, a.stride(), a.dtype, a.device, a.requires_grad) == (b.shape, b.stride(), b.dtype, b.device, b.requires_grad)
                assert torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8))


@pytest.mark.parametrize("name, error", [
    ("block", TypeError), ("block_zero", ZeroDivisionError), ("mxfp8", ValueError), ("mxfp4", AssertionError), ("int4", RuntimeError),
    ("asym", RuntimeError), ("dequant", AssertionError), ("cast", AssertionError), ("unpack", ValueError), ("nvfp4", ValueError)])
def test_refusals_are_worded_in_python(name, error):
    calls = {"block": lambda: convert_hf_to_fp8.block_fp8(_w(8, 8), None), "block_zero": lambda: convert_hf_to_fp8.block_fp8(_w(8, 8), [0, 1]),
             "mxfp8": lambda: mxfp8.mxfp8_quantize(_w(8, 40)), "mxfp4": lambda: mxfp4.quantize_mxfp4(_w(8, 40), 32),
             "int4": lambda: int4_fake.pack_layer(_w(8, 40), 32), "asym": lambda: int4_fake.pack_layer(_w(9, 64), 32, False),
             "dequant": lambda: fp8_cast_bf16.weight_dequant(_fp8(8, 64)[0].t(), _w(1, 1).float()),
             "cast": lambda: convert_mxfp4_to_fp8.cast_e2m1fn_to_e4m3fn(*_fp4(64, 128, True)),
             "unpack": lambda: convert_kimi_int4_to_bf16._dequantize_tensor(*_int4(24, 96), (24, 104), 32),
             "nvfp4": lambda: quantizer_nvfp4.quantize_nvfp4(_w(2, 3, 24))}
    with pytest.raises(error):
        calls[name]()


def test_a_recording_keeps_the_python_jobs():
    """Jobs of a list that its caller keeps: whole records that can be looked up by the tensors it holds."""
    stack = _w(3, 16, 64)
    with launch.recording() as batch:
        codes, _scales, published = quantizer_nvfp4.quantize_nvfp4(stack)
    assert len(batch.records) == 3 and len(batch.amax_records()) == 3
    batch.run()
    want = quantizer_nvfp4.quantize_nvfp4(stack)
    assert torch.equal(codes, want[0]) and torch.equal(published, want[2])


@pytest.mark.parametrize("n", [1, 3])
def test_records_of_a_deferred_stack(n):
    """A block that is submitted at its end: the records of a stack, which are one tensor, and of what was recorded beside it."""
    stack, single = _w(n * 16, 64).view(n, 16, 64), _w(8, 32)
    with launch.deferred() as batch:
        quantizer_nvfp4.quantize_nvfp4(stack)
        quantizer_nvfp4.quantize_nvfp4(single)
    records = batch.amax_records()
    assert [tuple(r.shape) for r in records] == [(_lib.RECORD_WORDS,)] * (n + 1)
    assert [r.data_ptr() for r in records] == [job[batch.AUX] for job in batch.records]
    assert [r[_lib.RECORD_AMAX_WORD].view(torch.float32).item() for r in records] == [w.abs().max().float().item() for w in (*stack, single)]
