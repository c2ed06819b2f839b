"""The native host layer: the same jobs, in the order of the calls, and the same graph nodes as the Python path makes."""

import threading

import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.kernels.quant import fake_quant as fq
from miles_amd.kernels.quant import fp8_act_quant as aq
from miles_amd.kernels.quant import nvfp4_qdq as nq
from miles_amd.kernels.quant.int4_fake import fake_int4_quant_cuda, pack_layer
from miles_amd.tools.convert_hf_to_fp8 import quant_fp8
from miles_amd.tools.fp8_cast_bf16 import weight_dequant
from miles_amd.utils.mxfp8 import mxfp8_quantize

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
CONFIG = nq.NVFP4QDQConfig()


class Tagged(torch.Tensor):
    """A subclass: never taken by the native layer."""


def _x(*shape, dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV).to(dtype)


STRAIGHT = {
    "fp8": (fq.fake_quant_fp8, lambda x: fq._IdentityGradient.apply(x, fq.fake_quant_fp8_forward)),
    "fp4": (fq.fake_quant_fp4, lambda x: fq._IdentityGradient.apply(x, fq.fake_quant_fp4_forward)),
    "kv": (fq.fake_quant_compressed_kv, lambda x: fq._IdentityGradient.apply(x, fq.fake_quant_compressed_kv_forward)),
    "simulate": (lambda x: aq.fp8_simulate_qat(x, 64), lambda x: aq.DeepSeekV4LinearQATFunc.apply(x, 64)),
    "simulate_128": (aq.fp8_simulate_qat, aq.DeepSeekV4LinearQATFunc.apply),
    "nvfp4": (lambda x: nq.fake_nvfp4_quantization_ste(x, CONFIG),
              lambda x: nq._QDQStraightThrough.apply(x, iter(nq._images([x], CONFIG)))),
}


@pytest.mark.parametrize("name", sorted(STRAIGHT))
def test_nodes_hand_the_gradient_through(name):
    native, python = STRAIGHT[name]
    x = _x(48, 256).requires_grad_(True)
    y, ref = native(x), python(x)
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16)) and y.grad_fn is not None and not y.is_leaf
    gy = _x(48, 256, seed=1)
    assert torch.equal(torch.autograd.grad(y, x, gy, retain_graph=True)[0], gy)
    assert torch.equal(torch.autograd.grad(y, x, gy)[0], gy)
    # through a double backward, as the identity it is
    first = torch.autograd.grad((native(x).float() ** 3).sum(), x, create_graph=True)[0]
    again = torch.autograd.grad((python(x).float() ** 3).sum(), x, create_graph=True)[0]
    assert torch.equal(first, again)
    assert torch.equal(torch.autograd.grad(first.float().sum(), x)[0], torch.autograd.grad(again.float().sum(), x)[0])
    # hooks and an undefined gradient from downstream, which counts as zeros
    seen = []

    class Drops(torch.autograd.Function):
        @staticmethod
        def forward(ctx, a):
            return a.clone()

        @staticmethod
        def backward(ctx, g):
            return None

    for f in (native, python):
        z = f(x)
        z.register_hook(lambda g: seen.append(None if g is None else g.abs().sum().item()))
        grad = torch.autograd.grad(z.float().sum(), x)[0]
        dropped = torch.autograd.grad(Drops.apply(f(x)).float().sum(), x, allow_unused=True)[0]
        seen.append((grad.abs().sum().item(), None if dropped is None else dropped.abs().sum().item()))
    assert seen[:2] == seen[2:]
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            a, b = native(x), python(x)
        assert (a.requires_grad, a.grad_fn, a.is_inference()) == (b.requires_grad, b.grad_fn, b.is_inference())
    plain = native(x.detach())
    assert plain.grad_fn is None and not plain.requires_grad


@pytest.mark.parametrize("name", sorted(STRAIGHT))
def test_what_is_not_ordinary_takes_the_python_path(name):
    """Transforms, forward mode and subclasses: whatever the Python function answers, a refusal or a result."""
    import torch.autograd.forward_ad as fwAD

    native, python = STRAIGHT[name]

    def answer(call):
        try:
            out = call()
        except Exception as e:
            return type(e), str(e).split("\n")[0][:60]
        return type(out), out.as_subclass(torch.Tensor).detach().cpu().view(torch.int16).tolist()

    x = _x(4, 128)

    def dual(f):
        with fwAD.dual_level():
            return f(fwAD.make_dual(x, x))

    for how in (lambda f: torch.func.grad(lambda a: f(a).float().sum())(x), lambda f: torch.func.vmap(f)(torch.stack([x, x])),
                lambda f: torch.func.jvp(f, (x,), (x,))[0], dual, lambda f: f(x.as_subclass(Tagged))):
        assert answer(lambda: how(native)) == answer(lambda: how(python))


def test_jobs_keep_the_order_of_the_calls():
    """Jobs recorded in native code, from Python and by hand in one block: each reads what the one before wrote."""
    w = _x(256, 384)
    with launch.deferred() as batch:
        q, s = quant_fp8(w, "block", [128, 128])
        back = weight_dequant(q, s)
        tagged = mxfp8_quantize(back.as_subclass(Tagged))                 # recorded from Python
        copy = torch.empty_like(back)
        batch.add(_lib.JOB_COPY, 0, back.data_ptr(), copy.data_ptr(), None, None, None, 1, back.numel() * 2, back.numel() * 2, 0, 0)
        packed = pack_layer(copy, 128)
        assert len(batch) == 5
        kinds = [r[batch.KIND] for r in batch.records]
        last = mxfp8_quantize(copy)
        assert len(batch) == 6
    assert kinds == [_lib.JOB_FP8_BLOCK, _lib.JOB_FP8_DEQUANT, _lib.JOB_MXFP8, _lib.JOB_COPY, _lib.JOB_INT4_PACK]
    q1, s1 = quant_fp8(w, "block", [128, 128])
    b1 = weight_dequant(q1, s1)
    for have, want in [*zip((q, s, back), (q1, s1, b1)), *zip(tagged, mxfp8_quantize(b1)), *zip(packed[:2], pack_layer(b1, 128)[:2]),
                       *zip(last, mxfp8_quantize(b1))]:
        assert torch.equal(have.view(torch.uint8), want.view(torch.uint8))


def test_a_block_left_by_an_exception_submits_nothing_and_nested_blocks_join():
    w = _x(128, 128)
    with pytest.raises(KeyError), launch.deferred():
        quant_fp8(w, "block", [128, 128])
        raise KeyError
    assert launch.active_batch() is None
    with launch.deferred() as outer:
        with launch.deferred() as inner:
            q, s = quant_fp8(w, "block", [128, 128])
        assert inner is outer and len(outer) == 1
    assert torch.equal(weight_dequant(q, s).float(), weight_dequant(*quant_fp8(w, "block", [128, 128])).float())


def test_threads_have_lists_and_streams_of_their_own():
    weights = {i: _x(256, 512, seed=i) for i in range(4)}
    want = {i: [t.clone() for t in mxfp8_quantize(w * 2)] for i, w in weights.items()}
    torch.cuda.synchronize()
    got, errors = {}, []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                w = weights[i] * 2
                for _ in range(20):
                    with launch.deferred() as batch:
                        got[i] = mxfp8_quantize(w)
                    assert len(batch) == 1
                x = w.detach().requires_grad_(True)
                assert torch.equal(torch.autograd.grad(fq.fake_quant_fp4(x), x, w)[0], w)
            stream.synchronize()
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in weights]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors
    for i, pair in got.items():
        for have, ref in zip(pair, want[i]):
            assert torch.equal(have.view(torch.uint8), ref.view(torch.uint8))


def test_calls_inside_a_list_are_counted_and_run_at_once():
    x = _x(16, 256)
    want = [t.clone() for t in aq.act_quant(x, 128, "ue8m0")] + [fq.fake_quant_fp8(x).clone(), fake_int4_quant_cuda(x, (1, 128), True)[0].clone()]
    for block in (launch.deferred, launch.recording):
        with block() as batch:
            got = [*aq.act_quant(x, 128, "ue8m0"), fq.fake_quant_fp8(x), fake_int4_quant_cuda(x, (1, 128), True)[0]]
            assert batch.direct_calls == 3 and len(batch) == 0
        for have, ref in zip(got, want):
            assert torch.equal(have.view(torch.uint8), ref.view(torch.uint8))


def test_a_refused_job_raises_the_library_error():
    x = _x(16, 250)
    with pytest.raises(_lib.MilesQuantError):
        launch.produce(_lib.JOB_MXFP8, x, 16, 250, 250, 0, 0, (torch.uint8, 16, 250), (torch.uint8, 16, 8))
    with pytest.raises(_lib.MilesQuantError), launch.deferred():
        launch.produce(_lib.JOB_MXFP8, x, 16, 250, 250, 0, 0, (torch.uint8, 16, 250), (torch.uint8, 16, 8))
    assert launch.active_batch() is None
