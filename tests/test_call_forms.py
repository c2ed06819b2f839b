"""Forms of a call that the host layer does not take itself: each is answered, or refused, as the Python path does it."""

import threading

import pytest
import torch

from miles_amd import launch
from miles_amd._host import native
from miles_amd.kernels.quant import fp8_act_quant as aq
from miles_amd.kernels.quant import nvfp4_qdq as nq


@pytest.mark.parametrize("weights", [(), (torch.zeros(16, 16),), iter([]), None, 7],
                         ids=["empty", "tuple", "iterator", "none", "number"])
def test_what_is_no_list_of_weights_is_handed_back(weights):
    assert native.nvfp4_images(weights, 16, 256, 448, 0) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_tuple_of_weights_is_taken_like_a_list(dtype):
    weights = [torch.randn(rows, 96, device="cuda").to(dtype).requires_grad_(rows != 5) for rows in (33, 5, 64)]
    config = nq.NVFP4QDQConfig()
    images, want = (nq.fake_nvfp4_quantization_ste_list(form(weights), config) for form in (tuple, list))
    for w, image, ref in zip(weights, images, want, strict=True):
        assert torch.equal(image.view(torch.int16), ref.view(torch.int16)) and image.requires_grad == w.requires_grad
        if w.requires_grad:
            assert torch.equal(torch.autograd.grad(image, w, ref.detach())[0], ref.detach())
    assert nq.fake_nvfp4_quantization_ste_list((), config) is None


@pytest.mark.gpu
@pytest.mark.parametrize("block", [64, True, 1 << 70, 64.0, "64", None], ids=repr)
def test_the_block_size_is_taken_or_refused_as_in_python(block):
    x = torch.randn(8, 256, device="cuda").bfloat16()

    def answer(call):
        try:
            return call(x, block).view(torch.int16).tolist()
        except Exception as e:
            return type(e)

    assert answer(aq.fp8_simulate_qat) == answer(aq.DeepSeekV4LinearQATFunc.apply)


def test_deferred_decorates_a_function():
    """Every call has a block of its own: calls inside join it, threads do not, and it is gone afterwards."""
    @launch.deferred()
    def call(depth, seen):
        batch = launch.active_batch()
        seen.append(batch)
        if depth:
            call(depth - 1, seen)
        if depth == 7:
            raise KeyError
        assert launch.active_batch() is batch
        return len(batch)

    seen = []
    assert call.__name__ == "call" and call(1, seen) == 0 and call(0, seen) == 0
    assert seen[0] is seen[1] is not seen[2] and None not in seen and launch.active_batch() is None
    with pytest.raises(KeyError):
        call(7, [])
    assert launch.active_batch() is None
    both = threading.Barrier(2, timeout=30)
    found = []

    @launch.deferred()
    def meet():
        both.wait()
        found.append(launch.active_batch())
        both.wait()

    threads = [threading.Thread(target=meet) for _ in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert len(found) == 2 and found[0] is not found[1] and None not in found


def test_a_deferred_block_is_entered_once():
    block = launch.deferred()
    with block as outer:
        with pytest.raises((RuntimeError, AttributeError)), block:
            pass
        assert launch.active_batch() is outer
    assert launch.active_batch() is None
    with pytest.raises((RuntimeError, AttributeError)), block:
        pass
    assert launch.active_batch() is None
