"""Forms of a call that the host layer does not take itself: each is answered, or refused, as the Python path does it."""

import pytest
import torch

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
