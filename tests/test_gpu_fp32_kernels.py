"""fp32 instances of the tuned kernels against the oracle: sizes at the edges of a workgroup, special values, grouped
and recorded job lists."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def oracle():
    from oracle import mq_oracle as O

    return O


def _bits(t):
    t = t.cpu().contiguous()
    return t.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])


def _assert_same(got, want, what):
    g, w = _bits(got), _bits(want)
    assert g.shape == w.shape, f"{what}: shape {tuple(g.shape)} vs {tuple(w.shape)}"
    if not torch.equal(g, w):
        bad = (g != w).nonzero()
        i = tuple(bad[0].tolist())
        raise AssertionError(f"{what}: {bad.shape[0]} of {g.numel()} differ; first at {i}: got {g[i].item()} want {w[i].item()}")


def fp32_case(shape, seed, specials=False):
    """Values over forty binades with all 24 significant bits in use; optionally the format's extremes, subnormals,
    signed zeros, infinities and NaN strewn over them, and a row of zeros."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g) * torch.exp2(torch.randint(-20, 21, (shape[0], 1), generator=g).float())
    if specials:
        values = torch.tensor([0.0, -0.0, 1e-45, -1e-40, 1.1754944e-38, 3.4028235e38, -3.4028235e38, float("inf"),
                               -float("inf"), float("nan"), 448.0, 464.0, 2.0**-9, 6.0, 5.0000005, 2.5])
        at = torch.rand(shape, generator=g) < 0.004
        x = torch.where(at, values[torch.randint(0, len(values), shape, generator=g)], x)
        if shape[0] > 2:
            x[2] = 0
    return x


# one group, ragged last workgroups (a workgroup covers 2048 elements), several of them
FLAT_SHAPES = [(1, 32), (5, 96), (1, 2048), (1, 2080), (129, 2016), (3, 12288), (513, 1024)]


@pytest.mark.parametrize("shape", FLAT_SHAPES)
@pytest.mark.parametrize("specials", [False, True])
def test_mxfp8_fp32(oracle, shape, specials):
    from miles_amd.utils.mxfp8 import mxfp8_quantize

    w = fp32_case(shape, 10 + shape[1], specials)
    q, s = mxfp8_quantize(w.to(DEV))
    q_o, s_o = oracle.mxfp8_quantize(w)
    _assert_same(s, s_o, "scales")
    _assert_same(q, q_o, "codes")


def test_mxfp8_fp32_in_one_list_with_16_bit_tensors(oracle):
    """A recorded list of seventy tensors (more than the kernel arguments of a launch hold), run twice."""
    from miles_amd import launch
    from miles_amd.utils.mxfp8 import mxfp8_quantize

    tensors = [fp32_case((33, 160), 50 + i) for i in range(72)]
    tensors[5], tensors[6] = tensors[5].bfloat16(), tensors[6].half()
    dev = [t.to(DEV) for t in tensors]
    with launch.recording() as batch:
        outs = [mxfp8_quantize(t) for t in dev]
    batch.freeze()
    for rep in range(2):
        batch.run()
        torch.cuda.synchronize()
        for i, t in enumerate(tensors):
            for got, want, what in zip(outs[i], oracle.mxfp8_quantize(t), ("codes", "scales")):
                _assert_same(got, want, f"tensor {i} ({t.dtype}) {what}, run {rep}")
        for o in outs:
            for t in o:
                t.view(torch.uint8).fill_(0x5A)
