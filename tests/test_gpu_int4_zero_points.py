"""The packer of asymmetric INT4 zero points at the edges of its tiles."""

import pytest
import torch

from miles_amd import launch
from miles_amd.kernels.quant.int4_fake import pack_layer

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("rows", [8, 248, 256, 264, 520])
@pytest.mark.parametrize("groups", [1, 15, 16, 17, 31, 48])
def test_packed_zero_points_of_any_tile_remainder(rows, groups):
    from oracle import mq_oracle as oracle

    g = torch.Generator().manual_seed(1000 * rows + groups)
    # (groups shifted by different amounts: zero points of every value, clamped ones among them)
    weights = [((torch.rand(rows, groups, 32, generator=g) + torch.rand(rows, groups, 1, generator=g) * 1.4 - 1.2) * 0.02)
               .reshape(rows, groups * 32).bfloat16() for _ in range(3)]
    with launch.deferred():
        got = [pack_layer(w.to(DEV), 32, False) for w in weights]
    for w, result in zip(weights, got):
        for have, want in zip(result, oracle.pack_layer(w, 32, False)):
            assert torch.equal(have.cpu().view(torch.uint8), want.view(torch.uint8))
