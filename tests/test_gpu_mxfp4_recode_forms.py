"""MXFP4 -> FP8 lists on both sides of the size from which they take the flat form instead of the tile form (2^25 elements)."""

import pytest
import torch

from miles_amd import launch
from miles_amd.tools.convert_mxfp4_to_fp8 import cast_e2m1fn_to_e4m3fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    [(128, 128), (256, 384)],
    [(4096, 4096), (4096, 4096)],                       # 2^25 elements: the tile form still
    [(4096, 4096), (4096, 4096), (128, 128)],           # past it
    [(33024, 128), (128, 33024), (5120, 5120)],         # one tile a row, more tiles a row than a wavefront has lanes
])
def test_recode_list(shapes, oracle):
    g = torch.Generator().manual_seed(len(shapes) + shapes[0][0])
    ins = []
    for out_dim, in_dim in shapes:
        packed = torch.randint(0, 256, (out_dim, in_dim // 2), dtype=torch.uint8, generator=g)
        scale = torch.randint(110, 135, (out_dim, in_dim // 32), dtype=torch.uint8, generator=g)
        scale.view(-1)[-1] = 255                        # E8M0's NaN in the last tile
        ins.append((packed.view(torch.int8), scale.view(torch.float8_e8m0fnu)))
    with launch.deferred():
        outs = [cast_e2m1fn_to_e4m3fn(p.cuda(), s.cuda()) for p, s in ins]
    for (p, s), (y, ts) in zip(ins, outs):
        y_o, ts_o = oracle.cast_e2m1fn_to_e4m3fn(p, s)
        assert torch.equal(ts.cpu().view(torch.int32), ts_o.view(torch.int32))
        assert torch.equal(y.cpu().view(torch.uint8), y_o.view(torch.uint8))
