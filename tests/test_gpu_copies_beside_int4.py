"""Copies behind INT4 jobs in one list: those that depend on nothing share a launch with them, and whatever the order and the
overlaps, memory ends as if the jobs had run one after the other."""

import ctypes

import numpy as np
import pytest
import torch

from miles_amd import _lib, launch
from miles_amd.kernels.quant.int4_fake import pack_layer

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
ROWS, COLS, GROUP = 16, 512, 128
SIZES = [16, 8, 1, 17, 255, 4096, 16384, 16400, 40001, 65536]


@pytest.mark.parametrize("order", ["apart", "descending", "reads_codes", "reads_scales", "overwrites_codes", "overwrites_input", "reads_a_copy", "long"])
@pytest.mark.parametrize("n, table", [(1, False), (5, False), (64, False), (70, True)])
@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_as_if_one_after_the_other(dtype, symmetric, n, table, order):
    rng = np.random.default_rng(n)
    size = torch.tensor([], dtype=dtype).element_size()
    w = torch.randn(n, ROWS, COLS, device=DEV, generator=torch.Generator(device=DEV).manual_seed(n)).to(dtype)
    numel, groups = ROWS * COLS, ROWS * COLS // GROUP
    nbytes = {"in": numel * size, "out": numel // 2, "scale": groups * size, "aux": groups, "aux2": groups // 2}
    fields = ("out", "scale") if symmetric else ("out", "scale", "aux", "aux2")
    # the payload: codes, scales (zero points) and a record of every tensor, each 16-byte aligned; inputs and sources behind it
    at, place, copies = 0, [], []
    for i in range(n):
        mine = {}
        for f in fields:
            mine[f], at = at, at + nbytes[f] + -nbytes[f] % 16
        length = SIZES[i % len(SIZES)] if order != "long" else 65537
        copies.append([0, at, length])
        at += length + -length % 16
        place.append(mine)
    for mine in place:
        mine["in"], at = at, at + nbytes["in"]
    for c in copies:
        c[0], at = at, at + c[2] + 3                    # (sources at any alignment)
    if order == "descending":
        copies.reverse()
    elif order == "reads_codes":
        copies[n // 2][0] = place[-1]["out"] + 5
        copies[n // 2][2] = min(copies[n // 2][2], 64)
    elif order == "reads_scales":
        copies[-1][0], copies[-1][2] = place[0]["scale"], min(copies[-1][2], 16)
    elif order == "overwrites_codes":
        copies[0][1], copies[0][2] = place[-1]["out"] + 3, 9
    elif order == "overwrites_input":
        copies[n // 2][1], copies[n // 2][2] = place[-1]["in"] + 32, min(copies[n // 2][2], 64)
    elif order == "reads_a_copy":
        copies[-1][0], copies[-1][2] = copies[0][1], min(copies[0][2], copies[-1][2])
    memory = torch.from_numpy(rng.integers(0, 256, at + 64, dtype=np.uint8)).to(DEV)
    for i, mine in enumerate(place):
        memory[mine["in"]:mine["in"] + nbytes["in"]] = w[i].reshape(-1).view(torch.uint8)
    base = memory.data_ptr()
    with launch.recording() as batch:
        pass
    batch.device = memory.device
    for mine in place:
        batch.add(_lib.JOB_INT4_PACK if symmetric else _lib.JOB_INT4_PACK_ASYM, _lib.DTYPE_CODE[dtype], base + mine["in"],
                  *(base + mine[f] if f in mine else None for f in ("out", "scale", "aux", "aux2")), ROWS, COLS, COLS, GROUP, 0)
    for src, dst, length in copies:
        batch.add(_lib.JOB_COPY, 0, base + src, base + dst, None, None, None, 1, length, length, 0, 0)
    want = memory.cpu().numpy().copy()
    for i, mine in enumerate(place):
        packed, scale, zp = pack_layer(w[i], GROUP, symmetric)
        for f, t in (("out", packed), ("scale", scale), ("aux2", zp)):
            if f in mine:
                got = t.contiguous().reshape(-1).view(torch.uint8).cpu().numpy()
                want[mine[f]:mine[f] + got.size] = got
    for src, dst, length in copies:
        want[dst:dst + length] = want[src:src + length].copy()
    batch.run()
    assert (batch._table is not None) == table
    got = memory.cpu().numpy()
    if not symmetric:                                   # the unpacked zero points are the packer's own business
        for mine in place:
            got[mine["aux"]:mine["aux"] + nbytes["aux"]] = want[mine["aux"]:mine["aux"] + nbytes["aux"]]
    assert np.array_equal(got, want)


def _launches(batch):
    """Kernels of one run, counted in a capture of it."""
    nodes = _lib.load().hipGraphGetNodes        # (resolved in the HIP runtime that the library is linked against)
    nodes.restype, nodes.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        batch.run()
    count = ctypes.c_size_t()
    assert nodes(graph.raw_cuda_graph(), None, ctypes.byref(count)) == 0
    return count.value


# 32768 workgroups of tensors and more have the copies behind them; grid rows far wider than the copies need
@pytest.mark.parametrize("n, rows, table", [(15, 2048, False), (16, 2048, False), (17, 2048, False), (64, 1008, False), (70, 1008, True)])
def test_copies_behind_a_long_launch(n, rows, table):
    cols = 4096
    g = torch.Generator(device=DEV).manual_seed(n)
    w = torch.randn(n, rows, cols, device=DEV, generator=g).bfloat16()
    lengths = [SIZES[i % len(SIZES)] for i in range(n)]
    at, place = 0, []
    for length in lengths:                              # codes, scales and a record of every tensor, as in a packed payload
        mine = {}
        for name, size in (("out", rows * cols // 2), ("scale", rows * cols // GROUP * 2), ("copy", length)):
            mine[name], at = at, at + size + -size % 16
        place.append(mine)
    payload = torch.full((at,), 0xA5, dtype=torch.uint8, device=DEV)
    sources = torch.randint(0, 256, (n, max(SIZES) + 1), dtype=torch.uint8, device=DEV, generator=g)
    want = payload.clone()
    for mine, length, one, source in zip(place, lengths, w, sources):
        packed, scale, _ = pack_layer(one, GROUP)
        for name, t in (("out", packed), ("scale", scale), ("copy", source[:length])):
            t = t.reshape(-1).view(torch.uint8)
            want[mine[name]:mine[name] + t.numel()] = t
    with launch.recording() as batch:
        pass
    batch.device = payload.device
    base = payload.data_ptr()
    for mine, one in zip(place, w):
        batch.add(_lib.JOB_INT4_PACK, _lib.DTYPE_CODE[torch.bfloat16], one.data_ptr(), base + mine["out"], base + mine["scale"], None, None,
                  rows, cols, cols, GROUP, 0)
    for mine, length, source in zip(place, lengths, sources):
        batch.add(_lib.JOB_COPY, 0, source.data_ptr(), base + mine["copy"], None, None, None, 1, length, length, 0, 0)
    batch.freeze()
    assert (batch._table is not None) == table
    torch.cuda.synchronize()
    assert _launches(batch) == 1
    payload.fill_(0xA5)
    batch.run()
    assert torch.equal(payload, want)
