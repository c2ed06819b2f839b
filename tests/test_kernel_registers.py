"""Registers of kernels whose speed hangs on how many workgroups share a compute unit, as the built library states them."""

import struct

import msgpack

from miles_amd import _lib


def _vgprs() -> dict[str, int]:
    """Vector registers of every kernel, from the notes of the code objects inside the library."""
    data = open(_lib.lib_path(), "rb").read()
    out, at = {}, data.find(b"AMDGPU\0")
    while at >= 0:
        name_size, size, kind = struct.unpack_from("<III", data, at - 12)
        if (name_size, kind) == (7, 32):        # NT_AMDGPU_METADATA
            for k in msgpack.unpackb(data[at + 8:at + 8 + size], strict_map_key=False)["amdhsa.kernels"]:
                out[k[".name"]] = k[".vgpr_count"]
        at = data.find(b"AMDGPU\0", at + 1)
    return out


def test_tile_kernels_leave_room_for_four_workgroups():
    """512 lanes are two wavefronts on each SIMD: with more than 64 registers three workgroups fit a compute unit, with more
    than 80 only two."""
    tiles = {name: n for name, n in _vgprs().items() if "fp8_block128_any_kernel" in name}
    assert len(tiles) == 12 and max(tiles.values()) <= 64, tiles
