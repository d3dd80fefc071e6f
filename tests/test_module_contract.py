"""Kernel argument lists of the code object, as its metadata states them.

Hosts that load particles_gfx950.hsaco by kernel name pass the argument lists of
the reference (particles.cu, fluids4.0/fluid_kernels.cu) and of the ranked path
(FX_CAP_RANKED in include/fluidsx_params.h); a kernel that takes more would
read past the end of their args[].
"""
import os
import struct

import msgpack
import pytest

from fluids3_amd.particles import CODE_OBJECT

# name -> argument sizes in bytes
PUBLISHED = {
    "insertParticles": [4],
    "prefixSum": [8, 8, 8, 4, 4],
    "prefixFixup": [8, 8, 4],
    "countingSortIndex": [4],
    "countingSortFull": [4],
    "countingSortFullRanked": [4],
    "computePressure": [4],
    "computeForce": [4],
    "advanceParticles": [4, 4, 4, 4],
    "emitParticles": [4, 4, 4],
    "sampleParticles": [8, 12, 12, 12, 4, 4],
}


def kernel_arguments(path):
    """Explicit argument sizes of every kernel, from the AMDGPU metadata note of the code object's ELF image."""
    data = open(path, "rb").read()
    elf = data[data.index(b"\x7fELF"):] if b"\x7fELF" in data else b""
    assert elf, f"{path} holds no ELF image"
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(shnum):
        sh = shoff + k * shentsize
        kind, = struct.unpack_from("<I", elf, sh + 4)
        if kind != 7:  # SHT_NOTE
            continue
        off, size = struct.unpack_from("<QQ", elf, sh + 24)
        end = off + size
        while off + 12 <= end:
            nsz, dsz, ntype = struct.unpack_from("<III", elf, off)
            name = elf[off + 12:off + 12 + nsz].rstrip(b"\0")
            desc = off + 12 + (nsz + 3) // 4 * 4
            if name == b"AMDGPU" and ntype == 32:
                meta = msgpack.unpackb(elf[desc:desc + dsz])
                return {f[".name"]: [a[".size"] for a in f.get(".args", []) if not a[".value_kind"].startswith("hidden")]
                        for f in meta["amdhsa.kernels"]}
            off = desc + (dsz + 3) // 4 * 4
    raise AssertionError(f"{path}: no AMDGPU metadata")


@pytest.mark.parametrize("name", sorted(PUBLISHED))
def test_published_kernels_keep_their_arguments(name):
    assert os.path.exists(CODE_OBJECT), "run __graft_entry__.build()"
    assert kernel_arguments(CODE_OBJECT)[name] == PUBLISHED[name]
