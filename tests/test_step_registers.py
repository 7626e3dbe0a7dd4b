"""Registers of the forest step's instances, from the metadata of the built
code objects: what the occupancy that each was written for leaves."""
import re
import struct

import msgpack
import pytest

from saclaymocks_amd import _lib


def _kernels():
    """{kernel name: metadata} of every code object in the library."""
    with open(_lib.LIB_PATH, "rb") as f:
        b = f.read()
    out = {}
    for m in re.finditer(rb"AMDGPU\0\0", b):   # ELF notes: sizes and type, the name, the metadata
        name_size, size, kind = struct.unpack("<III", b[m.start() - 12:m.start()])
        if (name_size, kind) == (7, 32):
            note = msgpack.unpackb(b[m.end():m.end() + size])
            out.update((k[".name"], k) for k in note["amdhsa.kernels"])
    return out


# (classes, threads per block, waves per SIMD); 512 registers per SIMD lane
@pytest.mark.parametrize("classes,threads,waves", [(5, 256, 2), (3, 64, 3), (2, 64, 4), (1, 64, 5)])
def test_step_fits_its_occupancy(classes, threads, waves):
    names = [n for n in _kernels() if f"k_forest_stepILi{classes}ELi{threads}E" in n]
    fits = [n for n in names if _kernels()[n][".vgpr_count"] <= 512 // waves // 8 * 8
            and _kernels()[n][".private_segment_fixed_size"] == 0]
    assert names and fits, {n: (_kernels()[n][".vgpr_count"], _kernels()[n][".private_segment_fixed_size"])
                            for n in names}
