"""No kernel of the built library keeps an array in scratch memory.

A loop that the compiler declines to unroll indexes the accumulators by a
running number, and they move to scratch memory for the whole of the K loop
without an error anywhere (half a kilobyte a lane for the 32 blocks of a wave).
The code objects say how much scratch memory each kernel has. (CPU test: reads
the library's own metadata.)
"""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

from iree_amd import ukernel as uk


def _kernels(path):
    """Name and scratch bytes of each kernel, from the AMDGPU notes of the ELF
    images inside the library."""
    data = open(path, "rb").read()
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:  # EM_AMDGPU
            phoff, = struct.unpack_from("<Q", data, at + 32)
            phentsize, phnum = struct.unpack_from("<HH", data, at + 54)
            for i in range(phnum):
                kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", data, at + phoff + i * phentsize)
                if kind != 4:  # PT_NOTE
                    continue
                note = data[at + offset:at + offset + size]
                name_size, desc_size, note_type = struct.unpack_from("<III", note)
                start = 12 + (name_size + 3) // 4 * 4
                if note_type == 32 and note[12:18] == b"AMDGPU":
                    meta = msgpack.unpackb(note[start:start + desc_size], strict_map_key=False)
                    for k in meta.get("amdhsa.kernels", []):
                        yield k[".name"], k[".private_segment_fixed_size"]
        at = data.find(b"\x7fELF", at + 1)


def test_no_kernel_keeps_an_array_in_scratch_memory():
    assert os.path.exists(uk.LIB_PATH), "built by __graft_entry__.build()"
    kernels = list(_kernels(uk.LIB_PATH))
    assert sum("mmt4d_mfma_kernel" in name for name, _ in kernels) > 100
    # Spilled registers of the longest shapes are a few dozen bytes.
    assert not [(name, b) for name, b in kernels if b > 128]
