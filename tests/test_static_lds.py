"""LDS that the compiled kernels reserve themselves, from the code objects in the built library (host only)."""
import os
import struct

import msgpack
import moe_gfx950 as mg

NOTE = struct.pack("<I", 32) + b"AMDGPU\0\0"   # type NT_AMDGPU_METADATA, name


def kernels():
    blob, out, at = open(mg.LIB_PATH, "rb").read(), {}, 0
    while (at := blob.find(NOTE, at)) >= 0:
        size, = struct.unpack_from("<I", blob, at - 4)
        begin = at + len(NOTE)
        for k in msgpack.unpackb(blob[begin:begin + size])["amdhsa.kernels"]:
            out[k[".name"]] = k[".group_segment_fixed_size"]
        at = begin
    return out


def test_vector_kernels_leave_their_64_kb_to_the_launch():
    """They are launched with 64 KB of dynamic LDS, all that a kernel may have unless its limit has been raised."""
    assert os.path.exists(mg.LIB_PATH)
    vector = {n: s for n, s in kernels().items() if "gemv_kmajor_kernel" in n}
    assert len(vector) == 3 and set(vector.values()) == {0}, vector
