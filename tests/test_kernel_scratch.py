"""No kernel of the built library keeps registers in scratch.  For the grouped GEMMs this matters beyond the reloads: their
stream counts the vector memory operations in flight by hand, and a scratch reload is one more, which the compiler waits
for by draining the stream.  Read from the AMDGPU metadata notes of the code objects in libhymoe.so."""
import struct

import pytest

import hyper_amd.build

msgpack = pytest.importorskip("msgpack")


def kernels(lib: bytes):
    """the kernel records of every amdgcn code object bundled in the library"""
    at, out = 0, []
    while (at := lib.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        n, = struct.unpack_from("<Q", lib, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", lib, p)
            triple = lib[p + 24:p + 24 + tl]
            p += 24 + tl
            if b"amdgcn" in triple:
                out += notes(lib[at + off:at + off + size])
        at += 24
    return out


def notes(elf: bytes):
    phoff, = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    for i in range(count):
        kind, _, off, _, _, length = struct.unpack_from("<IIQQQQ", elf, phoff + i * size)
        q = off
        while kind == 4 and q < off + length:   # PT_NOTE
            ns, ds, nt = struct.unpack_from("<III", elf, q)
            name, d = elf[q + 12:q + 12 + ns], q + 12 + (ns + 3) // 4 * 4
            if nt == 32 and name.startswith(b"AMDGPU"):
                return msgpack.unpackb(elf[d:d + ds], strict_map_key=False)["amdhsa.kernels"]
            q = d + (ds + 3) // 4 * 4
    return []


def test_no_kernel_uses_scratch():
    ks = kernels(hyper_amd.build.OUT.read_bytes())
    assert sum("k_gemm" in k[".name"] for k in ks) >= 30
    bad = {k[".name"]: k[".private_segment_fixed_size"] for k in ks if k[".private_segment_fixed_size"] or k[".uses_dynamic_stack"]}
    assert not bad, bad
