"""Registers of kernels whose launch shapes count on them, from the metadata of the built library's gfx950 code objects (no GPU)."""
from __future__ import annotations

import os
import re
import struct

import msgpack
import pytest

import turboinfer_amd as T


def kernels(path):
    """{mangled name: metadata} of every kernel in the library's offload bundles."""
    data, out = open(path, "rb").read(), {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        n, at = struct.unpack_from("<Q", data, m.end())[0], m.end() + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, at)
            name, at = data[at + 24 : at + 24 + idlen], at + 24 + idlen
            if b"gfx950" in name and size:
                out.update(code_object(data[m.start() + off : m.start() + off + size]))
    return out


def code_object(elf):
    shoff, shentsize, shnum = struct.unpack_from("<Q", elf, 40)[0], *struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        kind, _, _, off, size = struct.unpack_from("<IQQQQ", elf, shoff + i * shentsize + 4)
        end = off + size if kind == 7 else off   # SHT_NOTE
        while off < end:
            namesz, descsz, typ = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3 & ~3)
            if typ == 32 and elf[off + 12 : off + 18] == b"AMDGPU":   # NT_AMDGPU_METADATA
                return {k[".name"]: k for k in msgpack.unpackb(elf[desc : desc + descsz])["amdhsa.kernels"]}
            off = desc + (descsz + 3 & ~3)
    return {}


@pytest.fixture(scope="module")
def built():
    T.lib()
    return kernels(os.path.join(os.path.dirname(T.__file__), "lib", "libturboinfer_amd.so"))


# (formats of int4, int8, fp16 and blocks of 32; a SIMD's 512 registers go to its waves in steps of 8)
@pytest.mark.parametrize("shape,fmts,waves", [((1, 4, 1, 1, 3), (4, 8, 16, 36, 40), 6), ((1, 4, 2, 1, 3), (4, 8, 16, 36, 40), 5), ((1, 4, 4, 2, 2), (4,), 3)])
def test_many_rows_blocks_keep_their_waves(built, shape, fmts, waves):
    """What the epilogue asks for ahead does not cost the blocks of 16 and 32 rows, and int4's 64 x 128, a wave a SIMD or scratch."""
    for f in fmts:
        name = "_ZN2ti16gemm_wide_kernelI" + "".join("Li%dE" % v for v in (f, *shape)) + "EEvNS_8GemvArgsEiii"
        k = built[name]
        assert k[".vgpr_count"] <= 512 // waves // 8 * 8, (f, k[".vgpr_count"])
        assert k[".private_segment_fixed_size"] == 0, f
