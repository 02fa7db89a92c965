"""What the built kernels take, from the library's own code object: the
per-program resolves keep their values in registers.  Held to eight waves
per SIMD, a program that needs more than their 64 registers spills to memory
in every pixel."""
import os
import struct

import msgpack
import pytest

from rsr_amd import rgl

NT_AMDGPU_METADATA = 32
ET_NOTE = 7


def _code_object(path):
    """The gfx950 ELF of a library built by hipcc (an uncompressed bundle)."""
    d = open(path, "rb").read()
    i = d.index(b"__CLANG_OFFLOAD_BUNDLE__")
    at = i + 24 + 8
    for _ in range(struct.unpack_from("<Q", d, i + 24)[0]):
        off, size, n = struct.unpack_from("<QQQ", d, at)
        name = d[at + 24:at + 24 + n]
        at += 24 + n
        if name.startswith(b"hip") and b"gfx950" in name:
            return d[i + off:i + off + size]
    raise AssertionError("no gfx950 code object")


def _kernels(elf):
    """The kernels' metadata (a msgpack note) by mangled name."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for k in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + k * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + k * shentsize + 24)
        end = off + size
        while kind == ET_NOTE and off < end:
            nsz, dsz, typ = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (nsz + 3) // 4 * 4
            if typ == NT_AMDGPU_METADATA:
                m = msgpack.unpackb(elf[desc:desc + dsz], strict_map_key=False)
                return {x[".name"]: x for x in m["amdhsa.kernels"]}
            off = desc + (dsz + 3) // 4 * 4
    raise AssertionError("no kernel metadata")


def test_resolves_keep_out_of_scratch():
    if not os.path.exists(rgl.LIB_PATH):
        pytest.skip("library not built")
    resolves = {n: k for n, k in _kernels(_code_object(rgl.LIB_PATH)).items() if "k_resolve" in n}
    assert len(resolves) >= 15
    for n, k in resolves.items():
        # Blinn-Phong needs one register more than eight waves leave, and
        # gains by them in spite of its few spills
        most = 20 if "ProgManyBlinnPhong" in n and "ShadeOne" in n else 0
        assert k[".private_segment_fixed_size"] <= most, n
