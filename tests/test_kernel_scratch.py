"""Properties of the pipelined kernels' code that no result shows.

Scratch: the pipelined kernels order their direct loads by counting outstanding memory
operations; the compiler does not know of those loads, so a scratch access
inside such a loop also waits for all of them (measured: the pair layout's
long GEMM ran 3 to 5 times as slow). The code objects' own metadata says what
each kernel uses.

m0: an asm block that writes it names it as clobbered, or the compiler may keep
a value of its own there across the block."""
import re
import struct

import msgpack
import pytest

from dtree_hip import _native as N

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    at = blob.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 1)


def _kernels(elf):
    """Kernel records of an amdgcn ELF's metadata note (type 32)."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        p = off
        while p < off + size:
            nlen, dlen, ntype = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3) // 4 * 4
            if ntype == 32:
                yield from msgpack.unpackb(elf[d:d + dlen], strict_map_key=False)["amdhsa.kernels"]
            p = d + (dlen + 3) // 4 * 4


def test_pipelined_kernels_use_no_scratch():
    if not N.LIB_PATH.exists():
        pytest.skip("library not built")
    kernels = [k for o in _code_objects(N.LIB_PATH.read_bytes()) for k in _kernels(o)]
    pipelined = [k for k in kernels if any(n in k[".name"] for n in ("long_kernel", "longq_kernel", "causal_attn"))]
    assert len(pipelined) >= 50, [k[".name"] for k in kernels]
    assert [k[".name"] for k in pipelined if k[".private_segment_fixed_size"]] == []


def test_asm_that_writes_m0_names_it():
    blocks = []
    for f in sorted((N.LIB_PATH.parent.parent / "csrc").glob("*.h*")):
        blocks += [(f.name, b) for b in re.findall(r"\basm\b[^;]*?\(.*?\);", f.read_text(), re.S)
                   if re.search(r"\b(s_mov_b32|v_readfirstlane_b32|s_add_u32)\s+m0\b", b)]
    assert len(blocks) >= 2
    assert [f for f, b in blocks if '"m0"' not in b.rsplit(":", 1)[1]] == []
