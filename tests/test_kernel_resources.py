"""CPU-only: what the compiler gave the library's kernels, read from the metadata notes of the code objects in the built
library.  A kernel that keeps registers in scratch memory pays a trip to memory for every one of them, and nothing
else here would show it: results stay right."""
import os
import struct
import subprocess

import pytest

msgpack = pytest.importorskip("msgpack")


def code_objects(blob):
    """The gfx950 ELF images of a library's offload bundles."""
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + 24)
        q = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", blob, q)
            name = blob[q + 24:q + 24 + length]
            q += 24 + length
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def kernels(elf):
    """The kernel records of an image's AMDGPU metadata note (SHT_NOTE = 7, NT_AMDGPU_METADATA = 32)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3a)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 24)
        q = off
        while kind == 7 and q < off + size:
            nlen, dlen, note = struct.unpack_from("<III", elf, q)
            desc = q + 12 + (nlen + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[desc:desc + dlen])["amdhsa.kernels"]
            q = desc + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def built():
    from gfx1151_engine_amd import LIB, build
    if not os.path.exists(LIB):
        build()
    with open(LIB, "rb") as f:
        blob = f.read()
    found = [k for elf in code_objects(blob) for k in kernels(elf)]
    text = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in found), text=True, capture_output=True, check=True).stdout
    return dict(zip(text.split("\n"), found))


def test_the_few_token_router_keeps_its_registers(built):
    small = {n: k for n, k in built.items() if "k_router_small<" in n}
    assert len(small) == 8
    assert {n: (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) for n, k in small.items()} == dict.fromkeys(small, (0, 0))


def test_no_kernel_keeps_its_loops_registers_in_scratch(built):
    """None at all, but for one of the streaming GEMM that is named, with its reason, in gemm_stream.hip: the down launch of 64 pairs of
    table codebooks."""
    kept = {n.replace("(anonymous namespace)::", "").split("(")[0]: k[".vgpr_spill_count"] for n, k in built.items()
            if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert set(kept) <= {"void k_moe_stream<2, false, 4, 3, 16>"}, kept
    assert all(v <= 4 for v in kept.values()), kept
