"""Register use of the built gfx950 kernels, read from the code object notes of the library that this repository builds: a
kernel that a change pushes over a register limit still computes the same results, only slower, which no other test sees.
CDNA4 has 512 vector registers (accumulation registers included) per SIMD lane, allocated in eights: a kernel of at most
128 runs four waves per SIMD."""
import re
import struct

import msgpack
import pytest

from ijah_amd import build

NT_AMDGPU_METADATA = 32


def _notes(elf):
    """the kernels' metadata of one gfx950 code object (an ELF64 file)"""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        sh = shoff + i * shentsize
        if struct.unpack_from("<I", elf, sh + 4)[0] != 7:  # SHT_NOTE
            continue
        p, size = struct.unpack_from("<QQ", elf, sh + 24)
        end = p + size
        while p < end:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namesz + 3 & ~3)
            if ntype == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            p = desc + (descsz + 3 & ~3)


@pytest.fixture(scope="module")
def kernels():
    if not build.LIB.exists():
        build.build()
    lib, found = build.LIB.read_bytes(), {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", lib):  # one bundle per source file
        base, p = m.start(), m.start() + 32
        for _ in range(struct.unpack_from("<Q", lib, base + 24)[0]):
            off, size, idlen = struct.unpack_from("<QQQ", lib, p)
            target = lib[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in target and size:
                found.update((k[".name"], k) for k in _notes(lib[base + off:base + off + size]))
    assert found, "no gfx950 kernels in the library"
    return found


def _named(kernels, name):
    got = {n: k for n, k in kernels.items() if re.search(rf"\d{name}I", n)}  # a mangled template's name
    assert got, name
    return got


@pytest.mark.parametrize("name", ["lin_mx", "lin_mxl", "lin_mxw"])
def test_linears_keep_four_waves(kernels, name):
    """The linears' grids may be larger than what is resident at once (2560 -> 10240: 1600 workgroups of four waves): the
    finisher, which one workgroup per output block runs, must not size the registers of all of them."""
    over = {n: k[".vgpr_count"] for n, k in _named(kernels, name).items() if k[".vgpr_count"] > 128}
    assert not over, over


def test_no_kernel_spills_vector_registers(kernels):
    """No kernel keeps vector registers in scratch memory: a reload waits for every earlier request of its wave, so in a
    kernel that streams through LDS rings one spilled register drains the ring."""
    over = {n: (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) for n, k in kernels.items()
            if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not over, over
