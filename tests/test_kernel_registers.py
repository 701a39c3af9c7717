"""Registers and scratch of the built kernels, from the notes of the library's own
code objects: variants that no timed workload runs must not lose a wave per SIMD
unseen. 512 registers a lane hold 3 waves of up to 168 each."""
import os
import struct
import subprocess

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pdekit_amd", "libpdekit_rd.so")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    at = data.find(BUNDLE)
    while at >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + n] and size:
                yield data[at + off:at + off + size]
            pos += 24 + n
        at = data.find(BUNDLE, at + 24)


def notes(elf):
    table, = struct.unpack_from("<Q", elf, 0x28)
    size, count = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(count):
        kind, = struct.unpack_from("<I", elf, table + k * size + 4)
        off, length = struct.unpack_from("<QQ", elf, table + k * size + 0x18)
        pos = off
        while kind == 7 and pos < off + length:
            name, desc, what = struct.unpack_from("<III", elf, pos)
            pos += 12 + (name + 3 & ~3)
            if what == 32:
                yield msgpack.unpackb(elf[pos:pos + desc])
            pos += desc + 3 & ~3


@pytest.fixture(scope="module")
def kernels():
    """{"rd_patch_kernel<2, 3, ...>": (registers, bytes of scratch)}"""
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    found = {}
    with open(LIB, "rb") as f:
        for elf in code_objects(f.read()):
            for n in notes(elf):
                for k in n["amdhsa.kernels"]:
                    found[k[".name"]] = (k[".vgpr_count"], k[".private_segment_fixed_size"])
    plain = subprocess.run(["c++filt"], input="\n".join(found), text=True, check=True, capture_output=True).stdout
    return {p.split("(")[0].replace("void pdrd::", ""): found[m] for m, p in zip(found, plain.splitlines())}


# physics Burgers; schemes LDA, N, B, PSI and the PSI / LDA blend; plain, nodal
# inputs (LDA and B) and source fields
@pytest.mark.parametrize("scheme,form", [(s, f) for s in range(5) for f in (0, 2, 3) if f != 2 or s in (0, 2)])
def test_q2_burgers_runs_three_waves(kernels, scheme, form):
    regs, scratch = kernels[f"rd_patch_kernel<2, 4, 9, 16, 8, false, 1, {scheme}, {form}>"]
    assert regs <= 168 and scratch == 0


def test_p2_lda_cells_run_two_waves(kernels):
    regs, scratch = kernels["rd_cell_kernel<2, 3, 6, 10, 6, true, 2, 0, 0>"]
    assert regs <= 256 and scratch <= 32
