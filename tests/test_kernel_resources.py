"""Registers and LDS of the built gfx950 kernels, read from the code object
metadata of lib/libpfh.so: what decides how many workgroups share a compute
unit (160 KiB of LDS, 512 vector registers for each SIMD lane)."""
import struct

import pytest

from pfh import abi

msgpack = pytest.importorskip("msgpack")

LDS_BYTES = 160 * 1024
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
NOTE = 7                                    # SHT_NOTE


def _code_objects(blob: bytes):
    at = blob.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(BUNDLE))
        o = at + len(BUNDLE) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", blob, o)
            triple = blob[o + 24:o + 24 + n]
            o += 24 + n
            if size and triple.endswith(b"gfx950"):
                yield blob[at + off:at + off + size]
        at = blob.find(BUNDLE, at + len(BUNDLE))


def _metadata(elf: bytes):
    shoff, = struct.unpack_from("<Q", elf, 40)
    entsize, count = struct.unpack_from("<HH", elf, 58)
    for s in range(count):
        base = shoff + s * entsize
        kind, = struct.unpack_from("<I", elf, base + 4)
        if kind == NOTE:
            at, = struct.unpack_from("<Q", elf, base + 24)
            name, desc, _ = struct.unpack_from("<III", elf, at)
            start = at + 12 + (name + 3) // 4 * 4
            yield from msgpack.unpackb(elf[start:start + desc])["amdhsa.kernels"]


@pytest.fixture(scope="module")
def kernels():
    found = {k[".name"]: k for elf in _code_objects(abi.LIB_PATH.read_bytes())
             for k in _metadata(elf)}
    assert found, f"no gfx950 kernels in {abi.LIB_PATH}"
    return found


def _matching(kernels, part):
    hits = [k for n, k in kernels.items() if part in n]
    assert hits, f"no kernel named {part}"
    return hits


def test_measurement_of_small_bricks_fills_a_compute_unit(kernels):
    """A brick of edge 8 or 16 is measured by one wave with a strip of 2 KiB.
    The four SIMDs hold four waves each of the kernel's 128 registers: LDS
    must leave room for these sixteen one-wave workgroups too."""
    measure, = _matching(kernels, "k3_measure")
    assert measure[".vgpr_count"] <= 128
    assert 16 * (measure[".group_segment_fixed_size"] + 2048) <= LDS_BYTES


@pytest.mark.parametrize("kernel", ["k3_measure", "k3_update"])
def test_planes_stay_in_registers(kernels, kernel):
    """No spills: a reload waits for every plane in flight. (Scratch that is
    not a spill belongs to the out-of-line rare paths.)"""
    k, = _matching(kernels, kernel)
    assert k[".vgpr_spill_count"] == 0 and k[".sgpr_spill_count"] == 0


@pytest.mark.parametrize("kernel", ["k_sur_commitI", "k_sur_commit_cellsI"])
def test_commit_has_a_build_for_each_population(kernels, kernel):
    """Two 16-wave workgroups share a compute unit at 64 registers; the build
    for populations that leave each workgroup a unit of its own is not held to
    them. Neither spills."""
    shared, = _matching(kernels, kernel + "Lb0E")
    whole, = _matching(kernels, kernel + "Lb1E")
    assert shared[".vgpr_count"] <= 64 < whole[".vgpr_count"] <= 128
    assert shared[".vgpr_spill_count"] == whole[".vgpr_spill_count"] == 0
