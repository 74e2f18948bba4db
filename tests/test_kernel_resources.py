"""Register counts of the kernels as built, read from the gfx950 code object
inside libdendrite_hip.so (the kernel metadata the compiler writes into it).
CPU only: occupancy is a property of the build, and the host code's
scheduling rests on it."""
import functools
import os
import re
import struct
import subprocess

import msgpack
import pytest

from dendrite_amd import build as dbuild

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The device ELF images of every offload bundle in the library."""
    at = blob.find(BUNDLE)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + len(BUNDLE))
        o = at + len(BUNDLE) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, o)
            name = blob[o + 24:o + 24 + idlen]
            o += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(BUNDLE, at + 1)


def _metadata(elf):
    """The AMDGPU metadata note (type 32) of a device ELF image."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    size, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        _, kind, _, _, off, length = struct.unpack_from("<IIQQQQ", elf, shoff + i * size)
        if kind != 7:
            continue
        end = off + length
        while off < end:
            nlen, dlen, ntype = struct.unpack_from("<III", elf, off)
            name, off = elf[off + 12:off + 12 + nlen], off + 12 + (nlen + 3) // 4 * 4
            if name.startswith(b"AMDGPU") and ntype == 32:
                return msgpack.unpackb(elf[off:off + dlen])
            off += (dlen + 3) // 4 * 4
    return {"amdhsa.kernels": []}


@functools.lru_cache(maxsize=None)
def kernels():
    """Demangled name without its arguments -> metadata of each kernel."""
    if not os.path.exists(dbuild.LIB):
        pytest.skip("libdendrite_hip.so is not built")
    with open(dbuild.LIB, "rb") as f:
        blob = f.read()
    recs = [k for elf in _code_objects(blob) for k in _metadata(elf)["amdhsa.kernels"]]
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in recs), text=True, capture_output=True,
                           check=True).stdout.splitlines()
    short = [re.match(r"(?:void )?dh::(?:\(anonymous namespace\)::)?([^(]*)", n) for n in names]
    return {m.group(1): k for m, k in zip(short, recs) if m}


def waves_per_simd(k):
    """Waves a SIMD holds by registers: 512 of them, given out in eights."""
    return min(8, 512 // ((k[".vgpr_count"] + 7) // 8 * 8))


PLAN = [f"attend16_kernel<{d}, {fmt}>" for d in (64, 128, 256)
        for fmt in ("0u, true", "1u, false", "3u, false", "3u, true", "4u, false", "4u, true")]


@pytest.mark.parametrize("name", PLAN + [f"attend32_kernel<{d}>" for d in (64, 128, 256)])
def test_device_table_kernels_hold_as_many_waves(name):
    """The loop over units of the device-table kernels may not cost what runs
    beside it: as many waves a SIMD as the plan path's kernel of the same
    types, no scratch, and hardly a scalar register spilled (kernel arguments
    held across the loop used to spill 25-63 of them, a VGPR lane each)."""
    plan, table = kernels()[name], kernels()["csr_" + name]
    assert waves_per_simd(table) >= waves_per_simd(plan)
    assert table[".private_segment_fixed_size"] == 0
    assert table[".vgpr_spill_count"] == 0 and table[".sgpr_spill_count"] <= 8


@pytest.mark.parametrize("d", [64, 128, 256])
def test_prefill_slots_are_what_the_kernels_allow(d):
    """prefill_slots (dh_device.hpp), which the prefill planner schedules
    against, is what every prefill kernel of that head_dim allows by its
    registers and its share of a CU's 160 KiB of LDS."""
    with open(os.path.join(dbuild.CSRC, "dh_device.hpp")) as f:
        rule = re.search(r"prefill_slots\(int head_dim\) { return 256u \* \(head_dim == 256 \? (\d)u : (\d)u\); }",
                         f.read())
    per_cu = int(rule.group(1 if d == 256 else 2))
    found = [k for n, k in kernels().items() if n.startswith(f"prefill16_kernel<{d},")]
    assert len(found) == (2 if d == 64 else 6)
    for k in found:
        assert min(waves_per_simd(k), 160 * 1024 // k[".group_segment_fixed_size"]) == per_cu
