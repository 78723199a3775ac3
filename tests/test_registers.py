"""Registers that the compiler gives the attention kernels of the built library, from the metadata of its code objects: an instance
that begins to spill in its key loop gets slower (by up to a third) with every result unchanged, so no other test would notice."""
import os
import re
import struct

import msgpack
import pytest

import lvar_amd.build as build

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    at = blob.find(BUNDLE)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + len(BUNDLE))
        pos = at + len(BUNDLE) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            if build.ARCH.encode() in blob[pos + 24:pos + 24 + idlen]:
                yield blob[at + off:at + off + size]
            pos += 24 + idlen
        at = blob.find(BUNDLE, at + 1)


def _kernels(elf):
    """The kernel records of the AMDGPU metadata note (type 32, msgpack) of a 64-bit ELF."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    entsize, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 24)
        if kind != 7:      # SHT_NOTE
            continue
        pos = off
        while pos + 12 <= off + size:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (namesz + 3) // 4 * 4
            if ntype == 32 and elf[pos + 12:pos + 18] == b"AMDGPU":
                yield from msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]
            pos = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def attn_kernels():
    """{(kernel, template arguments): metadata} of the attention kernels"""
    if not os.path.exists(build.LIB_PATH):
        build.build_library()
    blob = open(build.LIB_PATH, "rb").read()
    found = {}
    for elf in _code_objects(blob):
        for k in _kernels(elf):
            m = re.match(r"_ZN4lvar\d+(attn_fwd_kernel|attn_fwd_balanced_kernel)I((?:L[ib]\d+E)+)E", k[".name"])
            if m:
                found[(m[1],) + tuple(int(x) for x in re.findall(r"L[ib](\d+)E", m[2]))] = k
    assert len(found) >= 30
    return found


# attn_fwd_kernel<D, NWAVES, MODE, ACCUM, LSE_ONLY, NPROD, IDLE, THIRD, PAIR>, attn_fwd_balanced_kernel<D, NWAVES, MODE, ACCUM>:
# what spills, and how much at most; nothing else may
MAY_SPILL = {
    ("attn_fwd_kernel", 64, 4, 1, 0, 0, 0, 0, 1, 0): 2,      # limited to 168 registers: three workgroups per compute unit
    ("attn_fwd_kernel", 128, 2, 2, 1, 0, 0, 0, 0, 0): 14,    # token lists of 64-row groups
    ("attn_fwd_balanced_kernel", 128, 3, 2, 1): 6,
    ("attn_fwd_kernel", 256, 2, 2, 1, 0, 0, 0, 0, 0): 4,
}


def test_spilled_registers(attn_kernels):
    spilled = {name: k[".vgpr_spill_count"] for name, k in attn_kernels.items() if k.get(".vgpr_spill_count", 0) > MAY_SPILL.get(name, 0)}
    assert not spilled, spilled


def test_statistics_at_head_dim_64_run_four_waves_per_simd(attn_kernels):
    assert attn_kernels[("attn_fwd_kernel", 64, 4, 1, 0, 1, 0, 0, 0, 0)][".vgpr_count"] <= 512 // 4
