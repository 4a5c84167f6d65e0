"""Registers and scratch memory of the built kernels, from the metadata of the
library's own code objects (no GPU)."""
import re
import struct

import msgpack

from fd23_amd import _lib


def kernels():
    data = open(_lib.LIB_PATH, "rb").read()
    found, magic = {}, b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in target:
                found.update(notes(data[at + off:at + off + size]))
        at = data.find(magic, p)
    return found


def notes(elf):
    """Kernel name -> metadata of one AMDGPU ELF (its NT_AMDGPU_METADATA note)."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phsize)
        p = off
        while kind == 4 and p < off + size:
            namelen, desclen, note = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namelen + 3) // 4 * 4
            if note == 32:
                meta = msgpack.unpackb(elf[desc:desc + desclen], strict_map_key=False)
                return {k[".name"]: k for k in meta["amdhsa.kernels"]}
            p = desc + (desclen + 3) // 4 * 4
    return {}


def instances(pattern):
    got = {n: k for n, k in kernels().items() if re.search(pattern, n)}
    assert got, pattern
    return got


def test_fp32_march_keeps_its_rows_in_registers():
    """No instance of the FP32 marching steps spills a vector register or has
    arrays in scratch memory."""
    for n, k in instances(r"k_psv_marchIf|k_sh_march").items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, (n, k)


def test_whole_grid_passes_do_not_spill():
    for n, k in instances(r"k_(psv|sh)_(stress|velocity)I").items():
        assert k[".vgpr_spill_count"] == 0, (n, k[".vgpr_spill_count"])


def test_passes_of_several_shots_keep_three_wavefronts():
    """Four rows and several shots per workgroup: at most 168 registers, three
    wavefronts per SIMD, with 16-bit P-SV and FP64 SH storage."""
    got = instances(r"k_psv_(stress|velocity)I(6__half|14__hip_bfloat16)Li4ELi[248]ELi0E")
    got.update(instances(r"k_sh_(stress|velocity)IdLi4ELi[48]E"))
    for n, k in got.items():
        assert k[".vgpr_count"] <= 168, (n, k[".vgpr_count"])


def test_one_row_sh_passes_stay_small():
    """One row per thread in FP32, bound by memory on large grids: no registers
    for values loaded ahead (33 without, 38 with them)."""
    for n, k in instances(r"k_sh_(stress|velocity)IfLi1ELi1E").items():
        assert k[".vgpr_count"] <= 33, (n, k[".vgpr_count"])
