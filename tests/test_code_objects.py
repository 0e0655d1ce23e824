"""Launch bounds of the built-in kernels, read from the embedded code object's
own metadata (no GPU needed)."""
from __future__ import annotations

import ctypes
import re
import struct

import msgpack


def _kernels(elf: bytes) -> dict:
    """name -> metadata of every kernel in an AMDGPU code object (the msgpack
    document of its NT_AMDGPU_METADATA note)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        if kind != 7:  # SHT_NOTE
            continue
        namesz, descsz, note = struct.unpack_from("<III", elf, off)
        if note == 32 and elf[off + 12:off + 12 + namesz] == b"AMDGPU\0":
            at = off + 12 + (namesz + 3) // 4 * 4
            doc = msgpack.unpackb(elf[at:at + descsz], strict_map_key=False)
            return {k[".name"]: k for k in doc["amdhsa.kernels"]}
    raise AssertionError("no AMDGPU metadata note")


def test_one_pass_matvecs_are_compiled_for_eight_waves(axc):
    """The one-pass kernels that 8-wave workgroups run have the launch bound of
    8 waves: the forms for 9 to 12 waves are other kernels, whose run-time wave
    count these do not pay for."""
    kernels = _kernels(axc.builtin_code_object())
    one = {n: k for n, k in kernels.items() if re.search(r"_matvec_one[px]?_i\d+$", n)}
    assert len(one) > 100
    assert {k[".max_flat_workgroup_size"] for k in one.values()} == {512}
    assert not any(k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]
                   for k in one.values())


def test_matmul_kernels_hold_one_body(axc):
    """The 32 x 32 tiles that take the place of other variants' kernels are a kernel
    of their own: as a second body they cost the first ones their launch size of
    four waves and a third more registers."""
    lib = axc.load_library()
    begin, end = (ctypes.addressof(ctypes.c_char.in_dll(lib, f"axh_q4_matmul_co_{n}"))
                  for n in ("begin", "end"))
    kernels = _kernels(ctypes.string_at(begin, end - begin))
    assert kernels["axh_q4k_matmul_t32"][".max_flat_workgroup_size"] == 512
    assert kernels["axh_q4k_matmul_kx_r4_n1_k4_p3"][".max_flat_workgroup_size"] == 256
    # 6 waves per SIMD (512 VGPRs), against 4 with both bodies
    assert kernels["axh_q4k_matmul_kx_r4_n1_k4_p3"][".vgpr_count"] <= 80
