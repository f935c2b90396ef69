"""Registers of the built kernels (code object metadata of the library): the counts on which the number of resident workgroups
depends, and spills."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "indexsdk_amd", "libindexsdk_amd.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
SCAN = re.compile(r"ivfpq_scan_kernelILi(\d+)E(f|6__half)Li(\d)ELi(\d+)ELb([01])EE")
GROUPS = re.compile(r"ivfpq_scan_groups_kernelILi(n?\d+)E(f|6__half)Li(\d)ELb([01])EE")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: (registers per lane, spilled registers)} of every gfx950 kernel in the library"""
    if not (os.path.exists(LIB) and os.path.exists(READELF)):
        pytest.skip("needs the built library and the ROCm toolchain")
    data, found, at = open(LIB, "rb").read(), {}, 0
    path = str(tmp_path_factory.mktemp("co") / "kernels.co")
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length].decode()
            entry += 24 + length
            if "gfx950" in target and size:
                with open(path, "wb") as f:
                    f.write(data[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", path], capture_output=True, text=True, check=True).stdout
                for block in notes.split("- .agpr_count")[1:]:
                    def field(key):
                        return re.search(rf"\.{key}:\s+(\S+)", block).group(1)
                    found[field("name")] = int(field("vgpr_count")), int(field("vgpr_spill_count"))
        at = entry
    assert len(found) > 100
    return found


def test_register_selection(kernels):
    select = [v for n, v in kernels.items() if re.search("select_rows_reg_kernelI[fi]Li[124]ELb0EE", n)]
    assert len(select) == 6 and all(spilled <= 8 for _, spilled in select)


def test_scan_kernels_of_short_codes_leave_room_for_four_workgroups(kernels):
    """Row layout, eight wavefronts: 64 registers let four workgroups share a CU (private pools up to M 32, the shared pool up
    to M 8)."""
    seen = 0
    for name, (registers, spilled) in kernels.items():
        m = SCAN.search(name)
        if m and m.group(3) == "0" and m.group(4) == "8" and 0 < int(m.group(1)) <= (8 if m.group(5) == "1" else 32):
            assert registers <= 64 and spilled == 0, (name, registers, spilled)
            seen += 1
    assert seen >= 16


def test_scan_kernels_by_groups_have_the_registers_of_those_by_lists(kernels):
    """Eight wavefronts; row layout: 64 registers for private pools up to M 32 and the shared pool up to M 8, as above."""
    seen = 0
    for name, (registers, spilled) in kernels.items():
        m = GROUPS.search(name)
        if m:
            assert spilled == 0 and registers <= 256, (name, registers, spilled)
            if m.group(3) == "0" and not m.group(1).startswith("n") and 0 < int(m.group(1)) <= (8 if m.group(4) == "1" else 32):
                assert registers <= 64, (name, registers)
                seen += 1
    assert seen >= 16


def test_encoders_do_not_spill(kernels):
    """32 vectors and the fragments of 256 codewords per wavefront: two wavefronts per SIMD up to 24 dimensions, one at 32."""
    encoders = {n: v for n, v in kernels.items() if "pq_encode_kernelILi" in n}
    assert len(encoders) == 11
    for name, (registers, spilled) in encoders.items():
        dsub = int(re.search(r"pq_encode_kernelILi(\d+)E", name).group(1))
        assert spilled == 0 and registers <= (256 if dsub <= 24 else 512), (name, registers, spilled)


def test_merge_of_slices(kernels):
    merge = [v for n, v in kernels.items() if "ivfpq_merge_kernel" in n]
    assert merge and all(registers <= 64 and spilled == 0 for registers, spilled in merge)      # two workgroups per CU


def test_scan_kernels_of_sixteen_wavefronts_spill_only_at_96_bytes(kernels):
    limit = {("f", "0"): 194, ("6__half", "0"): 194, ("f", "1"): 66, ("6__half", "1"): 17}
    for name, (registers, spilled) in kernels.items():
        m = SCAN.search(name)
        if m and m.group(4) == "16":
            allowed = limit[m.group(2), m.group(3)] if m.group(1) == "96" else 0
            assert registers <= 128 and spilled <= allowed, (name, registers, spilled)


def test_kernels_that_split_in_registers_do_not_spill(kernels):
    """Their fragments are read by instructions whose arrival the compiler does not track: a spill would store them too early."""
    resident = [v for n, v in kernels.items() if "resident_f32_kernel" in n]
    assert len(resident) == 21 and all(registers <= 256 and spilled == 0 for registers, spilled in resident)
