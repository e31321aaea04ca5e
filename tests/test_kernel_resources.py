"""
What the built kernels take of a compute unit, read from the metadata of libnsmoe.so's own
code objects (the LDS and register figures that the compiler writes beside each kernel).
The launch rules count on these workgroups per CU; a larger table or tile lowers them
without a word.
"""

import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

from nanospeaker_amd import _native as nat

LDS_PER_CU = 160 * 1024
READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
OBJCOPY = shutil.which("llvm-objcopy") or "/opt/rocm/llvm/bin/llvm-objcopy"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: {"lds": bytes, "vgprs": n, "spills": n}} of every kernel."""
    if not (Path(READELF).exists() and Path(OBJCOPY).exists() and nat.LIB_PATH.exists()):
        pytest.skip("needs the LLVM binutils and the built library")
    tmp = tmp_path_factory.mktemp("code_objects")
    fat = tmp / "fatbin"
    subprocess.run([OBJCOPY, f"--dump-section=.hip_fatbin={fat}", str(nat.LIB_PATH), "/dev/null"],
                   check=True)
    blob, out = fat.read_bytes(), {}
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for at in (m.start() for m in re.finditer(magic, blob)):
        n, pos = struct.unpack_from("<Q", blob, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if "gfx950" not in triple or not size:
                continue
            obj = tmp / "object.elf"
            obj.write_bytes(blob[at + off:at + off + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], check=True,
                                   capture_output=True, text=True).stdout
            for part in notes.split("- .agpr_count:")[1:]:
                field = lambda key: re.search(rf"\.{key}:\s+(\S+)", part).group(1)
                name = re.search(r"^    \.name:\s+(\S+)", part, re.M).group(1)
                out[name] = {"lds": int(field("group_segment_fixed_size")),
                             "vgprs": int(field("vgpr_count")),
                             "spills": int(field("vgpr_spill_count"))}
    assert len(out) > 100
    return out


def _of(kernels, pattern):
    found = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert found, pattern
    return found


def test_general_dw_kernel_fits_three_times_in_a_cu(kernels):
    """dw_kernel in 16-bit types (DT 0 and 1, both modes)."""
    for name, k in _of(kernels, r"dw_kernelILi[01]ELi[01]E").items():
        assert 3 * k["lds"] <= LDS_PER_CU, (name, k)


def test_dw_pair_kernel_fits_twice_in_a_cu(kernels):
    """dw_pair_kernel at two stages in every type, and at three in 16-bit types: two
    workgroups beside their token tables of 4 bytes a row, for the longest chunks (8192 rows)
    at two stages and chunks of 5000 rows (184 k rows of work) at three."""
    for pattern, rows in ((r"dw_pair_kernelILi[012]ELi2E", 8192), (r"dw_pair_kernelILi[01]ELi3E", 5000)):
        for name, k in _of(kernels, pattern).items():
            assert 2 * (k["lds"] + 4 * rows) <= LDS_PER_CU, (name, k)


@pytest.mark.parametrize("pattern,spills", [
    (r"expert_fwd_reg_kernelILi0ELi2ELi6ELi2ELb0E", 3),      # 96-row tiles
    (r"expert_fwd_reg_kernelILi0ELi2ELi[24]ELi[26]ELb[01]E", 0),
    (r"expert_bwd_reg_kernelILi0ELi2ELi2ELi[36]ELb[01]E", 0),
    (r"expert_bwd_reg_kernelILi0ELi2ELi3ELi4ELb1E", 0),
    (r"expert_dx_reg_kernelILi0ELi2ELi4E", 0),
    (r"expert_dx_res_kernelILi0ELi2E", 0),
    (r"dw_pair_kernelILi[012]ELi2E", 0),
    (r"dw_kernelILi[012]E", 0),
    (r"expert_fwd_kernelILi[012]E", 0),
    (r"expert_bwd_kernelILi[01]E", 0),
    (r"expert_bwd_kernelILi2E", 6),                          # fp32
    (r"linear_kernelILi[01]ELi[24567]E", 0),
    (r"linear_kernelILi[01]ELi8E", 8),                       # 128 rows
    (r"attn_fwd_kernel", 0), (r"router_fwd_kernel", 0), (r"combine_dx_kernel", 0)])
def test_registers_spilled_by_the_kernels_taken_by_default(kernels, pattern, spills):
    """The forms that the launch rules take without an option: what each keeps in scratch."""
    for name, k in _of(kernels, pattern).items():
        assert k["spills"] <= spills, (name, k)
