"""Register counts that a kernel's occupancy rests on, from the metadata of the built libtsr_hip.so. No GPU calls."""
import glob
import os
import re
import shutil
import subprocess

import pytest

import tsr_hip

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """kernel symbol -> (scalar, vector) registers."""
    objdump, readelf = os.path.join(LLVM, "llvm-objdump"), os.path.join(LLVM, "llvm-readelf")
    if not (os.path.exists(objdump) and os.path.exists(readelf)):
        pytest.skip("no llvm-objdump / llvm-readelf")
    tmp = tmp_path_factory.mktemp("co")
    shutil.copy(tsr_hip.LIB_PATH, tmp / "lib.so")
    subprocess.run([objdump, "--offloading", "lib.so"], cwd=tmp, check=True, capture_output=True)
    regs = {}
    for co in glob.glob(str(tmp / "*gfx950*")):
        notes = subprocess.run([readelf, "--notes", co], check=True, capture_output=True, text=True).stdout
        for name, sgpr, vgpr in re.findall(r"\.name: +(_Z\w+).*?\.sgpr_count: +(\d+).*?\.vgpr_count: +(\d+)", notes, re.S):
            regs[name] = (int(sgpr), int(vgpr))
    assert regs
    return regs


def test_q80_matvec_two_workgroups_a_cu(registers):
    """The Q8_0 matvec of up to two passes without the norm: eight waves a SIMD (64 vector, 80 scalar registers)."""
    k = {n: r for n, r in registers.items() if re.search(r"k_mv_q80ILi[12]E", n)}
    assert len(k) == 6
    assert all(s <= 80 and v <= 64 for s, v in k.values()), k


def test_rope_kv_four_workgroups_a_cu(registers):
    """ROPE + SET_ROWS_KV: four workgroups of eight waves on a CU (64 vector, 80 scalar registers)."""
    k = {n: r for n, r in registers.items() if "k_rope_kv" in n}
    assert len(k) == 1
    assert all(s <= 80 and v <= 64 for s, v in k.values()), k


def test_attention_pv_eight_waves_a_simd(registers):
    """The P.V kernel of FLASH_ATTN_EXT: at most 64 vector registers, so that its workgroups of up to eight waves fill
    the SIMDs."""
    k = {n: r for n, r in registers.items() if re.search(r"k_fa_pvILi\d+E", n)}
    assert len(k) == 18
    assert all(v <= 64 for _, v in k.values()), k
