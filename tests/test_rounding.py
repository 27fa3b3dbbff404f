"""The device's forms of EXPK, of the A32 quantizer's rounding and of the P.V digit sums' rounding on the CPU, against
the oracle and exact integers. TSR_FULL_SWEEP=1: every f32 bit pattern (17 CPU minutes), else a sample of each
exponent. No GPU calls."""
import os
import shutil

import pytest

from conftest import REPO

CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")   # vector types as hipcc has them


def test_device_rounding(native):
    if shutil.which(CLANG) is None:
        pytest.skip("no clang++")
    full = os.environ.get("TSR_FULL_SWEEP") == "1"
    oracle = os.path.join(REPO, "oracle")
    out = native("rounding_check", os.path.join(oracle, "liboracle.so"), "-Wl,-rpath," + oracle, "-lpthread", cxx=CLANG,
                 args=("1", str(os.cpu_count())) if full else ("257", "4"))
    assert "every value" in out
