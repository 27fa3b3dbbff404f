"""The host planner of FLASH_ATTN_EXT (csrc/fa_plan.hpp) on the CPU: the work lists and tile maps of the
matrix-core score route, for every number of KV heads. No GPU calls."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def native(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")

    def run(name: str, *flags: str) -> str:
        exe = str(tmp_path_factory.mktemp("native") / name)
        subprocess.run([cxx, "-std=c++20", "-O2", "-Wall", "-I" + os.path.join(REPO, "include"),
                        "-I" + os.path.join(REPO, "tesseract-npu_amd", "csrc"), *flags, "-o", exe,
                        os.path.join(REPO, "tests", "native", name + ".cpp")], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, f"{name}: status {r.returncode}: {r.stdout}{r.stderr}"
        return r.stdout

    return run


def test_score_route_tile_map(native):
    """1 .. 64 KV heads: the cap on the chunk length (4 floor(9344 / (16 n_head_kv)) groups) is no multiple of a
    tile for most counts from 19 on; such rows of several chunks stay on the one-row score kernel."""
    assert "on the matrix cores" in native("fa_plan_check")
