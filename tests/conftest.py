"""Shared fixtures. GPU tests carry @pytest.mark.gpu and call libtsr_hip through its C ABI; the CPU
checkers (oracle/) are used only as checkers."""
import os
import shutil
import subprocess
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(REPO, "oracle"))
sys.path.insert(0, os.path.join(REPO, "tesseract-npu_amd"))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs libtsr_hip kernels)")


@pytest.fixture(scope="session")
def oc():
    import oracle
    return oracle.Oracle()


@pytest.fixture(scope="session")
def ref():
    import oracle
    if not oracle.ref_available():
        pytest.skip("oracle/_ref/libtsr_ref.so not built (needs /root/reference)")
    return oracle.Ref()


@pytest.fixture(scope="session")
def dev():
    import tsr_hip
    d = tsr_hip.Device(0)
    yield d
    d.close()


@pytest.fixture(scope="session")
def native(tmp_path_factory):
    """run(name, *compiler arguments, cxx=..., args=()): builds tests/native/<name>.cpp for the CPU against the
    library's own headers, runs it and returns what it printed; its exit status has to be 0."""
    def run(name: str, *flags: str, cxx: str = "g++", args: tuple = ()) -> str:
        if shutil.which(cxx) is None:
            pytest.skip(f"no {cxx}")
        here = os.path.join(REPO, "tests", "native")
        exe = str(tmp_path_factory.mktemp("native") / name)
        subprocess.run([cxx, "-std=c++20", "-O2", "-ffp-contract=off", "-Wall", "-I" + os.path.join(here, "host"),
                        "-I" + os.path.join(REPO, "include"), "-I" + os.path.join(REPO, "tesseract-npu_amd", "csrc"),
                        "-o", exe, os.path.join(here, name + ".cpp"), *flags], check=True)
        r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, f"{name}: status {r.returncode}: {r.stdout}{r.stderr}"
        return r.stdout

    return run
