"""The host side of plain edits, compiled for the host alone over a stand-in for the HIP runtime
(cpp/edit_host_check.cpp): which passes are queued, which buffers they take, what follows one that did not hold."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")
CLANG = os.path.join(ROCM, "llvm", "bin", "clang++")
pytestmark = pytest.mark.skipif(not (os.path.exists(HIPCC) and os.path.exists(CLANG)), reason="no ROCm compiler")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = tmp_path_factory.mktemp("edit_host")
    obj, exe = str(out / "check.o"), str(out / "check")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++20", "-ffp-contract=off", "-w",
                    "-I", os.path.join(ROOT, "include"), "-c", os.path.join(ROOT, "tests", "cpp", "edit_host_check.cpp"),
                    "-o", obj], check=True)
    # (the device code's image, which the object refers to, does not exist)
    subprocess.run([CLANG, "-no-pie", "-Wl,--unresolved-symbols=ignore-all", "-o", exe, obj], check=True)
    return exe


@pytest.mark.parametrize("name", ["piece", "table", "lists", "memory", "refused", "column", "air", "ground", "cut"])
def test_edit_host(check, name):
    r = subprocess.run([check, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
