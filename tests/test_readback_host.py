"""The host side of the readback (0buf_amd/csrc/pic_readback.hip), compiled for
the CPU over a stand-in for the runtime calls it makes
(tests/cpu/readback_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which(HIPCC) is None:
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("readback")
    objs = []
    for src in (("0buf_amd", "csrc", "pic_readback.hip"), ("tests", "cpu", "readback_check.cpp")):
        objs.append(str(d / (src[-1] + ".o")))
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O2", "-fPIC", "-I",
                        os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "0buf_amd", "csrc"),
                        "-c", os.path.join(ROOT, *src), "-o", objs[-1]], check=True)
    exe = str(d / "readback_check")
    subprocess.run(["g++", *objs, "-pthread", "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("name", ["device", "failed", "waiting"])
def test_readback(check, name):
    r = subprocess.run([check, name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
