"""The short form of the FP64 push's move along an axis against the reference's
tests of cell, direction and receivers, compiled for the CPU
(tests/cpu/receiver_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_axis_step(tmp_path):
    exe = tmp_path / "receiver_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "0buf_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpu", "receiver_check.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
