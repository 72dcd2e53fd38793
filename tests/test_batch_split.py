"""The cut of a batch's columns into one range per block, on the CPU
(tests/cpp/batch_split_check.cpp on lbman3d_amd/csrc/batch_split.hpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_plane_once_and_no_range_too_long(tmp_path):
    exe = tmp_path / "batch_split_check"
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", os.path.join(ROOT, "tests", "cpp", "batch_split_check.cpp"),
                        "-o", str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
