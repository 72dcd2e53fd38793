"""The host side of the field transfers (lbman3d_amd/csrc/transfer.hip) on a
stand-in for the HIP runtime (tests/cpp/transfer_check.cpp), compiled here for
the host alone: no GPU. Each scenario runs in a process of its own, on a set
that one thread moves and on one that several threads move, and compares every
value."""
import os
import subprocess

import pytest

from lbman3d_amd.build import _hipcc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("transfer") / "transfer_check"
    cmd = [_hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "cpp", "transfer_check.cpp"), "-no-hip-rt", "-pthread",
           "-Wl,--unresolved-symbols=ignore-in-object-files", "-o", str(exe)]   # the device code's image
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("scenario", ["plain", "earlier-error", "other-device", "helper-buffer", "helper-event",
                                      "helper-device", "host-memory"])
def test_transfer(check, scenario):
    r = subprocess.run([str(check), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
