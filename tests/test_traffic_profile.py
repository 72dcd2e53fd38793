"""The committed HBM traffic of the FP64 step names the schedules that run."""
import json
import os
import re

from test_bench_contract import ROOT, _bench


def test_fp64_traffic_of_the_current_schedules():
    V = 256 ** 3
    with open(os.path.join(ROOT, "profiles", "fused_step_f64_256cube_traffic.json")) as fp:
        entries = json.load(fp)["by_schedule"]
    with open(os.path.join(ROOT, "lbman3d_amd", "csrc", "kernels_fp64.hip")) as fp:
        names = ["fused:" + n for n in re.findall(r'"(fp64:[0-9x]+)"', fp.read())]
    assert len(names) == 7
    # the tiles that tuning chooses from have a measurement of their kernel
    for name in names[:2]:
        _, roof = _bench().roofline({"fused_step_f64": 1.6}, V, name, step_ms=1.6)
        assert 368 * V < roof["traffic"] < 1.5 * 368 * V
        assert "same_launch_as" not in entries[name]
    # an entry belongs to a kernel that runs, or says that it does not
    for name, e in entries.items():
        runs = "fused64_kernel" in e["symbol"]
        assert runs == (name in names) and runs != e.get("retired", False), name
