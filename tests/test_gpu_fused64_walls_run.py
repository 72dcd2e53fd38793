"""On walled FP64 domains from 2^20 cells on every fused schedule runs the fused
kernel (the name of the launch says so) and gives the two-kernel step's bits
(needs a GPU). One cell plane less than the limit, the same numbers run the
two-kernel step."""
import numpy as np
import pytest

from conftest import BC_BY_NAME
from lbman3d_amd import abi

pytestmark = pytest.mark.gpu

DIMS = (128, 91, 91)   # 1,059,968 cells


def run(cfg, q, schedule):
    from lbman3d_amd.solver import DeviceSolver
    with DeviceSolver(cfg) as s:
        s.set_schedule(schedule)
        s.upload_state(q=q)
        s.step(3)
        kernels = set(s.profile_kernels(1))
        return kernels, dict(s.state(), F=s.force(), f=s.populations())


def schedules(cfg):
    from lbman3d_amd.solver import DeviceSolver, LbmError
    names = []
    with DeviceSolver(cfg) as s:
        auto = s.schedule_name(0)
        while True:
            try:
                names.append(s.schedule_name(2 + len(names)))
            except LbmError:
                return auto, names


@pytest.mark.parametrize("bc", ["Channel", "AnchoredZ", "MovingLidZ"])
def test_walled_domains_run_the_fused_kernel(bc):
    cfg = abi.make_config(*DIMS, BC_BY_NAME[bc], abi.Params(ALPHA=0.03, LAMBDA=0.5, MU=0.002), advection=abi.ADV_UPWIND,
                          precision=abi.FP64)
    q = abi.seed_director_field(19, *DIMS)
    auto, names = schedules(cfg)
    assert auto == "auto" and len(names) == 7 and len(set(names)) == 7
    kernels, ref = run(cfg, q, 1)
    assert kernels == {"qstep_f64", "force_lbm_f64"}
    for i, name in enumerate(names):
        print(f"case walled FP64 {bc} {name}", flush=True)
        kernels, got = run(cfg, q, 2 + i)
        assert kernels == {"fused_step_f64"}, name
        for k, v in ref.items():
            np.testing.assert_array_equal(got[k], v, err_msg=f"{name} {k}")


def test_smaller_walled_domains_run_the_two_kernel_step():
    dims = (DIMS[0], DIMS[1], 90)
    assert np.prod(dims) < 1 << 20 < np.prod(DIMS)
    print("case walled FP64 below the limit", flush=True)
    cfg = abi.make_config(*dims, BC_BY_NAME["Channel"], precision=abi.FP64)
    assert schedules(cfg)[0] == "auto:two-kernel"
    kernels, _ = run(cfg, abi.seed_director_field(19, *dims), 2)
    assert kernels == {"qstep_f64", "force_lbm_f64"}
