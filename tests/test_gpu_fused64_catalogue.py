"""Every FP64 schedule number that the library has taken (needs a GPU): 2 to 8
are accepted, run the fused kernel and give the two-kernel step's bits, also
where a fixed chunk length is longer than the grid; 9 is refused. On a small
walled domain the numbers are accepted and run the two-kernel step."""
import numpy as np
import pytest

from lbman3d_amd import abi

pytestmark = pytest.mark.gpu

SCHEDULES = range(2, 9)


def run(cfg, q, schedule):
    from lbman3d_amd.solver import DeviceSolver
    with DeviceSolver(cfg) as s:
        s.set_schedule(schedule)
        s.upload_state(q=q)
        s.step(3)
        kernels = list(s.profile_kernels(1))
        return s.schedule_name(schedule), kernels, dict(s.state(), F=s.force(), f=s.populations())


@pytest.mark.parametrize("bc,dims", [(abi.FullyPeriodicConfig, (33, 18, 70)), (abi.FullyPeriodicConfig, (40, 9, 131)),
                                     (abi.ChannelConfig, (20, 13, 40))], ids=["periodic70", "periodic131", "channel"])
def test_every_schedule_number(bc, dims):
    from lbman3d_amd.solver import DeviceSolver, LbmError
    periodic = bc is abi.FullyPeriodicConfig
    cfg = abi.make_config(*dims, bc, abi.Params(ALPHA=0.03, LAMBDA=0.5), advection=abi.ADV_UPWIND, precision=abi.FP64)
    q = abi.seed_director_field(23, *dims)
    _, _, ref = run(cfg, q, 1)
    names = set()
    for schedule in SCHEDULES:
        name, kernels, got = run(cfg, q, schedule)
        print(f"case FP64 schedule {schedule} {name} {dims}", flush=True)
        names.add(name)
        assert kernels == (["fused_step_f64"] if periodic else ["force_lbm_f64", "qstep_f64"])
        for k in ref:
            np.testing.assert_array_equal(got[k], ref[k], err_msg=f"{name} {k}")
    assert len(names) == len(SCHEDULES) and all(n.startswith("fused:fp64:") for n in names)
    with DeviceSolver(cfg) as s, pytest.raises(LbmError, match="schedule out of range"):
        s.set_schedule(9)
