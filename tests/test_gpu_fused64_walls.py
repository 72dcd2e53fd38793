"""The fused FP64 step on domains with walls (needs a GPU): the periodic kernel
over every tile, then the shell passes over the cells within two cells of an
open face. Its results must be the two-kernel step's bit for bit. Grids with
walls have the fused schedules from 2^20 cells on; the sides here leave partial
tiles and a partial last z chunk."""
import numpy as np
import pytest

from conftest import BC_BY_NAME
from lbman3d_amd import abi

pytestmark = pytest.mark.gpu

BOX = abi.BCConfig(name="Box")
CASES = [(BC_BY_NAME["Channel"], (129, 101, 83), True), (BC_BY_NAME["AnchoredZ"], (110, 97, 101), False),
         (BC_BY_NAME["MovingLidZ"], (160, 96, 70), True), (BC_BY_NAME["SpecularXNoSlipY"], (67, 130, 125), False),
         (BOX, (103, 103, 103), True)]


@pytest.mark.parametrize("bc,dims,upwind", CASES, ids=[c[0].name for c in CASES])
def test_walled_fp64_tiles_equal_the_two_kernel_step(bc, dims, upwind):
    from lbman3d_amd.solver import DeviceSolver, LbmError
    cfg = abi.make_config(*dims, bc, abi.Params(ALPHA=0.03, LAMBDA=0.5, MU=0.002),
                          advection=abi.ADV_UPWIND if upwind else abi.ADV_CENTRED, precision=abi.FP64)
    q = abi.seed_director_field(17, *dims)

    def run(schedule):
        with DeviceSolver(cfg) as s:
            s.set_schedule(schedule)
            name = s.schedule_name(schedule)
            print(f"case walled FP64 {bc.name} {dims} {name}", flush=True)
            s.upload_state(q=q)
            s.step(2)
            s.step(3)
            return name, dict(s.state(), F=s.force(), f=s.populations())

    _, ref = run(1)
    schedule = 2
    while True:
        try:
            name, got = run(schedule)
        except LbmError:
            break
        assert name.startswith("fused:fp64:")
        for k, v in ref.items():
            np.testing.assert_array_equal(got[k], v, err_msg=f"{name} {k}")
        schedule += 1
    assert schedule > 2
