"""The two-kernel step at the edges of its grids (needs a GPU).

FP64 must reproduce the oracle bit for bit (rho, u, Q, populations and the
force of the last step); FP32 must stay within rounding of it: after 4 steps
from Q of order 0.3 an FP32 field has collected some tens of roundings of
6e-8, so Q and populations are held to 4e-6 and u, whose scale (the force of
one step) is formed from cancelling differences, to 1e-4 of its maximum.

The grids: single cells and planes (both faces at one cell), rows shorter
and longer than a wavefront, cell counts just below, at and above whole
blocks; every wall tag, walls on every face, mixed Q and velocity
periodicity, and a moving wall (whose slots read the density of every step).
"""
import numpy as np
import pytest

from conftest import BC_BY_NAME
from lbman3d_amd import abi
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu

_W = abi.WallSpec
BOX = abi.BCConfig(name="Box")   # Neumann, no-slip on every face
MIXED = abi.BCConfig(_W(abi.Neumann(), abi.Periodic()), _W(abi.Neumann(), abi.Periodic()),
                     _W(abi.Periodic(), abi.NoSlip()), _W(abi.Periodic(), abi.NoSlip()),
                     _W(abi.Periodic(), abi.Periodic()), _W(abi.Periodic(), abi.Periodic()), "Mixed")
LID = abi.BCConfig(_W(abi.Anchoring(0.4, 0.3, 1.1), abi.NoSlip()), _W(abi.Neumann(), abi.MovingWall(0.0, 0.02, -0.01)),
                   _W(abi.Periodic(), abi.Periodic()), _W(abi.Periodic(), abi.Periodic()),
                   _W(abi.Periodic(), abi.Periodic()), _W(abi.Periodic(), abi.Periodic()), "LidX")
ONE_SIDED = abi.BCConfig(_W(abi.Neumann(), abi.NoSlip()), _W(abi.Periodic(), abi.NoSlip()),
                         _W(abi.Periodic(), abi.NoSlip()), _W(abi.Anchoring(0.5, 0.9, 0.4), abi.NoSlip()),
                         _W(abi.Anchoring(0.5, 0.9, 0.4), abi.Periodic()), _W(abi.Periodic(), abi.Periodic()), "OneSided")
CASES = [(abi.FullyPeriodicConfig, (1, 1, 1)), (abi.FullyPeriodicConfig, (2, 1, 3)), (abi.FullyPeriodicConfig, (16, 16, 1)),
         (abi.FullyPeriodicConfig, (17, 5, 3)), (abi.FullyPeriodicConfig, (129, 2, 1)), (abi.ChannelConfig, (20, 13, 5)),
         (abi.SlitConfig, (64, 4, 2)), (abi.SlitNoSlipConfig, (65, 3, 4)), (BOX, (5, 7, 9)), (BOX, (3, 2, 2)),
         (MIXED, (9, 6, 5)), (ONE_SIDED, (8, 7, 6)), (ONE_SIDED, (2, 1, 1)), (LID, (7, 11, 6)), (BC_BY_NAME["MovingLidZ"], (33, 4, 8)),
         (BC_BY_NAME["AnchoredZ"], (10, 9, 2))]


@pytest.mark.parametrize("bc,dims", CASES, ids=[f"{b.name}-{'x'.join(map(str, d))}" for b, d in CASES])
@pytest.mark.parametrize("upwind", [False, True])
def test_two_kernel_step_on_edge_grids(bc, dims, upwind):
    from lbman3d_amd.solver import DeviceSolver
    print(f"case two-kernel {bc.name} {dims} upwind={upwind}", flush=True)
    params = abi.Params(ALPHA=0.04, LAMBDA=0.5, MU=0.01)
    adv = abi.ADV_UPWIND if upwind else abi.ADV_CENTRED
    cfg = abi.make_config(*dims, bc, params, advection=adv, precision=abi.FP64)
    q = abi.seed_director_field(5, *dims)
    o = Oracle(cfg)
    o.set_state(q=q)
    o.step(4)
    ref = dict(o.state(), f=o.populations(), F=o.force())
    got = {}
    for precision in (abi.FP64, abi.FP32_SHIFTED):
        with DeviceSolver(abi.config_copy(cfg, precision=precision)) as s:
            s.set_schedule(1)
            s.upload_state(q=q)
            s.step(1)
            s.step(3)
            got[precision] = dict(s.state(), f=s.populations(), F=s.force())
    for k in ("rho", "u", "q", "f", "F"):
        np.testing.assert_array_equal(np.asarray(got[abi.FP64][k]).reshape(-1), np.asarray(ref[k]).reshape(-1), err_msg=k)
    rel = lambda k: np.max(np.abs(np.asarray(got[abi.FP32_SHIFTED][k]).reshape(-1) - np.asarray(ref[k]).reshape(-1))) \
        / max(np.max(np.abs(ref[k])), 1e-30)
    assert rel("q") < 4e-6 and rel("f") < 4e-6
    if np.max(np.abs(ref["u"])) > 1e-6:
        assert rel("u") < 1e-4
