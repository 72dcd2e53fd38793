"""Third-pipeline batch tiles: every simulation's tile shape and the cut of
all columns into one range per block (needs a GPU).

Every plane of a range runs the same code, so a tile shape gives the same bits
however the columns are cut. (Between tile shapes a column changes between the
tile and its ring, whose Q updates are two copies that the compiler may
contract differently.) Against single simulations, both FP32, the agreement
is to rounding after a few steps (the tolerances of test_gpu_batch.py).
"""
import numpy as np
import pytest

from conftest import BC_BY_NAME
from lbman3d_amd import abi

pytestmark = pytest.mark.gpu

# One column tile and several, rows shorter and longer than a tile, planes
# fewer than the shortest piece and more than the longest chunk; periodic,
# wall-aware and shell-pass simulations.
SIMS = [("FullyPeriodic", (33, 9, 7), abi.ADV_UPWIND), ("SlitFreeSlip", (48, 30, 8), abi.ADV_CENTRED),
        ("FullyPeriodic", (24, 17, 70), abi.ADV_CENTRED), ("Channel", (97, 8, 10), abi.ADV_UPWIND),
        ("SlitNoSlip", (65, 12, 20), abi.ADV_UPWIND), ("MovingLidZ", (16, 18, 22), abi.ADV_CENTRED)]
STEPS = 5


def rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


@pytest.fixture(scope="module")
def reference():
    from lbman3d_amd.solver import BatchSolver, DeviceSolver, batch_tile_index
    cfgs = [abi.make_config(*dims, BC_BY_NAME[bc], abi.Params(LAMBDA=0.5, ALPHA=0.03), advection=adv,
                            precision=abi.FP32_SHIFTED) for bc, dims, adv in SIMS]
    qs = [abi.seed_director_field(600 + i, c.nx, c.ny, c.nz) for i, c in enumerate(cfgs)]

    def run(tile, limit):
        with BatchSolver(cfgs) as b:
            b.set_tile(batch_tile_index(tile))
            b.set_grid_limit(limit)
            for i, q in enumerate(qs):
                b.upload_state(i, q=q)
            b.step(STEPS, use_graph=True)
            return [b.state(i) for i in range(len(cfgs))]

    single = []
    for c, q in zip(cfgs, qs):
        with DeviceSolver(c) as s:
            s.set_schedule(1)
            s.upload_state(q=q)
            s.step(STEPS)
            single.append(s.state())
    return run, {t: run(t, 0) for t in ("p2:rows:64", "p2:32x8x16", "p2:64x4x32")}, single


@pytest.mark.parametrize("tile,limit,uncut", [("p2:rows:64", 200, "p2:rows:64"), ("p2:rows:64", 1, "p2:rows:64"),
                                              ("p2:rows:64", 5, "p2:rows:64"), ("p2:32x8x64", 9, "p2:32x8x16"),
                                              ("p2:64x4x32", 3, "p2:64x4x32")])
def test_every_cut_gives_the_same_bits(reference, tile, limit, uncut):
    print(f"case batch split tile={tile} limit={limit}", flush=True)
    run, base, single = reference
    out, base = run(tile, limit), base[uncut]
    for i in range(len(SIMS)):
        for k in ("rho", "u", "q"):
            np.testing.assert_array_equal(out[i][k], base[i][k], err_msg=f"{i} {k}")
        assert rel(out[i]["q"], single[i]["q"]) < 2e-6, i
        assert rel(out[i]["u"], single[i]["u"]) < 2e-5, i
        assert np.max(np.abs(out[i]["rho"] - single[i]["rho"])) < 2e-6, i
