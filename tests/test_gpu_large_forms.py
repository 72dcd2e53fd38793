"""The two-kernel step in the forms that large arrays take (needs a GPU): plain
block order and non-temporal stores above 9 MB an array, and 64-bit cell
offsets where the 15 populations exceed 4 GiB.

A state that repeats along a periodic z axis stays so, cell by cell the same
arithmetic, so a long grid is compared with the oracle on one period of it:
FP64 bit for bit, FP32 to rounding (the tolerances of test_gpu_split_step.py).
A box with walls on every face and odd sides is compared whole. The boundary
sets are those that select different kernels: no wall; walls whose clamped
values are the ghosts; anchored and moving walls, whose are not."""
import numpy as np
import pytest

from conftest import BC_BY_NAME
from lbman3d_amd import abi
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu

_W = abi.WallSpec
LID_X = abi.BCConfig(_W(abi.Anchoring(0.4, 0.3, 1.1), abi.NoSlip()), _W(abi.Neumann(), abi.MovingWall(0.0, 0.02, -0.01)),
                     _W(abi.Periodic(), abi.Periodic()), _W(abi.Periodic(), abi.Periodic()),
                     _W(abi.Periodic(), abi.Periodic()), _W(abi.Periodic(), abi.Periodic()), "LidX")
BOX = abi.BCConfig(name="Box")   # Neumann, no-slip on every face
RUN_BYTES = 9 << 20              # arrays up to this size take the other form
STEPS = 3


def config(dims, bc, upwind, precision):
    return abi.make_config(*dims, bc, abi.Params(ALPHA=0.04, LAMBDA=0.5, MU=0.01),
                           advection=abi.ADV_UPWIND if upwind else abi.ADV_CENTRED, precision=precision)


def oracle(cfg, q):
    o = Oracle(cfg)
    o.set_state(q=q)
    o.step(STEPS)
    return {k: np.asarray(v) for k, v in dict(o.state(), F=o.force()).items()}


def compare(cfg, q, ref, periods, cells, with_force):
    """ref: the oracle's fields of one period of `cells` cells."""
    from lbman3d_amd.solver import DeviceSolver
    fp32 = cfg.precision == abi.FP32_SHIFTED
    with DeviceSolver(cfg) as s:
        s.set_schedule(1)
        s.upload_state(q=q)
        s.step(1)
        s.step(STEPS - 1)
        got = dict(s.state(), **({"F": s.force()} if with_force else {}))
    for k, v in got.items():
        v = np.asarray(v).reshape(-1, periods, cells)
        r = ref[k].reshape(-1, cells)
        for c in range(len(r)):
            for p in range(periods):
                if not fp32:
                    np.testing.assert_array_equal(v[c, p], r[c], err_msg=f"{k}{c} period {p}")
                elif k != "F":
                    scale = np.max(np.abs(r)) if k != "u" else max(np.max(np.abs(ref["u"])), 1e-30)
                    assert np.max(np.abs(v[c, p] - r[c])) < (1e-4 if k == "u" else 4e-6) * scale, f"{k}{c} period {p}"


PERIODS = {"above9MB": {abi.FP64: 101, abi.FP32_SHIFTED: 211}, "above4GiB": {abi.FP64: 2801, abi.FP32_SHIFTED: 5601}}
BCS = [(abi.FullyPeriodicConfig, True), (abi.ChannelConfig, False), (LID_X, True)]


@pytest.mark.parametrize("size,bc,upwind,precision",
                         [("above9MB", b, u, p) for b, u in BCS for p in (abi.FP64, abi.FP32_SHIFTED)]
                         + [("above4GiB", b, u, abi.FP64) for b, u in BCS]
                         + [("above4GiB", LID_X, True, abi.FP32_SHIFTED)],
                         ids=lambda v: v if isinstance(v, str) else getattr(v, "name", str(v)))
def test_repeated_state(size, bc, upwind, precision):
    dims = (37, 29, 12)
    cells = dims[0] * dims[1] * dims[2]
    periods = PERIODS[size][precision]
    value = 8 if precision == abi.FP64 else 4
    assert cells * periods * value > RUN_BYTES
    assert (15 * cells * periods * value >= 1 << 32) == (size == "above4GiB")
    print(f"case two-kernel {size} {bc.name} precision={precision} periods={periods}", flush=True)
    q = abi.seed_director_field(11, *dims).reshape(5, cells)
    ref = oracle(config(dims, bc, upwind, abi.FP64), q)
    big = config((dims[0], dims[1], dims[2] * periods), bc, upwind, precision)
    compare(big, np.tile(q, (1, periods)), ref, periods, cells, size == "above9MB")


@pytest.mark.parametrize("bc,dims", [(BOX, (109, 107, 103)), (BC_BY_NAME["AnchoredZ"], (113, 110, 97)),
                                     (BC_BY_NAME["MovingLidZ"], (131, 67, 137))],
                         ids=["Box", "AnchoredZ", "MovingLidZ"])
def test_walls_on_a_large_grid(bc, dims):
    cells = dims[0] * dims[1] * dims[2]
    assert 8 * cells > RUN_BYTES
    print(f"case two-kernel large {bc.name} {dims}", flush=True)
    cfg = config(dims, bc, True, abi.FP64)
    q = abi.seed_director_field(12, *dims)
    compare(cfg, q, oracle(cfg, q), 1, cells, True)
