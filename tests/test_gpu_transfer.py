"""Fields between host and device at the edges of the transfer's pieces (needs
a GPU). Everything here is exact: FP64 fields are copies, FP32 fields are the
values (or, for the density, the values less rho0) rounded once to 32 bits, and
the populations of an uploaded state are Feq in the stated operand order."""
import threading

import numpy as np
import pytest

from lbman3d_amd import abi

pytestmark = pytest.mark.gpu

E = np.array([(0, 0, 0), (1, 0, 0), (0, 1, 0), (-1, 0, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 1), (-1, 1, 1),
              (-1, -1, 1), (1, -1, 1), (1, 1, -1), (-1, 1, -1), (-1, -1, -1), (1, -1, -1)], dtype=float)
W = np.array([2.0 / 9] + [1.0 / 9] * 6 + [1.0 / 72] * 8)
# one cell, a lane short of and past a wavefront, one piece and a cell more
# (1 MiB over 9 values of 8 bytes: 14,528 cells; of 4 bytes: 29,120), several
# pieces, and enough bytes for several threads (24 MiB of host values)
DIMS = [(1, 1, 1), (63, 1, 1), (13, 5, 1), (14528, 1, 1), (14529, 1, 1), (29121, 1, 1), (41, 37, 29), (80, 75, 60)]


def feq(rho, u):
    u2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
    out = []
    for e, w in zip(E, W):
        ue = u[0] * e[0] + u[1] * e[1] + u[2] * e[2]
        out.append(w * rho * (1.0 + 3.0 * ue + 4.5 * ue * ue - 1.5 * u2))
    return np.array(out)


def fields(V, seed):
    rng = np.random.default_rng(seed)
    return 1.1 + 0.01 * rng.normal(size=V), 0.02 * rng.normal(size=(3, V)), 0.3 * rng.normal(size=(5, V))


def stored(x, fp32, base=0.0):
    return base + (x - base).astype(np.float32).astype(np.float64) if fp32 else x


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_SHIFTED])
@pytest.mark.parametrize("dims", DIMS)
def test_state_round_trip_and_equilibrium(dims, precision):
    from lbman3d_amd.solver import DeviceSolver
    print(f"case transfer {dims} precision={precision}", flush=True)
    fp32 = precision == abi.FP32_SHIFTED
    cfg = abi.make_config(*dims, abi.FullyPeriodicConfig, abi.Params(kDensity=1.1), precision=precision)
    V = int(np.prod(dims))
    rho, u, q = fields(V, 3)
    pops = lambda r, v: feq(r, v) if not fp32 else \
        (feq(r, v) - W[:, None] * 1.1).astype(np.float32).astype(np.float64) + W[:, None] * 1.1
    with DeviceSolver(cfg) as s:
        st = s.state()
        np.testing.assert_array_equal(st["rho"], np.full(V, 1.1))
        assert not st["u"].any() and not st["q"].any()
        np.testing.assert_array_equal(s.populations(), pops(np.full(V, 1.1), np.zeros((3, V))))
        s.upload_state(rho=rho, u=u, q=q)
        st = s.state()
        np.testing.assert_array_equal(st["rho"], stored(rho, fp32, 1.1 if fp32 else 0.0))
        np.testing.assert_array_equal(st["u"], stored(u, fp32))
        np.testing.assert_array_equal(st["q"], stored(q, fp32))
        np.testing.assert_array_equal(s.populations(), pops(rho, u))
        # a partial upload keeps the other fields and takes them from the device
        rho2, _, q2 = fields(V, 4)
        s.upload_state(q=q2)
        np.testing.assert_array_equal(s.populations(), pops(st["rho"], st["u"]))
        s.upload_state(rho=rho2)
        np.testing.assert_array_equal(s.populations(), pops(rho2, st["u"]))
        now = s.state()
        np.testing.assert_array_equal(now["q"], stored(q2, fp32))
        np.testing.assert_array_equal(now["u"], st["u"])
        f = pops(rho, u)
        s.upload_populations(f)
        np.testing.assert_array_equal(s.populations(), stored_pops(f, fp32))
        s.upload_force(u)
        np.testing.assert_array_equal(s.force(), stored(u, fp32))


def stored_pops(f, fp32):
    b = W[:, None] * 1.1
    return b + (f - b).astype(np.float32).astype(np.float64) if fp32 else f


def test_handles_of_several_threads_share_the_staging():
    from lbman3d_amd.solver import DeviceSolver
    print("case transfer threads", flush=True)
    bad = []

    def work(seed):
        dims = (60 + seed, 40, 30)
        V = int(np.prod(dims))
        rho, u, q = fields(V, seed)
        for _ in range(3):
            with DeviceSolver(abi.make_config(*dims, precision=abi.FP64)) as s:
                s.upload_state(rho=rho, u=u, q=q)
                st = s.state()
                if not (np.array_equal(st["rho"], rho) and np.array_equal(st["u"], u) and np.array_equal(st["q"], q)):
                    bad.append(seed)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
