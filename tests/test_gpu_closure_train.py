"""Training kernels of the closure on grids at the edges of their tiles (needs
a GPU): one tile and several per block, z and y extents that are no multiple of
a block's tile, and more steps in one call than are kept before the losses are
read. Gradients against the oracle with bf16-rounded operands, to the tolerance
of test_gpu_closure.py; one long call against the same steps taken one by one,
whose arithmetic is the same in the same order.
"""
import numpy as np
import pytest

from oracle import closure_ref as cr

pytestmark = pytest.mark.gpu

H = 32


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def case(dims, seed):
    v = dims[0] * dims[1] * dims[2]
    rng = np.random.default_rng(seed)
    return rng.normal(size=(8, v)), rng.normal(size=(5, v)) * 0.2, cr.he_init(H, seed)


@pytest.mark.parametrize("dims", [(16, 8, 8), (16, 12, 20), (48, 8, 12), (80, 20, 8), (64, 32, 36)])
def test_gradient_matches_oracle(dims):
    from lbman3d_amd.closure import ClosureNet
    print(f"case closure gradient dims={dims}", flush=True)
    nx, ny, nz = dims
    x, t, p = case(dims, 11)
    with ClosureNet(*dims, hidden=H, seed=1) as n:
        n.params = p
        loss, g = n.loss_and_grad(x, t)
    grid = lambda a: a.reshape(a.shape[0], nz, ny, nx).transpose(1, 2, 3, 0)
    loss_r, gr = cr.loss_and_grad(p, grid(x), grid(t), H, bf16=True)
    assert loss == pytest.approx(loss_r, rel=2e-3)
    o = 0
    for ci, co in cr.layer_shapes(H):
        nw = 27 * ci * co
        for lo, hi in ((o, o + nw), (o + nw, o + nw + co)):
            assert rel(g[lo:hi], gr[lo:hi]) < 2e-2, (ci, co, lo)
        o += nw + co


@pytest.mark.parametrize("iters", [1, 64, 65, 130])
def test_one_call_equals_single_steps(iters):
    from lbman3d_amd.closure import ClosureNet
    print(f"case closure train iters={iters}", flush=True)
    dims = (16, 12, 20)
    x, t, p = case(dims, 12)
    out = []
    for calls in ([iters], [1] * iters):
        with ClosureNet(*dims, hidden=H, seed=1) as n:
            n.params = p
            n.add_sample(x, t)
            losses = [n.train(c, 1e-3) for c in calls]
            out.append((n.params, float(np.mean(losses))))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == pytest.approx(out[1][1], rel=1e-12)
