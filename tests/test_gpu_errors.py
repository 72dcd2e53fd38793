"""Calls after a failed one in the same thread (needs a GPU). A grid of 10^9
FP64 cells takes 464 GB, so its creation is refused with the allocation's error
and nothing runs; what the thread does next must not report that error again."""
import numpy as np
import pytest

from lbman3d_amd import abi

pytestmark = pytest.mark.gpu

DIMS = (9, 8, 7)


def too_large():
    from lbman3d_amd.solver import DeviceSolver, LbmError
    with pytest.raises(LbmError, match="out of memory"):
        DeviceSolver(abi.make_config(1000, 1000, 1000, precision=abi.FP64))


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32_SHIFTED])
def test_calls_after_a_grid_that_does_not_fit(precision):
    from lbman3d_amd.solver import DeviceSolver
    print(f"case after out of memory precision={precision}", flush=True)
    cfg = abi.make_config(*DIMS, precision=precision)
    q = abi.seed_director_field(3, *DIMS)
    with DeviceSolver(cfg) as s:
        s.upload_state(q=q)
        s.step(2)
        ref = s.state()
    too_large()
    with DeviceSolver(cfg) as s:
        too_large()
        s.upload_state(q=q)
        too_large()
        s.step(2)
        too_large()
        st = s.state()
    for k in ref:
        np.testing.assert_array_equal(st[k], ref[k])
