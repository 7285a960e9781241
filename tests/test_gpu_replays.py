"""GPU test of iterations replayed back to back against iterations with a wait
after each."""
import numpy as np
import pytest

from helpers import gpu_for
from mrfmap_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wait", ["timed", "reference"])
@pytest.mark.parametrize("iters", [1, 63, 64, 65, 130])
def test_replays_give_every_residual_and_the_marginals(iters, wait):
    """Iterations launched without a wait (the residuals are read once per 64)
    against the same number with one: launched kernel by kernel, and replayed
    with a reference that stops nothing.  Both run every iteration whatever the
    residual is; the map still changes in each of the 130, so that a residual read
    from another iteration is seen."""
    p, frames, _ = synth.make_workload("small", res=0.06, seed=9)
    g = gpu_for(p, frames)
    st = g.perform_inference(max_iters=iters)
    assert st["graph"] == 1 and st["iters"] == iters
    resid, _ = g.get_trace()
    assert len(resid) == iters and (resid > 0).all() and st["residual"] == resid[-1]
    h = gpu_for(p, frames)
    if wait == "timed":
        h.set_launch_mode(_lib.LAUNCH_TIMED)
    else:
        h.prepare()
        h.set_reference(np.zeros((h.num_bricks(), 512), np.float32))
    sh = h.perform_inference(max_iters=iters)
    assert sh["iters"] == iters and sh["residual"] == st["residual"]
    np.testing.assert_array_equal(resid, h.get_trace()[0])
    np.testing.assert_array_equal(g.get_beliefs().view(np.uint32), h.get_beliefs().view(np.uint32))
