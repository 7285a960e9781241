"""GPU tests of the incidence lists' layout at the edges of its tiles and batches."""
import numpy as np
import pytest

from helpers import gpu_for, oracle_for
from mrfmap_amd import _lib, gvdb_params

pytestmark = pytest.mark.gpu


def _room(rows, cols, focal, near, far, vis, seed=5):
    """Two keyframes of random depths in a 2 x 2 x 1 m grid at 4 cm."""
    p = gvdb_params()
    p.rows, p.cols = rows, cols
    p.K = np.array([[focal, 0, cols / 2], [0, focal, rows / 2], [0, 0, 1]], np.float32)
    p.res, p.prior, p.dims = 0.04, 0.1, np.array([2.0, 2.0, 1.0], np.float32)
    p.const_sigmasq_poly = [0.02, 0.0, 0.0]
    p.brick_local_vis = vis
    rng = np.random.default_rng(seed)
    frames = []
    for yaw in (0.0, 0.4):
        c, s = np.cos(yaw), np.sin(yaw)
        pose = np.eye(4, dtype=np.float32)
        pose[:3, :3] = np.array([[s, 0, c], [-c, 0, s], [0, -1, 0]])
        pose[:3, 3] = (-0.9, 0.03, 0.5)
        depth = rng.uniform(near, far, (rows, cols)).astype(np.float32)
        depth[rng.uniform(size=depth.shape) < (0.2 if depth.size < 100000 else 0.98)] = 0
        frames.append((pose, p.K, depth))
    return p, frames


@pytest.mark.parametrize("vis", [_lib.VIS_BRICK_LOCAL, _lib.VIS_CARRY])
@pytest.mark.parametrize("rows,cols,focal,near,far", [
    (1, 1, 5.0, 1.0, 1.5),     # one ray
    (8, 8, 9.0, 0.05, 0.3),    # one tile, rays of window records only and short fronts
    (9, 17, 12.0, 0.1, 1.8),   # ragged tiles, rays of every length, beyond the grid
    (40, 24, 30.0, 1.6, 1.8),  # long fronts, several batches per slice
    (48, 48, 400.0, 0.3, 0.4),  # voxels met by every ray: segments over several 512-position tiles
    (744, 760, 700.0, 0.2, 1.8),  # 8835 tiles, most of few rays
])
def test_lists_and_marginals_match_oracle(rows, cols, focal, near, far, vis):
    """Lists bit for bit; marginals after 2 iterations within the 1e-3 that
    the other parity tests allow."""
    p, frames = _room(rows, cols, focal, near, far, vis)
    frames[0][2].flat[0] = 0.5 * (near + far)
    g, o = gpu_for(p, frames), oracle_for(p, frames)
    g.perform_inference(max_iters=2)
    o.perform_inference(2)
    for k in range(len(frames)):
        (gr, gi), (orr, oi) = g.get_traversal(k), o.traversal(k)
        np.testing.assert_array_equal(gr, orr)
        np.testing.assert_array_equal(gi, oi)
    assert np.abs(g.get_alphas().astype(np.float64) - o.alphas()).max() <= 1e-3


@pytest.mark.parametrize("iters", [1, 64, 65, 130])
def test_replays_without_a_wait_match_replays_with_one(iters):
    """Without a tolerance the host waits once per 64 iterations; the residual
    of every iteration and the marginals are those of a call that waits after
    each (a tolerance below every residual but 0)."""
    p, frames = _room(9, 17, 12.0, 0.1, 1.8, _lib.VIS_BRICK_LOCAL)
    runs = []
    for tol in (0.0, 1e-300):
        g = gpu_for(p, frames)
        st = g.perform_inference(max_iters=iters, tol=tol)
        runs.append((st["iters"], g.get_trace()[0], g.get_alphas()))
    (n0, r0, a0), (n1, r1, a1) = runs
    assert n0 == len(r0) == iters and n1 == len(r1)
    np.testing.assert_array_equal(r0[:n1], r1)
    if n1 == iters:
        np.testing.assert_array_equal(a0, a1)
