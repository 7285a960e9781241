"""GPU tests of the ray walks in the ranges where they change their arithmetic."""
import numpy as np
import pytest

from helpers import gpu_for, oracle_for
from mrfmap_amd import _lib, gvdb_params

pytestmark = pytest.mark.gpu


def _tube(res, activation):
    """Two keyframes along a 2 x 0.2 x 0.2 m tube, one looking obliquely; at
    1 mm the walks' products exceed 2^52 and stay in 64-bit integers, at 4 mm
    they are held in FP64."""
    p = gvdb_params()
    p.rows, p.cols = 21, 27
    p.K = np.array([[20, 0, 13], [0, 20, 10], [0, 0, 1]], np.float32)
    p.res, p.prior, p.dims = res, 0.1, np.array([2.0, 0.2, 0.2], np.float32)
    p.const_sigmasq_poly = [1.5 * res, 0.0, 0.0]
    p.activation = activation
    rng = np.random.default_rng(3)
    frames = []
    for yaw, x in ((0.0, -0.9), (0.03, -0.7)):
        c, s = np.cos(yaw), np.sin(yaw)
        pose = np.eye(4, dtype=np.float32)
        pose[:3, :3] = np.array([[s, 0, c], [-c, 0, s], [0, -1, 0]])  # optical axis along x, turned by yaw
        pose[:3, 3] = (x, 0.01, 0.1)
        depth = rng.uniform(0.25, 1.2, (p.rows, p.cols)).astype(np.float32)
        depth[::5, ::4] = 0
        frames.append((pose, p.K, depth))
    return p, frames


@pytest.mark.parametrize("activation", [_lib.ACT_FULL_RAY, _lib.ACT_ENDPOINT])
@pytest.mark.parametrize("res", [0.001, 0.004])
def test_walks_match_oracle_on_both_sides_of_the_fp64_range(res, activation):
    """Lists bit for bit, marginals after 2 iterations, and the scoring walk's
    expected depth (a weighted mean of depths below 1.3 m in FP32 over up to
    2500 voxels, so within 2500 roundings of 1.3 x 2^-24 = 2e-4)."""
    p, frames = _tube(res, activation)
    g, o = gpu_for(p, frames), oracle_for(p, frames)
    g.perform_inference(max_iters=2)
    o.perform_inference(2)
    for k in range(len(frames)):
        (gr, gi), (orr, oi) = g.get_traversal(k), o.traversal(k)
        assert len(gi) > 100
        np.testing.assert_array_equal(gr, orr)
        np.testing.assert_array_equal(gi, oi)
    assert np.abs(g.get_alphas().astype(np.float64) - o.alphas()).max() <= 1e-3
    pose, K, depth = frames[1]
    rg, ro = g.evaluate(pose=pose, depth=depth, K=K), o.evaluate(pose, depth, K, acc_thresh=p.acc_thresh)
    # the maps themselves may differ by 1e-3 (above) at single voxels
    assert np.median(np.abs(rg["expected_depth"] - ro["expected_depth"])) <= 2e-4
