"""GPU test of the traversal lists kept across changes of the keyframe set."""
import numpy as np
import pytest

from helpers import gpu_for, oracle_for
from mrfmap_amd import _lib, synth

pytestmark = pytest.mark.gpu


def _same_lists(g, o, ncam):
    for k in range(ncam):
        (gr, gi), (orr, oi) = g.get_traversal(k), o.traversal(k)
        np.testing.assert_array_equal(gr, orr)
        np.testing.assert_array_equal(gi, oi)


@pytest.mark.parametrize("activation", [_lib.ACT_FULL_RAY, _lib.ACT_ENDPOINT])
def test_lists_after_adding_moving_and_loading_match_oracle(activation):
    """Keyframes that do not change keep their lists when another is added or
    moved or a map is loaded (whose bricks may lie on their rays): after each
    change every list is the oracle's, bit for bit, and the marginals of a
    2-iteration call stay within the FP32 bound of 1e-3."""
    p, frames, _ = synth.make_workload("small", activation=activation)
    g, o = gpu_for(p, frames[:2]), oracle_for(p, frames[:2])

    def check(ncam):
        g.perform_inference(max_iters=2)
        o.perform_inference(2)
        assert g.num_bricks() == o.num_bricks()
        _same_lists(g, o, ncam)
        assert np.abs(g.get_alphas().astype(np.float64) - o.alphas()).max() <= 1e-3

    check(2)
    for pose, K, depth in frames[2:]:
        g.add_camera_with_depth(pose, depth, K)
        o.add_camera(pose, depth, K)
    check(4)
    moved = frames[1][0].copy()
    moved[:3, 3] += (0.05, -0.1, 0.02)
    g.set_pose(1, moved)
    o.set_pose(1, moved)
    check(4)
    pts = np.random.default_rng(2).uniform(1, 70, (200, 3)).astype(np.float32)
    occ = np.full(len(pts), 0.8, np.float32)
    g.load_map(pts, occ)
    o.load_map(pts, occ)
    check(4)
    g.set_pose(1, frames[1][0])
    o.set_pose(1, frames[1][0])
    check(4)
