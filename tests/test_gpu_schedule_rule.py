"""GPU test of the rule that picks the ray kernels' schedule."""
import numpy as np
import pytest

from helpers import gpu_for
from mrfmap_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("msg,tables,ahead", [
    (_lib.MSG_F32, False, (16, 16)),
    (_lib.MSG_F16, False, (16, 8)),   # half the bytes per pair
    (_lib.MSG_BF16, False, (16, 8)),
    (_lib.MSG_MIXED_F16, False, (16, 16)),  # the window kernel reads FP32 messages
    (_lib.MSG_F16, True, (16, 16)),
])
def test_schedule_of_a_camera_with_many_pairs(msg, tables, ahead, monkeypatch):
    """One keyframe with more than 32 M pairs."""
    monkeypatch.delenv("MRF_RAY_SCHED", raising=False)
    p, frames, _ = synth.make_workload("batched", frames=1, res=0.0115, shapes=[(480, 640)], msg_dtype=msg)
    if tables:
        n = p.lookup_cells()
        p.use_polys = True
        p.depth_sigma_lookup = np.tile(np.array([p.res, 0.1 * p.res, 0.0], np.float32), n)
        p.depth_bias_lookup = np.zeros(3 * n, np.float32)
    g = gpu_for(p, frames)
    st = g.perform_inference(max_iters=1)
    assert st["pairs_per_iter"] > 32 << 20
    assert _lib.RAY_SCHEDULES[st["ray_sched"]] == ahead


def test_schedule_of_a_small_camera(monkeypatch):
    monkeypatch.delenv("MRF_RAY_SCHED", raising=False)
    p, frames, _ = synth.make_workload("small", frames=1)
    assert _lib.RAY_SCHEDULES[gpu_for(p, frames).perform_inference(max_iters=1)["ray_sched"]] == (16, 8)
