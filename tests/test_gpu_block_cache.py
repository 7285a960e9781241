"""GPU test of the device-block cache over small blocks."""
import numpy as np
import pytest

from helpers import gpu_for
from mrfmap_amd import release_device_cache, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [0, 2])
def test_small_blocks_left_by_other_contexts_give_the_same_map(first):
    """A map built on fresh memory, on blocks left by a different map (other
    frames at another voxel size, whose contents are in them), and on its own
    blocks again: bit for bit the same beliefs."""
    p, frames, _ = synth.make_workload("small")
    q, others, _ = synth.make_workload("small", res=0.05, seed=9)

    def build(params, fr):
        g = gpu_for(params, fr)
        g.perform_inference(max_iters=3)
        b = g.get_beliefs().view(np.uint32).copy()
        g.close()
        return b

    release_device_cache()
    want = build(p, frames[first:])
    release_device_cache()
    build(q, others)
    for _ in range(2):
        np.testing.assert_array_equal(build(p, frames[first:]), want)
