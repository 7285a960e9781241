"""GPU test of the gradient's reduction over per-wave rows at its chunk edges."""
import numpy as np
import pytest

import oracle.mlp as omlp
from mrfmap_amd import GVDBInference, gvdb_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 8192, 8193, 16385, 65537])
def test_gradient_over_one_and_several_chunks_of_rows(n):
    """256 rows of partial sums fill a chunk exactly at 8192 samples; one
    sample more starts a second; 65537 samples take the largest grid.  Each
    sample's BF16 operands may round to the other neighbour (2^-9) than in
    the oracle, and FP32 sums of n terms add n 2^-24 / 2 of the largest: well
    inside 1/256 of the largest gradient entry of each tensor."""
    g = GVDBInference(params=gvdb_params())
    rng = np.random.default_rng(n)
    params = omlp.init_params(7)
    X = rng.normal(0, 1, (n, 32)).astype(np.float32)
    t = rng.normal(0, 2, n).astype(np.float32)
    loss, grad = g.mlp_grad(params, X, t)
    lo, go = omlp.loss_and_grad(params, X, t, bf16_ops=True)
    assert abs(loss - lo) <= 1e-5 * max(1.0, lo)
    for name, sl in (("W1", omlp.W1), ("b1", omlp.B1), ("W2", omlp.W2), ("b2", omlp.B2), ("w3", omlp.W3),
                     ("b3", omlp.B3)):
        assert np.abs(grad[sl] - go[sl]).max() <= np.abs(go[sl]).max() / 256 + 1e-9, name
