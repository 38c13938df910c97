"""The gradient kernel on the matrix cores against the float64 oracle: chunk remainders, one to all workgroups, one chunk and
several a workgroup; and the two halves of a training step (summed gradient, weight update) against the oracle's own."""
import numpy as np
import pytest

from oracle import mlp_oracle as M
from tests.test_mlp import rand_problem

pytestmark = pytest.mark.gpu

# a parameter's gradient is a mean of products of three sums of at most 64 float32 terms each, and at most 64 samples are
# added one after another: (4 * 64 + 12) * 2^-24 of the largest, times 6 for the spread between parameters
TOL = 1e-4


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 63, 65, 1000, 4096, 16383, 16384, 16385, 40000])
def test_gradient_at_chunk_and_grid_edges(n):
    from canu_amd import oic
    w, z, t = (a.astype(np.float32) for a in rand_problem(n, n))
    loss, g = oic.Engine().model_grad(w, z, t, 0.3)
    ol, og = M.loss_grad(w.astype(np.float64), z.astype(np.float64), t.astype(np.float64), 0.3)
    assert abs(loss - ol) <= TOL * abs(ol)
    assert np.max(np.abs(g - og)) <= TOL * np.abs(og).max()


@pytest.mark.parametrize("n, batch", [(2, 1), (100, 33), (500, 100000)])
def test_training_loss_is_the_oracles_at_a_vanishing_rate(n, batch):
    """With a rate of 0 the weights stay as drawn, so the last epoch's loss is the oracle's at those weights."""
    from canu_amd import oic
    r = np.random.default_rng(n)
    x = (r.normal(0, 1, (n, M.NIN)) * 3 + 1).astype(np.float32)
    t = np.stack([r.normal(8, 2, n), r.normal(0, 1, n)], 1).astype(np.float32)
    eng = oic.Engine()
    loss = eng.train_model(x, t, epochs=3, batch=batch, lr=0.0)
    w, mu, sd = eng.model()
    ol = M.loss_only(w.astype(np.float64), (x.astype(np.float64) - mu) / sd, t.astype(np.float64), 0.05)
    assert abs(loss - ol) <= TOL * abs(ol)
