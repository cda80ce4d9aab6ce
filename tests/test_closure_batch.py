"""The closure trainer's batch kernel (groups of 32 samples, at most 256
workgroups) and its device-drawn minibatches."""
import numpy as np
import pytest

import myfvcomcode_amd as F
from oracle import mlp

pytestmark = pytest.mark.gpu

A, C, MASK = 6364136223846793005, 1442695040888963407, (1 << 64) - 1


def _case(n, bmax):
    rng = np.random.default_rng(n)
    x = np.zeros((n, 8), np.float32)
    x[:, :5] = rng.normal(0, 1, (n, 5))
    x[:, 5] = 1.0
    y = np.exp(rng.uniform(np.log(1e-5), np.log(1e-1), (n, 2))).astype(np.float32)
    t = F.Trainer(x, y, bmax=bmax)
    p = rng.normal(0, 0.3, mlp.NPARAM).astype(np.float32)
    t.set_params(p)
    return x, y, t, p


# one sample; the edges of a group; a remainder after the 256 workgroups'
# first groups (8192 samples), so that some of them take two
@pytest.mark.parametrize("batch", [1, 31, 32, 33, 8225])
def test_gradient_at_group_edges(built, batch):
    x, y, t, p = _case(9000, 8225)
    print("case: MLP gradient, batch %d" % batch, flush=True)
    idx = np.random.default_rng(batch).integers(0, 9000, batch).astype(np.int32)
    loss, g = t.grad(idx)
    lr, gr = mlp.loss_grad(p.astype(np.float64), x[idx], y[idx])
    # FP32 rounding of 64-term products, the residual's logarithms (their
    # absolute error over residuals of order 1) and the batch sum: about 1e-6
    assert abs(loss - lr) <= 1e-5 * abs(lr)
    assert np.linalg.norm(g - gr) <= 1e-5 * np.linalg.norm(gr)
    first = t.grad(batch=batch)
    ident = t.grad(np.arange(batch, dtype=np.int32))
    assert first[0] == ident[0] and np.array_equal(first[1], ident[1])


# ntrain: one sample, a power of two, and the whole set
@pytest.mark.parametrize("batch,ntrain,seed", [(1, 1, 0), (33, 4096, 5), (200, 9000, (1 << 63) + 12345)])
def test_drawn_minibatch_is_the_seeded_one(built, batch, ntrain, seed):
    x, y, t, p = _case(9000, 512)
    print("case: MLP drawn minibatch %d of %d" % (batch, ntrain), flush=True)
    st = (seed * A + C) & MASK
    drawn = []
    for _ in range(3):
        idx = np.empty(batch, np.int32)
        for b in range(batch):
            st = (st * A + C) & MASK
            idx[b] = (st >> 33) % ntrain
        drawn.append(idx)
    # with lr = 0 the weights stay: the last step's loss is that of its batch
    for steps in (1, 3):
        t.set_params(p)
        assert t.train(steps, batch=batch, ntrain=ntrain, lr=0.0, wd=0.0, seed=seed) == t.grad(drawn[steps - 1])[0]
    assert np.array_equal(t.params(), p)
