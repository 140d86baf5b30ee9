"""MLP kernels at the edges of their tiles, against the CPU oracle.

Batches of one and of three 64-row tiles (the output layer's column sums go by
chunks of 128 rows: half a chunk, one and a half); predictions of 1 to 129
rows, below, at and past the tiles.  Tolerances as for the same comparison at
one size: weights, activations and output gradients round to BF16 at the same
points, so relative Frobenius errors stay within 2e-2 (gradients) and 1e-2
(predictions), the loss within 1e-3.
"""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as M  # noqa: E402

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _data(n, seed):
    rng = np.random.default_rng(seed)
    X = rng.uniform(0, 1, (n, 16)).astype(np.float32)
    return X, np.sin(X @ rng.normal(0, 1.0, (16, 720))).astype(np.float32)


@pytest.mark.parametrize("members,batch", [(1, 64), (3, 192), (2, 320)])
def test_gradients(members, batch):
    from pandemicthrust_amd.surrogate import Surrogate
    s = Surrogate(members=members, batch=batch, seed=2)
    X, Y = _data(400, 5)
    s.set_data(X, Y)
    rows = np.random.default_rng(1).permutation(400)[:batch]
    g, loss = s.gradients(rows)
    P = s.params()
    lay, _ = M.layout()
    for k in range(members):
        want_loss, want = M.loss_and_grads(P[k].astype(np.float64), X[rows], Y[rows], bf16_mode=True)
        assert abs(loss[k] - want_loss) <= 1e-3 * want_loss
        for l, (w, b) in enumerate(lay):
            for sl in (slice(w, b), slice(b, b + M.DIMS[l + 1])):
                assert _rel(g[k, sl], want[sl]) <= 2e-2, (k, l, sl)
    s.close()


@pytest.mark.parametrize("rows", [1, 15, 31, 33, 63, 64, 65, 129])
def test_predictions(rows):
    from pandemicthrust_amd.surrogate import Surrogate
    s = Surrogate(members=2, batch=64, seed=5)
    X, _ = _data(rows, 1)
    P = s.params()
    out = s.predict(X)
    for k in range(2):
        want, _, _ = M.forward(P[k].astype(np.float64), X, bf16_mode=True)
        assert _rel(out[k], want) <= 1e-2
    s.close()
