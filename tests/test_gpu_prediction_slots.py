"""Predictions of one part (one pinned slot, no event) and of several in turn
on one handle: slots grow and the second appears between calls.  A row's
result depends neither on the batch nor on the calls before it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members,batch", [(1, 64), (2, 64), (5, 1024), (1, 4096)])
def test_one_part_and_several_in_turn(members, batch):
    from pandemicthrust_amd.surrogate import Surrogate
    X = np.random.default_rng(8).uniform(0, 1, (5000, 16)).astype(np.float32)
    ref = Surrogate(members=members, batch=64, seed=4)
    want = ref.predict(X)
    ref.close()
    # one row; a full chunk; two chunks; the widest single part, and one row
    # more; more rows than a slot holds
    sizes = [1, min(batch, 400), batch + 1, min(batch, 2048 // members), min(batch, 2048 // members) + 1, 3, 5000, 1]
    for order in (sizes, sizes[::-1]):
        s = Surrogate(members=members, batch=batch, seed=4)
        for n in order:
            assert np.array_equal(s.predict(X[:n]), want[:, :n]), n
        s.close()
