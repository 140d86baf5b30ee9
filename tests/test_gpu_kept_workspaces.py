"""Workspaces kept between calls: the location tables' scratch block and the
predictions' pinned slots."""
import threading

import numpy as np
import pytest

from test_gpu_location_table import build, closed_form

pytestmark = pytest.mark.gpu

# Growing, shrinking (a block over four times too large is replaced) and equal
# sizes, one to four passes, and more than the kept 512 MiB.
SEQUENCE = [(1000, 10), (300_000, 545), (300_000, 70_000), (5, 3), (0, 4), (200_000, (1 << 25) + 3), (200_000, 256),
            (60_000_000, 61_597), (777, 777)]


def test_tables_of_changing_sizes():
    for n, K in SEQUENCE:
        keys = np.random.default_rng(n + K).integers(0, K, n, dtype=np.uint32)
        print("case: n=%d K=%d" % (n, K), flush=True)
        people, offsets = build(keys, K)
        want_p, want_o = closed_form(keys, K)
        assert np.array_equal(offsets, want_o) and np.array_equal(people, want_p)


def test_tables_of_two_threads():
    cases = [(400_000, 61_597), (500_000, 545)]
    wrong = []

    def work(n, K):
        for i in range(8):
            keys = np.random.default_rng(i * K).integers(0, K, n, dtype=np.uint32)
            got, want = build(keys, K), closed_form(keys, K)
            if not all(np.array_equal(a, b) for a, b in zip(got, want)):
                wrong.append((n, K, i))

    threads = [threading.Thread(target=work, args=c) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("members,batch,rows", [(2, 4096, 5000), (3, 704, 705), (1, 2048, 2048), (2, 1024, 2049)])
def test_predictions_in_parts(members, batch, rows):
    """Parts of one member's rows (more than 2,048 in a chunk) or of all
    members; a row's result does not depend on the batch it is in."""
    from pandemicthrust_amd.surrogate import Surrogate
    X = np.random.default_rng(3).uniform(0, 1, (rows, 16)).astype(np.float32)
    out = []
    for b in (batch, 64):
        s = Surrogate(members=members, batch=b, seed=9)
        out.append([s.predict(X[:5]), s.predict(X), s.predict(X[:70])])
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
