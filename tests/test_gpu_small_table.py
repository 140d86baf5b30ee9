"""One-launch location tables (at most 131,072 pairs and 8,000 buckets) at the
edges of their blocks and limits, against the closed form; beyond the limits
the radix build gives the same table."""
import numpy as np
import pytest

from test_gpu_location_table import build, closed_form

pytestmark = pytest.mark.gpu

CASES = [(1, 1), (63, 2), (1023, 8000), (1024, 1), (1025, 1024), (8193, 1025), (29919, 545), (65536, 7999),
         (131071, 3), (131072, 8000), (131073, 8000), (131072, 8001)]


@pytest.mark.parametrize("n,K", CASES)
@pytest.mark.parametrize("entry", ["pt_location_table", "pt_location_table_noalloc"])
def test_small_tables(n, K, entry):
    rng = np.random.default_rng(n * 31 + K)
    keys = rng.integers(0, K, n, dtype=np.uint32)
    keys[: n // 5] = K - 1                 # a crowded last bucket, and runs of one key
    keys[n // 2: n // 2 + n // 7] = 0
    print("case: %s n=%d K=%d" % (entry, n, K), flush=True)
    people, offsets = build(keys, K, entry)
    want_p, want_o = closed_form(keys, K)
    assert np.array_equal(offsets, want_o)
    assert np.array_equal(people, want_p)
