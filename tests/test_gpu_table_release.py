"""The scratch block that location tables keep: freed on request, and a call
after that works as the first one did."""
import time

import numpy as np
import pytest

from test_gpu_location_table import build, closed_form

pytestmark = pytest.mark.gpu


def test_kept_block_is_released():
    from pandemicthrust_amd.api import device_memory, lib
    L = lib()
    keys = np.random.default_rng(2).integers(0, 61_597, 20_000_000, dtype=np.uint32)
    people, offsets = build(keys, 61_597)       # keeps 190 MB and more
    held = device_memory()[0]
    assert L.pt_location_table_release(0) == 0
    for _ in range(100):                        # (freed memory is cleared before it counts as free)
        if device_memory()[0] - held >= 150 << 20:
            break
        time.sleep(0.02)
    assert device_memory()[0] - held >= 150 << 20
    assert L.pt_location_table_release(0) == 0  # nothing kept: no error
    again = build(keys, 61_597)
    want = closed_form(keys, 61_597)
    assert all(np.array_equal(a, w) and np.array_equal(b, w) for a, b, w in zip((people, offsets), again, want))
    assert L.pt_location_table_release(0) == 0
    assert L.pt_location_table_release(-1) != 0
