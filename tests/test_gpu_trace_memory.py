"""A trace that fits only without the counted tables' buffers: enabling it
succeeds, as before there were any, and the simulation goes on with sorted
tables.  2.35M agents over 200 times the locations: 245 MB of trace arrays, 80
MB and more of counted tables.  All but 200 MB of the device's free memory is
taken by the test (no kernel runs while all of it is)."""
import ctypes as C
import time

import numpy as np
import pytest

from hip_mem import DeviceArray, hip

pytestmark = pytest.mark.gpu

ROW = ["6", "2.4", "1.9", "3000", "3000", "1.0", "200.0", "0.8", "0.3"]
LEAVE = 204 << 20


def test_trace_when_memory_is_short():
    from pandemicthrust_amd import Params, PandemicSim
    from pandemicthrust_amd.api import lib
    want = PandemicSim(Params.from_row(ROW), 7)
    want.setup_sim()
    counts, inf = want.run()
    state = [want.array(w) for w in range(6)]
    want.close()
    s = PandemicSim(Params.from_row(ROW), 7)
    s.setup_sim()
    first = s.step()
    assert lib().pt_location_table_release(0) == 0      # (else it is given up first)
    gap = DeviceArray(LEAVE, np.uint8)
    hog = []
    try:
        quiet = 0
        while quiet < 5:        # what was freed before comes back bit by bit
            had, size = len(hog), 16 << 30
            while size >= 4 << 20:
                p = C.c_void_p()
                if hip().hipMalloc(C.byref(p), size) == 0:
                    hog.append(p)
                else:
                    size //= 2
            hip().hipGetLastError()
            quiet = quiet + 1 if len(hog) == had else 0
            time.sleep(0.1)
        gap.free()
        time.sleep(0.5)
        s.enable_trace(True)
    finally:
        for p in hog:
            hip().hipFree(p)
    rows = [first] + [s.step() for _ in range(3)]
    s.enable_trace(False)
    rows += [s.step() for _ in range(2)]
    for d, (_, c, i) in enumerate(rows):
        assert np.array_equal(c, counts[d]) and i == inf[d], d
    for w in range(6):
        assert np.array_equal(s.array(w), state[w])
    # a counted weekday logs two pairs per agent, a sorted one without the
    # children's second: day 4, not traced, is sorted
    pairs = s.table_log()[1]
    assert pairs[0] == 2 * s.n_people and pairs[4] < 2 * s.n_people, pairs
    s.close()
