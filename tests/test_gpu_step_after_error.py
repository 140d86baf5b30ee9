"""A step that reports another call's error has run its day all the same; the
next step goes on with the day after it (here from a weekday to a weekend)."""
import ctypes as C

import numpy as np
import pytest

from hip_mem import hip

pytestmark = pytest.mark.gpu

ROW = ["9", "2.4", "1.9", "300", "300", "0.05", "0.05", "0.8", "0.3"]


def test_step_after_a_failed_one():
    from pandemicthrust_amd import Params, PandemicSim, PTError
    want = PandemicSim(Params.from_row(ROW), 5)
    want.setup_sim()
    counts, inf = want.run()
    s = PandemicSim(Params.from_row(ROW), 5)
    s.setup_sim()
    for day in range(4):
        assert np.array_equal(s.step()[1], counts[day])
    p = C.c_void_p()
    assert hip().hipMalloc(C.byref(p), 1 << 50) != 0      # leaves its error for the next check
    try:
        s.step()                                          # day 4
    except PTError:
        pass
    for day in range(5, 9):
        _, c, i = s.step()
        assert np.array_equal(c, counts[day]) and i == inf[day], day
    for w in range(6):
        assert np.array_equal(s.array(w), want.array(w)), w
    s.close()
    want.close()
