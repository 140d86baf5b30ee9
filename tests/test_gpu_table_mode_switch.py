"""Counted days keep their matrices, keys and lists in buffers of the sorted
tables: days of all table modes in turn on one handle, with the table hooks and
a traced day between, equal the same days in one mode."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # people, locations
    (0.05, 0.05),    # matrices in the digit counts
    (3.0, 3.0),      # in the sorted keys
    (0.1, 13.0),     # of their own
    (0.05, 40.0),
]


@pytest.mark.parametrize("people,locations", CASES)
def test_modes_in_turn(people, locations):
    from pandemicthrust_amd import Params, PandemicSim
    from pandemicthrust_amd.api import PT_ERRAND_OFFSETS, PT_ERRAND_PEOPLE
    row = ["16", "2.5", "1.9", "600", "600", str(people), str(locations), "0.8", "0.3"]
    want = PandemicSim(Params.from_row(row), 41)
    want.set_table_mode(1)
    want.setup_sim()
    got = PandemicSim(Params.from_row(row), 41)
    got.setup_sim()
    for day in range(16):
        got.set_table_mode((0, 1, 0, 2, 0)[day % 5])
        if day in (3, 8):
            got.enable_trace(True)
        rw, cw, iw = want.step()
        rg, cg, ig = got.step()
        assert (rw, iw) == (rg, ig) and np.array_equal(cw, cg), day
        for w in range(6):
            assert np.array_equal(want.array(w), got.array(w)), (day, w)
        if day % 5 == 0:   # a counted day's table, made now
            for w in (PT_ERRAND_OFFSETS, PT_ERRAND_PEOPLE):
                assert np.array_equal(want.array(w), got.array(w)), (day, w)
        got.enable_trace(False)
    want.close()
    got.close()
