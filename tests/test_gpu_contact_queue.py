"""Two-phase contacts (filtered_contacts): infectors that pass the draw test
are queued per block and run 256 at a time.  Infected counts around one and
two tiles, and a run whose blocks take several tiles each (one block per CU,
over 65,536 infected), every day bit-exact against the oracle."""
import numpy as np
import pytest

import oracle_ctypes as O

pytestmark = pytest.mark.gpu


def _days(row, seed, days, blocks_per_cu=None):
    from pandemicthrust_amd import Params, PandemicSim
    gpu = PandemicSim(Params.from_row(row), seed)
    ref = O.OracleSim(O.params_from_row(row), seed)
    if blocks_per_cu:
        gpu.set_launch("contact_blocks_per_cu", blocks_per_cu)
    gpu.setup_sim()
    ref.setup()
    most = 0
    for day in range(days):
        rg, cg, ig = gpu.step()
        rr, cr, ir = ref.step()
        assert (rg, ig) == (rr, ir) and np.array_equal(cg, cr), day
        for which in range(6):
            assert np.array_equal(gpu.array(which), ref.array(which)), (day, which)
        most = max(most, ig)
    return most


@pytest.mark.parametrize("pandemic,seasonal", [(1, 0), (255, 0), (200, 56), (257, 0), (256, 256), (400, 113)])
def test_infected_counts_around_a_tile(pandemic, seasonal):
    row = ["8", "2.5", "1.8", str(pandemic), str(seasonal), "0.02", "0.02", "0.8", "0.4"]
    _days(row, 3 + pandemic, 7)


def test_blocks_with_several_tiles():
    row = ["25", "3.5", "2.5", "2000", "2000", "0.2", "0.2", "1", "0"]
    assert _days(row, 5, 22, blocks_per_cu=1) > 65536
