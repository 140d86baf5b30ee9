"""The loop's last day, on which nobody is infected any more, in every form of
a counted day: launches in pairs, split layouts, the plan inside the
compaction with one sweep block per thread and with several, a plan launch of
its own, and the replicate batch.  Its row (all sixteen counters), the day
counters and the table log must be those of the sorted tables."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # people, locations
    (0.02, 0.02),       # launches in pairs
    (0.05, 3.1),        # weekends split
    (0.05, 13.85),      # weekdays split too
    (2.2, 1.0),         # 5.2M agents: single launches
    (3.7, 1.0),         # 8.7M: each counter summed by a block of its own
    (12.0, 12.0),       # 28M, the same with split layouts
    (29.0, 1.0),        # 68M: a plan launch of its own
]


def _result(sim, rows):
    log = sim.table_log()
    return [rows[0], rows[1], sim.scalars()[3:], log[0].shape, *[sim.array(w) for w in range(6)]]


@pytest.mark.parametrize("people,locations", CASES)
def test_dies_out(people, locations):
    """No transmission: the seeded agents recover after ten days."""
    from pandemicthrust_amd import Params, PandemicSim
    row = ["20", "0", "0", "7", "5", str(people), str(locations), "1", "0"]
    res = []
    for mode in (0, 1):
        s = PandemicSim(Params.from_row(row), 29)
        s.set_table_mode(mode)
        s.setup_sim()
        s.snapshot()
        res.append(_result(s, s.run()))
        s.restore()
        steps = []
        for _ in range(20):
            ended, c, i = s.step()
            steps.append((c, i))
            if ended:
                break
        assert s.step()[0] == 1
        res.append(_result(s, (np.stack([c for c, _ in steps]), np.array([i for _, i in steps], np.int32))))
        s.close()
    assert len(res[0][1]) == 11 and res[0][1][-1] == 0
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert np.array_equal(a, b)


def test_batch_dies_out():
    """Replicates that end on different days, and one that starts without
    infected."""
    from pandemicthrust_amd import PandemicBatch, PandemicSim, Params
    rows = [["20", "0", "0", "7", "5", "0.05", "0.05", "1", "0"], ["6", "0", "0", "3", "0", "0.3", "0.3", "1", "0"],
            ["20", "1.8", "1.3", "0", "0", "0.01", "0.01", "1", "0"], ["20", "0.2", "0.1", "40", "40", "0.1", "0.1", "1", "0"]]
    params, seeds = [Params.from_row(r) for r in rows], [3, 4, 5, 6]
    b = PandemicBatch(params, seeds)
    b.setup()
    b.snapshot()
    first = b.run()
    b.restore()
    again = b.run()
    for r in range(len(rows)):
        s = PandemicSim(params[r], seeds[r])
        s.set_table_mode(1)
        s.setup_sim()
        counts, inf = s.run()
        for got in (first[r], again[r]):
            assert np.array_equal(got[0], counts) and np.array_equal(got[1], inf), r
        for w in range(6):
            assert np.array_equal(b.array(r, w), s.array(w)), (r, w)
        s.close()
    b.close()
