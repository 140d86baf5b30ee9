"""Counted errand tables (csrc/pt_count.h) against the sorted tables: the
automatic mode counts every bucket and picks single people, mode 1 sorts the
whole table.  Both must give the same days, state and generation tallies.

Sizes: populations below one chunk and at odd remainders; so few buckets that
a bucket's list in a chunk exceeds 64 ids (bisected instead of ranked); many
nearly empty buckets (empty chunks of a bucket); bucket counts on both sides
of the largest layout counted in one block (40,000: weekday 2,901 per
location scale, weekend 13,000), of the 65,535 locations per hour up to which
split weekday keys take 2 bytes, and of the 8 groups per hour up to which
layouts are split at all."""
import numpy as np
import pytest

import oracle_ctypes as O

pytestmark = pytest.mark.gpu

CASES = [
    # people, locations, days, seeds per strain
    (0.0004, 0.0004, 14, 20),
    (0.004, 0.0011, 9, 60),        # about 30 buckets for 9,400 agents
    (0.1, 0.0011, 9, 3000),        # the same for 235,000: lists of hundreds of ids
    (0.02, 0.3, 9, 300),
    (0.05, 3.05, 9, 2000),         # weekend 39,650 buckets: not split
    (0.05, 3.1, 9, 2000),          # weekend 40,300: split by hour
    (0.05, 13.75, 6, 2000),        # weekday 39,889
    (0.05, 13.85, 6, 2000),        # weekday 40,179: split
    (0.6, 21.24, 7, 20000),        # 1.4M agents: several chunks, one group per hour
    (0.0004, 25.1, 7, 20),         # 943 agents; weekday hour 0 in two groups (40,160 locations)
    (0.1, 40.9, 7, 5000),          # 65,440 locations in weekday hour 0
    (0.1, 41.0, 7, 5000),          # 65,600
    (0.3, 200.0, 7, 5000),         # 320,000: 8 groups
    (0.05, 200.5, 7, 5000),        # 320,800: weekday sorted
    (0.05, 2.98, 9, 2000),         # weekend 38,740 buckets: the largest counted beside the sweep
    (0.28, 0.28, 9, 3000),         # 658,000 agents: chunks of 3,072, picks found in the keys
    (0.4, 0.1, 9, 3000),           # 940,000, odd chunk and agent counts
    (0.45, 0.45, 9, 3000),         # 1.06M: chunks above 4,096, picks from lists
    (1.0, 1.0, 7, 20000),          # 2.35M agents: launches in pairs
    (2.2, 1.0, 7, 20000),          # 5.2M: single launches, the compaction plans the day
    (3.7, 1.0, 7, 20000),          # 8.7M: several sweep blocks per thread of the plan
    (29.0, 1.0, 4, 20000),         # 68M: a plan launch of its own
]


@pytest.mark.parametrize("people,locations,days,seeds", CASES)
def test_counted_equals_sorted(people, locations, days, seeds):
    from pandemicthrust_amd import Params, PandemicSim
    row = [str(days), "2.6", "1.9", str(seeds), str(seeds), str(people), str(locations), "0.8", "0.3"]
    runs = []
    for mode in (0, 1):
        s = PandemicSim(Params.from_row(row), 17)
        s.set_table_mode(mode)
        s.setup_sim()
        counts, inf = s.run()
        runs.append([counts, inf, *s.generation_offsets(), *[s.array(w) for w in range(6)]])
        s.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("people,locations", [(0.0007, 0.0007), (0.06, 0.0011), (0.05, 0.6)])
def test_counted_days_equal_the_oracle(people, locations):
    """Every day's counts and state; after a counted day the table hooks
    return that day's whole table."""
    from pandemicthrust_amd import Params, PandemicSim
    from pandemicthrust_amd.api import PT_ERRAND_OFFSETS, PT_ERRAND_PEOPLE
    row = ["9", "2.4", "1.7", "40", "40", str(people), str(locations), "0.9", "0.2"]
    gpu = PandemicSim(Params.from_row(row), 23)
    ref = O.OracleSim(O.params_from_row(row), 23)
    gpu.setup_sim()
    ref.setup()
    for day in range(9):
        rg, cg, ig = gpu.step()
        rr, cr, ir = ref.step()
        assert (rg, ig) == (rr, ir) and np.array_equal(cg, cr), day
        for w in range(6):
            assert np.array_equal(gpu.array(w), ref.array(w)), (day, w)
        if rr == 1:
            break
        if day in (1, 5):
            assert np.array_equal(gpu.array(PT_ERRAND_OFFSETS), ref.array(O.OR_ERRAND_OFFSETS)), day
            assert np.array_equal(gpu.array(PT_ERRAND_PEOPLE), ref.array(O.OR_ERRAND_PEOPLE)), day


def test_batch_counts_equal_sorts():
    """A batch of unlike replicates (sizes, location scales, lengths; one
    without infected, one that dies out early): counted days equal sorted
    ones, and equal each replicate's single run."""
    from pandemicthrust_amd import PandemicBatch, PandemicSim, Params
    rows = [["16", "2.2", "1.4", "30", "30", "0.05", "0.05", "1", "0"],
            ["9", "1.8", "1.3", "5", "0", "0.0004", "0.0004", "1", "0"],
            ["20", "2.6", "1.9", "200", "100", "0.02", "0.2", "0.8", "0.3"],
            ["12", "0", "0", "4", "4", "0.003", "0.003", "1", "0"],
            ["20", "1.8", "1.3", "0", "0", "0.004", "0.004", "1", "0"],
            ["14", "2.4", "1.7", "900", "400", "0.09", "0.0011", "1", "0"]]
    params, seeds = [Params.from_row(r) for r in rows], [11, 12, 13, 14, 15, 16]
    res = []
    for mode in (0, 1):
        b = PandemicBatch(params, seeds)
        b.set_table_mode(mode)
        b.setup()
        b.snapshot()
        first = b.run()
        b.restore()
        again = b.run()         # replayed graphs, from the same state
        for x, y in zip(first, again):
            assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])
        res.append((first, [[b.array(r, w) for w in range(6)] for r in range(len(rows))]))
        b.close()
    for r in range(len(rows)):
        for k in range(2):
            assert np.array_equal(res[0][0][r][k], res[1][0][r][k]), r
        for w in range(6):
            assert np.array_equal(res[0][1][r][w], res[1][1][r][w]), (r, w)
        s = PandemicSim(params[r], seeds[r])
        s.setup_sim()
        counts, inf = s.run()
        s.close()
        assert np.array_equal(res[0][0][r][0], counts) and np.array_equal(res[0][0][r][1], inf), r
