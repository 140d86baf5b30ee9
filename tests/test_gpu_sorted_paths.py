"""The sorted errand tables, where the automatic mode counts: contacts in two
phases (filtered_contacts), the launch settings of the sorts, and the automatic
choice between a full table and one of the queried buckets, on layouts that
are not counted (over a million agents in a few dozen buckets)."""
import numpy as np
import pytest

import oracle_ctypes as O

pytestmark = pytest.mark.gpu


def _days(row, seed, days, mode, blocks_per_cu=None):
    from pandemicthrust_amd import Params, PandemicSim
    gpu = PandemicSim(Params.from_row(row), seed)
    ref = O.OracleSim(O.params_from_row(row), seed)
    gpu.set_table_mode(mode)
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
    gpu.close()
    return most


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("pandemic,seasonal", [(1, 0), (255, 0), (200, 56), (257, 0), (256, 256), (400, 113)])
def test_infected_counts_around_a_tile(pandemic, seasonal, mode):
    row = ["8", "2.5", "1.8", str(pandemic), str(seasonal), "0.02", "0.02", "0.8", "0.4"]
    _days(row, 3 + pandemic, 7, mode)


@pytest.mark.parametrize("mode", [1, 2])
def test_blocks_with_several_tiles(mode):
    row = ["25", "3.5", "2.5", "2000", "2000", "0.2", "0.2", "1", "0"]
    assert _days(row, 5, 22, mode, blocks_per_cu=1) > 65536


SETTINGS = [{"contact_blocks_per_cu": 1, "gen_blocks_per_cu": 1, "sort_wide_bits": 9},
            {"contact_blocks_per_cu": 32, "gen_blocks_per_cu": 64, "sort_wide_bits": 1},
            {"contact_blocks_per_cu": 3, "gen_blocks_per_cu": 7, "sort_wide_bits": 6},
            {"mark_limit_pct": 0, "subset_share_pct": 0},          # never a subset table
            {"mark_limit_pct": 1000, "subset_share_pct": 100},     # a subset table on nearly every day
            {"mark_limit_pct": 50, "subset_share_pct": 90},
            {"sort_max_bits": 4}, {"sort_max_bits": 11, "sort_wide_bits": 1}]

FEW_BUCKETS = ["14", "2.2", "1.6", "3", "2", "0.45", "0.0011", "1", "0"]    # 1.06M agents, 40 weekend buckets
MANY = ["30", "1.8", "1.3", "10", "10", "0.0425", "0.0425", "1", "0"]


def _run(row, settings, mode):
    from pandemicthrust_amd import Params, PandemicSim
    s = PandemicSim(Params.from_row(row), 3)
    for k, v in settings.items():
        s.set_launch(k, v)
    s.set_table_mode(mode)
    s.setup_sim()
    counts, inf = s.run()
    out = [counts, inf, *[s.array(k) for k in range(6)]]
    full = s.table_log()[0]
    s.close()
    return out, full


@pytest.mark.parametrize("row,mode", [(MANY, 1), (MANY, 2), (FEW_BUCKETS, 0)])
def test_settings_of_the_sorts_do_not_change_results(row, mode):
    want, _ = _run(row, {}, 1)
    kinds = []
    for settings in [{}] + SETTINGS:
        got, full = _run(row, settings, mode)
        for a, b in zip(got, want):
            assert np.array_equal(a, b), settings
        kinds.append((settings, int(full.sum()), len(full)))
    if row is FEW_BUCKETS:      # the choice is made, and the settings move it
        default, never, often = kinds[0][1:], kinds[4][1:], kinds[5][1:]
        assert 0 < default[0] < default[1], kinds
        assert never[0] == never[1] and often[0] <= default[0], kinds


@pytest.mark.parametrize("mode,rows", [
    (1, [MANY, ["25", "2.4", "1.2", "8", "12", "0.02", "0.025", "1", "0"]]),
    (2, [MANY, ["25", "2.4", "1.2", "8", "12", "0.02", "0.025", "1", "0"]]),
    (0, [FEW_BUCKETS, MANY, ["20", "1.7", "1.3", "20", "5", "0.05", "0.04", "0.9", "0.2"]]),
])
def test_batch_settings_of_the_sorts_do_not_change_results(mode, rows):
    """(One replicate that cannot be counted: the whole batch sorts.)"""
    from pandemicthrust_amd import PandemicBatch, PandemicSim, Params
    params, seeds = [Params.from_row(r) for r in rows], [3 + i for i in range(len(rows))]
    want = []
    for p, seed in zip(params, seeds):
        s = PandemicSim(p, seed)
        s.set_table_mode(1)
        s.setup_sim()
        want.append(s.run())
        s.close()
    b = PandemicBatch(params, seeds)
    b.set_table_mode(mode)
    b.setup()
    b.snapshot()
    for settings in [{}, {"contact_blocks_per_cu": 1, "sort_wide_bits": 9}, {"contact_blocks_per_cu": 32, "sort_wide_bits": 2},
                     {"mark_limit_pct": 1000, "subset_share_pct": 100}, {"mark_limit_pct": 0, "subset_share_pct": 0},
                     {"sort_max_bits": 4}, {"sort_max_bits": 11}, {"segmented_tables": 0}, {"sort_max_bits": 9}]:
        for k, v in settings.items():
            b.set_launch(k, v)
        b.restore()
        got = b.run()
        for r, (counts, inf) in enumerate(want):
            assert np.array_equal(got[r][0], counts) and np.array_equal(got[r][1], inf), (settings, r)
    b.close()
