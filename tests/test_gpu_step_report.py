"""Days stepped one by one, in turn with every call that changes the loop's
state on the device, against one run of all days."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROW = ["12", "2.4", "1.9", "300", "300", "0.05", "0.05", "0.8", "0.3"]


def _sim(setup=True):
    from pandemicthrust_amd import Params, PandemicSim
    s = PandemicSim(Params.from_row(ROW), 5)
    if setup:
        s.setup_sim()
    return s


def _steps(s, n):
    return [s.step()[1:] for _ in range(n)]


def test_steps_between_runs_restores_and_checkpoints():
    s = _sim()
    s.snapshot()
    counts, inf = s.run()
    assert s.step()[0] == 1                     # the loop has ended

    def check(rows, first):
        for k, (c, i) in enumerate(rows):
            assert np.array_equal(c, counts[first + k]) and i == inf[first + k]

    s.restore()
    check(_steps(s, 3), 0)
    s.restore()                                 # the report of day 2 no longer holds
    check(_steps(s, 5), 0)
    saved = s.save_checkpoint()
    check(_steps(s, 2), 5)
    s.load_checkpoint(saved)                    # back to day 5
    check(_steps(s, 1), 5)
    rest, rest_inf = s.run()
    assert np.array_equal(rest, counts[6:]) and np.array_equal(rest_inf, inf[6:])
    assert s.step()[0] == 1
    s.load_checkpoint(saved)
    check(_steps(s, 7), 5)
    assert s.step()[0] == 1
    s.close()
