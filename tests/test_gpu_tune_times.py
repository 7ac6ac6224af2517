"""What the autotuner reports: the time of a step as a new handle takes it, and as the tuned one does."""
import time

import pytest

import sllg
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _step_ms(g, n=400):
    g.step(0, 20)
    g.sync()
    best = 1e9
    for _ in range(3):
        t = time.perf_counter()
        g.step(0, n)
        g.sync()
        best = min(best, time.perf_counter() - t)
    return best / n * 1e3


def test_default_time_is_that_of_line_blocks(gpu):
    """480,000 spins, 42 entries: packed entries take half as long again as line blocks."""
    s = W.fcc_3shell(dims=(100, 100, 12))[0]
    with sllg.Context(s) as g:
        g.set_temperature(100.0)
        r = g.autotune(20)
        assert r["line_mode"] == 2
        assert 0 < r["ms_per_step_default"] < 1.25 * r["ms_per_step"]


def test_times_of_one_workgroup_steps(gpu):
    """1,000 spins: two launches a step take four times as long as one-workgroup steps."""
    s = W.sc_ferro(dims=(10, 10, 10), precision="fp32")[0]
    with sllg.Context(s) as g:
        g.set_temperature(100.0)
        r = g.autotune(50)
        assert r["candidates"] > 1
        small = _step_ms(g)
        g.set_launch(256)
        launches = _step_ms(g)
        assert small < 0.6 * launches
        assert r["ms_per_step"] < 0.6 * launches and r["ms_per_step_default"] < 0.6 * launches
