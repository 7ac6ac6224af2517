"""What the batch's autotuner reports where every member takes one-workgroup steps."""
import time

import numpy as np
import pytest

from sllg import batch as SB
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _step_ms(b, ids, n=400):
    b.step(n)
    b.reduce(ids)
    best = 1e9
    for _ in range(3):
        t = time.perf_counter()
        b.step(n)
        b.reduce(ids)
        best = min(best, time.perf_counter() - t)
    return best / n * 1e3


@pytest.mark.parametrize("flags", [0, SB.BATCH_GRAPH])
def test_times_of_one_workgroup_steps(gpu, flags):
    """Eight members of 1,000 spins: two launches a step take some four times as long."""
    b = SB.Batch(flags=flags)
    ids = []
    for k in range(8):
        s = W.sc_ferro(dims=(10, 10, 10), precision="fp32", seed=k + 1)[0]
        ids.append(b.add(s, np.repeat([[0.0], [0.0], [1.0]], s.n, axis=1), T=100.0))
    r = b.autotune(50)
    small = _step_ms(b, ids)
    b.set_launch(256)
    launches = _step_ms(b, ids)
    assert small < 0.6 * launches
    assert 0 < r["ms_per_step"] < 0.6 * launches and 0 < r["ms_per_step_default"] < 0.6 * launches
    b.close()
