"""Captured chunks of one-workgroup steps, replayed, and then the launches the batch takes when its
mix or its launch shape changes: bit-equal to the same steps without graphs."""
import numpy as np
import pytest

import sllg
from sllg import batch as SB
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _start(n, seed):
    s = np.random.default_rng(seed).standard_normal((3, n))
    return s / np.linalg.norm(s, axis=0)


def _small():
    return [(W.sc_ferro(dims=(9, 10, 11), precision="fp32", seed=1)[0], 300.0),
            (W.sc_ferro(dims=(5, 6, 7), precision="fp32", seed=2)[0], 0.0),
            (W.fcc_3shell(dims=(3, 4, 5))[0], 200.0)]


def _tune_gather_copy(b):
    """Leave the batch with the gather copy in force and one-workgroup steps allowed: tuned beside
    a member of 42 entries a row and 100,000 spins, which gathers faster from the copy, then alone."""
    big = W.fcc_3shell(dims=(29, 29, 30), seed=5)[0]
    k = b.add(big, _start(big.n, 9), T=100.0)
    t = b.autotune(10)
    b.remove(k)
    return t["gather_copy"]


def _run(change, flags, tuned):
    b = SB.Batch(flags=flags)
    ids = [b.add(s, _start(s.n, k), T=T, B=(0.0, 0.1, 0.0)) for k, (s, T) in enumerate(_small())]
    if tuned:
        print("gather copy", _tune_gather_copy(b))
    for _ in range(3):
        b.step(10)
    mid = [b.get_spins(k) for k in ids]
    if change == "larger member":
        s = W.sc_ferro(dims=(15, 16, 17), precision="fp32", seed=4)[0]
        ids.append(b.add(s, _start(s.n, 7), T=50.0))
    elif change == "launch shape":
        b.set_launch(256, gather_copy=1)
    elif change == "persistent":
        b.set_persistent(True)
    for _ in range(2):
        b.step(10)
    out = mid + [b.get_spins(k) for k in ids]
    b.close()
    return out


@pytest.mark.parametrize("change", ["larger member", "launch shape", "persistent"])
def test_replayed_small_chunks_then_launches(gpu, change):
    want = _run(change, 0, False)
    got = _run(change, SB.BATCH_GRAPH, True)
    for a, c in zip(got, want):
        assert np.array_equal(a, c)
