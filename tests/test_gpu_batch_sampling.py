"""<M> of many batch members in one pair of launches against the single-handle reduction (same
blocks and order of sums: the same bits), and kept sample buffers against fresh ones."""
import numpy as np
import pytest

import helpers
import sllg
from sllg import batch as SB
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _start(n, seed):
    s = np.random.default_rng(seed).standard_normal((3, n))
    return s / np.linalg.norm(s, axis=0)


def _free(n):
    return sllg.System(n=n, species=[dict(mu=2.0, lambda_=0.3)], precision="fp32", seed=5)


# one spin, one block and one spin more, more spins than the grid's 512 blocks hold at once; two
# species on two sublattices
SYSTEMS = [lambda: _free(1), lambda: _free(256), lambda: _free(257), lambda: _free(512 * 256 + 3),
           lambda: helpers.tensor_csr_system(L=6, precision="fp32")[0], lambda: W.sc_ferro(L=10, precision="fp32")[0]]


@pytest.mark.parametrize("gather_copy", [0, 1])
def test_batch_reduce_equals_handle(gpu, gather_copy):
    systems = [f() for f in SYSTEMS]
    starts = [_start(s.n, 7 + k) for k, s in enumerate(systems)]
    nsub = []
    want = []
    for s, s0 in zip(systems, starts):
        with sllg.Context(s) as g:
            g.set_spins(s0)
            want.append(g.reduce(energy=False)[0].ravel())
            nsub.append(len(want[-1]) // 3)
    assert max(nsub) > 1
    stride = 3 * max(nsub)
    b = SB.Batch()
    ids = [b.add(s, s0) for s, s0 in zip(systems, starts)]
    order = [3, 0, 5, 4, 1, 2, 3]  # any order, a member twice, then fewer members
    for _ in range(2):
        for pick in (order, order[:2], order):
            got = np.asarray(b.reduce([ids[k] for k in pick], stride=stride)).reshape(len(pick), stride)
            for row, k in zip(got, pick):
                assert np.array_equal(row[:3 * nsub[k]], want[k])
    b.set_launch(256, 1, 1, gather_copy)
    b.step(3)
    after = [_handle_mag(s, b.get_spins(i)) for s, i in zip(systems, ids)]
    got = np.asarray(b.reduce(ids, stride=stride)).reshape(len(ids), stride)
    for row, k in zip(got, range(len(ids))):
        assert np.array_equal(row[:3 * nsub[k]], after[k])


def _handle_mag(s, spins):
    with sllg.Context(s) as g:
        g.set_spins(spins)
        return g.reduce(energy=False)[0].ravel()


@pytest.mark.parametrize("steps", [1, 1365, 1366])  # the longest series of the kept buffer and one more
def test_long_series(gpu, steps):
    s = W.sc_ferro(L=4, precision="fp32")[0]
    with sllg.Context(s) as g, sllg.Context(s) as h:
        for c in (g, h):
            c.set_spins(_start(s.n, 2))
            c.set_temperature(50.0)
        m = g.run_sampled(0, steps, 1)
        for t in range(0, steps, 100):  # the same steps in short series
            k = min(100, steps - t)
            assert np.array_equal(m[t:t + k], h.run_sampled(t, k, 1))
