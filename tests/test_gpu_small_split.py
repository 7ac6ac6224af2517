"""Runs of one-workgroup steps longer than one launch holds: every launch starts at its own step, so
the trajectory (and the noise it draws) is that of the two launches a step."""
import numpy as np
import pytest

import sllg
from sllg import batch as SB
from sllg import workloads as W

pytestmark = pytest.mark.gpu

SHAPE = (256, 1, 2, 1, 0, 0)  # two launches a step, packed entries
LONG = 4100  # several launches, the last one short


def _start(n, seed):
    s = np.random.default_rng(seed).standard_normal((3, n))
    return s / np.linalg.norm(s, axis=0)


def _systems():
    return [W.sc_ferro(dims=(3, 4, 5), precision="fp32", seed=6)[0], W.fcc_3shell(dims=(1, 2, 3), seed=7)[0]]


@pytest.mark.parametrize("nsteps", [1023, 1024, 1025, LONG])
def test_handle_runs_longer_than_a_launch(gpu, nsteps):
    s = _systems()[0]
    out = []
    for launch in (None, SHAPE):
        with sllg.Context(s) as g:
            if launch:
                g.set_launch(*launch)
            g.set_spins(_start(s.n, 1))
            g.set_temperature(200.0)
            g.step(5, nsteps)
            out.append((g.get_spins(), g.det_field()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("flags", [0, SB.BATCH_GRAPH])
def test_batch_chunks_longer_than_a_launch(gpu, flags):
    out = []
    for small in (True, False):
        b = SB.Batch(flags=flags)
        if not small:
            b.set_launch(256)
        ids = [b.add(s, _start(s.n, k), T=150.0, t0=3) for k, s in enumerate(_systems())]
        b.step(LONG)
        b.step(LONG)
        assert all(b.get_step(k) == 3 + 2 * LONG for k in ids)
        out.append([b.get_spins(k) for k in ids])
        b.close()
    for a, c in zip(*out):
        assert np.array_equal(a, c)
