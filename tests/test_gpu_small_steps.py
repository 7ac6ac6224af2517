"""One-workgroup Heun steps of small systems against the two launches a step that
llg_set_launch keeps: every row computes the same, so the bits are equal."""
import numpy as np
import pytest

import helpers
import sllg
from sllg import batch as SB
from sllg import workloads as W

pytestmark = pytest.mark.gpu

SHAPE = (256, 1, 2, 1, 0, 0)  # two launches a step, packed entries


def _start(n, seed):
    s = np.random.default_rng(seed).standard_normal((3, n))
    return s / np.linalg.norm(s, axis=0)


def _sc(dims, nc=1, **kw):
    return W.sc_ferro(dims=dims, precision="fp32", ncomp=nc, **kw)[0]


def _free(n):
    return sllg.System(n=n, species=[dict(mu=2.0, lambda_=0.3, k1u=2e-23)], precision="fp32", seed=5)


def _tensor():
    s = helpers.tensor_csr_system(L=6, precision="fp32")[0]  # two species, 18 entries a row
    return s


# one spin, part of a wave, a wave and one more, one row a thread and one more, the largest and one
# past it (which takes the launches); short rows with 1, 3 and 9 components; rows longer than the
# registers hold; no exchange; two species
SYSTEMS = {
    "sc1": lambda: _sc((1, 1, 1)), "sc63": lambda: _sc((3, 3, 7)), "sc65": lambda: _sc((1, 5, 13)),
    "sc1024": lambda: _sc((8, 8, 16)[::-1]), "sc1025": lambda: _sc((5, 5, 41)), "sc2048_nc3": lambda: _sc((16, 16, 8), 3),
    "sc2040_nc9": lambda: _sc((12, 17, 10), 9), "sc2057": lambda: _sc((11, 11, 17)), "free7": lambda: _free(7),
    "free2048": lambda: _free(2048), "fcc": lambda: W.fcc_3shell(dims=(5, 3, 7))[0],
    "fcc1024": lambda: W.fcc_3shell(dims=(4, 8, 8))[0], "tensor": _tensor,
}


@pytest.mark.parametrize("name", list(SYSTEMS))
@pytest.mark.parametrize("T", [0.0, 250.0])
def test_small_steps_equal_launches(gpu, name, T):
    s = SYSTEMS[name]()
    s0 = _start(s.n, 3)
    stag = 0.2 * _start(s.n, 4)
    out = []
    for launch in (None, SHAPE):
        with sllg.Context(s) as g:
            if launch:
                g.set_launch(*launch)
            g.set_spins(s0)
            g.set_temperature(T)
            g.set_applied((0.1, -0.2, 0.3))
            g.step(0, 1)
            a = g.det_field()
            g.set_staggered(stag)
            m = g.run_sampled(1, 25, 10)
            out.append((g.get_spins(), a, g.det_field(), m))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_small_batch_alone_and_in_a_mix(gpu):
    """Members of one-workgroup size step there when all are, and through the shared launches
    beside a larger one: the same trajectories."""
    members = [(_sc((10, 10, 10), seed=1), 300.0), (_free(65), 100.0), (_sc((9, 5, 7), 3), 0.0),
               (W.fcc_3shell(dims=(3, 4, 5))[0], 200.0)]
    large = (_sc((20, 20, 20), seed=2), 250.0)
    res = []
    for mix in ([], [large]):
        b = SB.Batch(flags=SB.BATCH_GRAPH)
        ids = [b.add(s, _start(s.n, k), T=T, B=(0.0, 0.1, 0.0)) for k, (s, T) in enumerate(members + mix)]
        b.step(7)
        b.set_temperature(ids[0], 50.0)
        b.step(30)
        assert all(b.get_step(k) == 37 for k in ids)
        res.append([b.get_spins(k) for k in ids[:len(members)]])
        b.close()
    for a, c in zip(*res):
        assert np.array_equal(a, c)
