"""Long rows of 9 components: one-workgroup steps up to 200,000 entries times components, two launches
a step beyond, unless a batch has many such members.  llg_profile_kernels names the kernels that ran."""
import numpy as np
import pytest

import sllg
from sllg import batch as SB
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _fcc(dims, nc):
    return W.fcc_3shell(dims=dims, ncomp=nc)[0]


def _start(n, seed):
    s = np.random.default_rng(seed).standard_normal((3, n))
    return s / np.linalg.norm(s, axis=0)


# entries x components: 181,440 (480 spins) and 204,120 (540) with 9, 127,008 with 3, 42,336 with 1
@pytest.mark.parametrize("dims, nc, small", [((4, 5, 6), 9, True), ((3, 5, 9), 9, False), ((6, 6, 7), 9, False),
                                             ((6, 6, 7), 3, True), ((6, 6, 7), 1, True)])
def test_which_steps_run(gpu, dims, nc, small):
    s = _fcc(dims, nc)
    out = []
    for launch in (None, (256, 1, 2, 1, 0, 0)):
        with sllg.Context(s) as g:
            if launch:
                g.set_launch(*launch)
            g.set_spins(_start(s.n, 1))
            g.set_temperature(200.0)
            names = set(g.profile_kernels(0, 3))
            assert names == ({"heun_steps"} if small and not launch else {"heun_predictor", "heun_corrector"})
            g.step(3, 20)
            out.append(g.get_spins())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("count", [2, 96])
def test_batches_of_few_and_many(gpu, count):
    """The same trajectories whichever steps run."""
    s = _fcc((3, 5, 9), 9)
    out = []
    for launch in (False, True):
        b = SB.Batch()
        if launch:
            b.set_launch(256)
        ids = [b.add(s, _start(s.n, k), T=2.0 * k) for k in range(count)]
        b.step(20)
        out.append([b.get_spins(k) for k in ids])
        b.close()
    for a, c in zip(*out):
        assert np.array_equal(a, c)
