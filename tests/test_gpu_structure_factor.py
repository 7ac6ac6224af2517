"""The two-pass structure factor (plane sums, then the plane axis) against the direct sum."""
import numpy as np
import pytest

import sllg
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _direct(S, mesh, grid, kpts, ua, ub, sel):
    c = S[0][sel] * ua[sel] + 1j * S[1][sel] * ub[sel]
    m, out = mesh[sel].astype(np.int64), []
    for k in kpts.astype(np.int64):
        turns = sum((k[d] * m[:, d]) % grid[d] / grid[d] for d in range(3))
        out.append((c * np.exp(-2j * np.pi * turns)).sum())
    return np.array(out)


# one plane of several chunks (40 x 41 = 1640 spins), a single spin, planes along z, a list with
# more projections than one block's tile, and an extent of one
@pytest.mark.parametrize("dims,line", [((3, 40, 41), 0), ((1, 1, 1), 0), ((33, 17, 5), 2), ((9, 7, 11), None),
                                       ((1, 65, 16), 1)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_structure_factor_planes(gpu, dims, line, prec):
    rng = np.random.default_rng(sum(dims))
    n = int(np.prod(dims))
    sysd = sllg.System(n=n, species=[dict(mu=2.0)], precision=prec)
    mesh = np.stack(np.meshgrid(*(np.arange(d) for d in dims), indexing="ij"), -1).reshape(-1, 3)
    if line is None:
        kpts = np.stack([rng.integers(0, d, 70) for d in dims], 1)
    else:
        kpts = np.zeros((dims[line], 3), np.int64)
        kpts[:, line] = np.arange(dims[line])
    group = rng.integers(0, 4, n)  # group 2 stays empty, 3 is left out
    group[group == 2] = 3
    one = np.ones(n)
    with sllg.Context(sysd) as g:
        s = rng.standard_normal((3, n))
        g.set_spins(s / np.linalg.norm(s, axis=0))
        S = g.get_spins()
        # n terms of modulus <= sqrt(2), each with a phase right to some 2^-51, summed in FP64
        tol = n * 8 * 2.0 ** -52 * np.sqrt(2) + 1e-15
        g.set_sq(dims, mesh, kpts)
        assert np.abs(g.sample_sq()[0] - _direct(S, mesh, dims, kpts, one, one, slice(None))).max() <= tol
        ua, ub = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
        g.set_sq(dims, mesh, kpts, ua=ua, ub=ub, ngroups=3, group=group)
        got = g.sample_sq()
        for k in range(3):
            assert np.abs(got[k] - _direct(S, mesh, dims, kpts, ua, ub, group == k)).max() <= tol
