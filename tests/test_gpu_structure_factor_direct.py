"""Structure factors of many wave-vectors and groups, which are summed directly, against FP64 sums."""
import time

import numpy as np
import pytest

import sllg

pytestmark = pytest.mark.gpu


def _handle(dims, prec, rng):
    n = int(np.prod(dims))
    g = sllg.Context(sllg.System(n=n, species=[dict(mu=2.0)], precision=prec))
    s = rng.standard_normal((3, n))
    g.set_spins(s / np.linalg.norm(s, axis=0))
    mesh = np.stack(np.meshgrid(*(np.arange(d) for d in dims), indexing="ij"), -1).reshape(-1, 3)
    return g, mesh, g.get_spins()


# groups of less than a chunk, of several chunks and one spin more, no spins, left-out spins; one
# wave-vector more than a block's threads; with and without weights
@pytest.mark.parametrize("dims, nk, ngroups", [((12, 13, 14), 257, 40), ((9, 16, 31), 300, 7), ((20, 20, 20), 90, 200),
                                               ((40, 33, 1), 256, 11), ((5, 4, 3), 513, 30)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_many_wave_vectors_and_groups(gpu, dims, nk, ngroups, prec):
    rng = np.random.default_rng(nk)
    g, mesh, S = _handle(dims, prec, rng)
    n = len(mesh)
    kpts = np.stack([rng.integers(0, d, nk) for d in dims], 1)
    group = rng.integers(0, ngroups + 1, n)  # the last value leaves a spin out
    group[group == 3] = 4  # a group without spins
    turns = sum(np.outer(mesh[:, d], kpts[:, d]) % dims[d] / dims[d] for d in range(3))
    ph = np.exp(-2j * np.pi * turns)
    # n terms of modulus <= sqrt(2), each with a phase right to some 2^-50, summed in FP64
    tol = n * 16 * 2.0 ** -52 * np.sqrt(2) + 1e-15
    for ua, ub in ((None, None), (rng.uniform(-1, 1, n), rng.uniform(-1, 1, n))):
        g.set_sq(dims, mesh, kpts, ua=ua, ub=ub, ngroups=ngroups, group=group)
        c = S[0] * (1 if ua is None else ua) + 1j * S[1] * (1 if ub is None else ub)
        want = np.stack([(c[group == k, None] * ph[group == k]).sum(0) for k in range(ngroups)])
        for _ in range(2):
            assert np.abs(g.sample_sq() - want).max() <= tol
    # a line of wave-vectors on the same handle afterwards (two passes), then many again
    line = np.zeros((dims[1], 3), np.int64)
    line[:, 1] = np.arange(dims[1])
    g.set_sq(dims, mesh, line)
    want = ((S[0] + 1j * S[1])[:, None] * np.exp(-2j * np.pi * (np.outer(mesh[:, 1], line[:, 1]) % dims[1] / dims[1]))).sum(0)
    assert np.abs(g.sample_sq()[0] - want).max() <= tol
    g.set_sq(dims, mesh, kpts)
    assert np.abs(g.sample_sq()[0] - ((S[0] + 1j * S[1])[:, None] * ph).sum(0)).max() <= tol
    g.close()


def test_many_groups_take_no_longer_than_one_sum(gpu):
    """48^3 spins in 300 groups, 300 wave-vectors: 15 ms with a block for every plane of a group, 0.4
    summed directly."""
    rng = np.random.default_rng(1)
    dims = (48, 48, 48)
    g, mesh, _ = _handle(dims, "fp32", rng)
    g.set_sq(dims, mesh, rng.integers(0, 48, (300, 3)), ngroups=300, group=rng.integers(0, 300, len(mesh)))
    g.sample_sq()
    best = 1e9
    for _ in range(3):
        t = time.perf_counter()
        g.sample_sq()
        best = min(best, time.perf_counter() - t)
    g.close()
    assert best < 4e-3
