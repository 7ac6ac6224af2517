"""Line-block reader (neighbours staged in LDS by whole lattice lines) against the packed entries
of the same encoding: rows keep their order of sums, so the bits are equal."""
import numpy as np
import pytest

import sllg
from sllg import workloads as W

pytestmark = pytest.mark.gpu

PACKED = dict(tpb=256, line_mode=1)


def _start(n, seed):
    s = np.random.default_rng(seed).standard_normal((3, n))
    return s / np.linalg.norm(s, axis=0)


def _system(kind, dims, shells, nc=1, pbc=(1, 1, 1), order=None, flags=0):
    uc = sllg.unit_cell(kind)
    ints, _ = sllg.shells(uc, [5e-21, 1e-21, -4e-22, 2e-22][:shells])
    na = {"sc": 1, "bct": 2, "fcc": 4}[kind]
    xadj, adj, vals = sllg.build_csr(uc, dims, ints, [2.0] * na, ncomp=nc, pbc=pbc)
    if order is not None:  # the entries of each row in another order
        rng = np.random.default_rng(order)
        p = np.concatenate([rng.permutation(np.arange(a, b)) for a, b in zip(xadj[:-1], xadj[1:])])
        adj, vals = adj[p], np.ascontiguousarray(vals[:, p])
    return sllg.System(n=int(np.prod(dims)) * na, species=[dict(mu=2.0, lambda_=0.1, k1u=1e-23)], precision="fp32",
                       exch=dict(format=sllg.EXCH_CSR, xadj=xadj, adjncy=adj, vals=vals, n_atoms=na), seed=9, flags=flags)


def _run(s, T, launch, stag=None):
    with sllg.Context(s) as g:
        if launch:
            g.set_launch(**launch)
        g.set_spins(_start(s.n, 3))
        g.set_temperature(T)
        g.set_applied((0.1, -0.2, 0.3))
        if stag is not None:
            g.set_staggered(stag)
        g.step(0, 3)
        m = g.reduce(energy=False)[0]
        g.step(3, 4)
        return g.get_spins(), m, g.info()["exch_encoding"]


# cells per line around what a wave load holds (30 + 2 staged cells, 62, 126), the shortest line,
# lines that do not fill a wave, several lines to a workgroup; one, two and four sublattices
SHAPES = [("fcc", (11, 12, 4), 2), ("fcc", (9, 10, 11), 3), ("fcc", (5, 7, 30), 3), ("fcc", (5, 7, 31), 3),
          ("fcc", (4, 5, 62), 2), ("fcc", (3, 5, 63), 2), ("fcc", (3, 4, 127), 1), ("fcc", (20, 41, 6), 3),
          ("sc", (17, 19, 23), 3), ("sc", (40, 41, 7), 4), ("sc", (5, 6, 101), 2), ("bct", (11, 13, 17), 1),
          ("bct", (9, 50, 12), 2)]


@pytest.mark.parametrize("kind, dims, shells", SHAPES)
@pytest.mark.parametrize("T", [0.0, 200.0])
def test_blocks_equal_packed(gpu, kind, dims, shells, T):
    s = _system(kind, dims, shells)
    want, m0, _ = _run(s, T, PACKED)
    got, m1, enc = _run(s, T, None)
    assert "-blocks%dx" % dims[2] in enc
    assert np.array_equal(got, want) and np.array_equal(m0, m1)


@pytest.mark.parametrize("nc", [3, 9])
@pytest.mark.parametrize("pbc", [(1, 1, 1), (0, 0, 1), (0, 1, 1), (1, 0, 1)])
def test_components_and_open_faces(gpu, nc, pbc):
    s = _system("fcc", (7, 8, 13), 2, nc, pbc)
    stag = 0.2 * _start(s.n, 5)
    want = _run(s, 100.0, PACKED, stag)[0]
    for launch in (None, dict(tpb=256, xcd=0, thermal_cache=0, line_mode=2)):
        got, _, enc = _run(s, 100.0, launch, stag)
        assert "-blocks13x" in enc
        assert np.array_equal(got, want)


@pytest.mark.parametrize("kw", [dict(pbc=(1, 1, 0)), dict(order=1), dict(dims=(20, 20, 3)), dict(flags=sllg.FLAG_NO_LINE_MODE)])
def test_other_encodings_keep_their_entries(gpu, kw):
    kw = dict(kw)
    s = _system("fcc", kw.pop("dims", (7, 8, 13)), 2, **kw)
    want = _run(s, 100.0, PACKED)[0]
    got, _, enc = _run(s, 100.0, None)
    assert "-blocks" not in enc
    assert np.array_equal(got, want)


def test_blocks_tuned(gpu):
    s = _system("fcc", (9, 10, 11), 3)
    with sllg.Context(s) as g:
        g.set_spins(_start(s.n, 3))
        g.set_temperature(50.0)
        before = g.get_spins()
        r = g.autotune(3)
        assert r["line_mode"] in (1, 2) and r["candidates"] > 4
        assert np.array_equal(g.get_spins(), before)
        g.step(0, 5)
        got = g.get_spins()
    with sllg.Context(s) as g:
        g.set_launch(**PACKED)
        g.set_spins(before)
        g.set_temperature(50.0)
        g.step(0, 5)
        assert np.array_equal(g.get_spins(), got)
