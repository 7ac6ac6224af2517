"""FP64 handles on the lane-uniform CSR records (and in the sublattice-major device order)
against the sliced CSR that LLG_FLAG_NO_SLICE_SHARING keeps: the same sums, so the same bits."""
import numpy as np
import pytest

import sllg
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _random_csr(n, k, seed, values):
    """Rows of uneven length with random neighbours; `values` distinct couplings."""
    rng = np.random.default_rng(seed)
    ln = rng.integers(0, k + 1, n)
    xadj = np.concatenate([[0], np.cumsum(ln)]).astype(np.uint32)
    adj = rng.integers(0, n, int(xadj[-1])).astype(np.uint32)
    v = rng.choice(rng.normal(0, 100, values), len(adj))
    return xadj, adj, v[None]


def _system(kind):
    if kind == "random":  # couplings and neighbours differ from row to row: no records
        x, a, v = _random_csr(700, 6, 1, 3)
        return sllg.System(n=700, species=[dict(mu=2.0)], exch=dict(format=sllg.EXCH_CSR, xadj=x, adjncy=a, vals=v))
    if kind == "one_class":  # every row its own neighbour
        n = 65
        x = np.arange(n + 1, dtype=np.uint32)
        return sllg.System(n=n, species=[dict(mu=2.0)],
                           exch=dict(format=sllg.EXCH_CSR, xadj=x, adjncy=np.arange(n, dtype=np.uint32),
                                     vals=np.full((1, n), 50.0)))
    dims, nc = kind[1], kind[2]
    if kind[0] == "fcc":
        return W.fcc_3shell(dims=dims, ncomp=nc)[0]
    if kind[0] == "film":
        s = W.sc_film_dip(*dims)[0]
        s.dip = {"enabled": 0}
        return s
    return W.sc_ferro(dims=dims, ncomp=nc)[0]


KINDS = ["random", "one_class", ("sc", (1, 1, 1), 1), ("sc", (2, 2, 2), 1), ("sc", (5, 7, 11), 3), ("sc", (3, 4, 64), 1),
         ("sc", (4, 3, 65), 9), ("fcc", (3, 3, 3), 1), ("fcc", (2, 5, 17), 3), ("film", (6, 9, 5), 1)]


@pytest.mark.parametrize("kind", KINDS, ids=str)
@pytest.mark.parametrize("scheme", ["heun", "rk4", "rk5"])
def test_uniform_records_equal_sliced_csr(gpu, kind, scheme):
    s = _system(kind)
    s.precision, s.scheme, s.seed = "fp64", scheme, 3
    rng = np.random.default_rng(4)
    s0 = rng.standard_normal((3, s.n))
    s0 /= np.linalg.norm(s0, axis=0)
    out = []
    for flags in (0, sllg.FLAG_NO_SLICE_SHARING | sllg.FLAG_NO_SUBLATTICE_ORDER):
        s.flags = flags
        with sllg.Context(s) as g:
            # a 3^3 fcc box wraps in too many ways for records, as does the random graph
            assert ("uniform" in g.info()["exch_encoding"]) == (flags == 0 and kind not in ("random", ("fcc", (3, 3, 3), 1)))
            g.set_spins(s0)
            assert np.array_equal(g.get_spins(), s0)
            g.set_temperature(200.0)
            g.step(0, 3)
            out.append((g.get_spins(), g.field(), g.det_field(), g.reduce()))
    for a, b in zip(out[0][:3], out[1][:3]):
        assert np.array_equal(a, b)
    # sums over the spins in another order: n terms of modulus <= 1 / n and <= |E| / n
    assert np.abs(out[0][3][0] - out[1][3][0]).max() <= s.n * 2.0 ** -52
    scale = np.abs(out[1][1]).max() * 9.27e-24 * 2.22 * s.n
    assert abs(out[0][3][1] - out[1][3][1]) <= s.n * 2.0 ** -50 * max(scale, 1e-30)


@pytest.mark.parametrize("n_cells", [(16, 16, 63), (16, 16, 64)])  # 64,512 and 65,536 spins
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_state_round_trip_across_io_paths(gpu, n_cells, prec):
    s, s0 = W.fcc_3shell(dims=n_cells, precision=prec)
    with sllg.Context(s) as g:
        for k in range(2):  # the second upload goes over a stepped handle
            g.set_spins(s0)
            got = g.get_spins()
            assert np.array_equal(got, s0 if prec == "fp64" else s0.astype(np.float32).astype(np.float64))
            g.step(0, 2)
