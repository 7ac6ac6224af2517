"""Which FP64 systems take the lane-uniform records: small ones whose longest slice has more than four
records an entry keep the sliced CSR, which is faster for them.  The sums are the same either way."""
import numpy as np
import pytest

import sllg
from sllg import workloads as W

pytestmark = pytest.mark.gpu


def _chain(n, k, distinct):
    """k neighbours a row along a ring, couplings drawn from `distinct` values (0: all different)."""
    rng = np.random.default_rng(0)
    adj = np.stack([(np.arange(n) + o) % n for o in (1, -1, 2, -2)[:k]], 1).astype(np.uint32)
    v = rng.normal(0, 100, distinct)[rng.integers(0, distinct, n * k)] if distinct else rng.normal(0, 100, n * k)
    return sllg.System(n=n, species=[dict(mu=2.0)], seed=3,
                       exch=dict(format=sllg.EXCH_CSR, xadj=np.arange(0, n * k + 1, k, dtype=np.uint32),
                                 adjncy=adj.ravel(), vals=v[None]))


def _bct(dims):
    uc = sllg.unit_cell("bct")
    x, a, v = sllg.build_csr(uc, dims, sllg.shells(uc, [5e-21])[0], [2.0] * 2)
    return sllg.System(n=2 * int(np.prod(dims)), species=[dict(mu=2.0)], seed=3,
                       exch=dict(format=sllg.EXCH_CSR, xadj=x, adjncy=a, vals=v, n_atoms=2))


CASES = [
    (lambda: _chain(64, 4, 0), False), (lambda: _chain(128, 2, 0), False), (lambda: _chain(40, 4, 0), False),
    (lambda: _chain(200, 4, 8), False), (lambda: _chain(200, 4, 2), True), (lambda: _bct((3, 3, 3)), False),
    (lambda: _bct((6, 6, 6)), True), (lambda: W.fcc_3shell(dims=(7, 7, 7), precision="fp64")[0], False),
    (lambda: W.fcc_3shell(dims=(40, 5, 3), precision="fp64")[0], False),
    (lambda: W.fcc_3shell(dims=(10, 10, 10), precision="fp64")[0], True),
    (lambda: W.fcc_3shell(dims=(30, 31, 20), precision="fp64")[0], True),  # 74,400 spins
    (lambda: W.sc_ferro(L=5, precision="fp64")[0], True),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_records_where_they_are_faster(gpu, case):
    make, uniform = CASES[case]
    s = make()
    s.precision = "fp64"
    s0 = np.random.default_rng(4).standard_normal((3, s.n))
    s0 /= np.linalg.norm(s0, axis=0)
    out = []
    for flags in (0, sllg.FLAG_NO_SLICE_SHARING | sllg.FLAG_NO_SUBLATTICE_ORDER):
        s.flags = flags
        with sllg.Context(s) as g:
            assert ("uniform" in g.info()["exch_encoding"]) == (uniform and flags == 0)
            g.set_spins(s0)
            g.set_temperature(200.0)
            g.step(0, 3)
            out.append((g.get_spins(), g.field()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
