"""The reader a new handle takes: line blocks by their lines' length and their rows' entries, at both
sides of the rule; whichever it is, the blocks give the packed entries' bits."""
import numpy as np
import pytest

import sllg

pytestmark = pytest.mark.gpu


def _system(kind, dims, shells):
    uc = sllg.unit_cell(kind)
    ints, _ = sllg.shells(uc, [5e-21, 1e-21, -4e-22, 2e-22][:shells])
    na = {"sc": 1, "bct": 2, "fcc": 4}[kind]
    xadj, adj, vals = sllg.build_csr(uc, dims, ints, [2.0] * na)
    return sllg.System(n=int(np.prod(dims)) * na, species=[dict(mu=2.0, lambda_=0.1, k1u=1e-23)], precision="fp32",
                       exch=dict(format=sllg.EXCH_CSR, xadj=xadj, adjncy=adj, vals=vals, n_atoms=na), seed=9)


# kind, cells, shells, the line_mode a new handle has, whether blocks are built: at the limits of the
# line length for short and long rows and one past them, at the sizes from which short rows and line
# encodings change reader, and small systems, which have the blocks either way
CASES = [
    ("sc", (13, 29, 56), 2, 2, True), ("sc", (13, 29, 57), 2, 1, False), ("bct", (11, 17, 63), 1, 2, True),
    ("bct", (11, 17, 65), 1, 1, False), ("sc", (7, 19, 128), 3, 2, True), ("sc", (7, 19, 129), 3, 1, False),
    ("fcc", (3, 11, 129), 3, 2, True), ("bct", (79, 95, 39), 1, 2, True), ("bct", (79, 97, 41), 1, 1, False),
    ("sc", (17, 23, 64), 2, 1, False), ("sc", (64, 64, 16), 2, 2, True), ("sc", (128, 64, 16), 2, 1, False),
    ("bct", (31, 33, 64), 2, 2, True), ("bct", (33, 33, 64), 2, 1, False), ("fcc", (41, 39, 64), 3, 1, False),
    ("fcc", (39, 39, 64), 3, 2, True), ("sc", (5, 6, 101), 2, 1, True), ("fcc", (3, 4, 127), 1, 1, True),
]


@pytest.mark.parametrize("kind, dims, shells, mode, built", CASES)
def test_default_reader(gpu, kind, dims, shells, mode, built):
    s = _system(kind, dims, shells)
    s0 = np.random.default_rng(3).standard_normal((3, s.n))
    s0 /= np.linalg.norm(s0, axis=0)
    out = {}
    for m in (None, 0, 2):
        with sllg.Context(s) as g:
            enc = g.info()["exch_encoding"]
            assert ("-blocks" in enc or len(enc) == 63) == built  # a long name is cut at 63 characters
            if m is None:
                f = s.flags
                s.flags = f | sllg.FLAG_TUNE_FIXED_READER
                with sllg.Context(s) as q:
                    assert q.autotune(1)["line_mode"] == mode
                s.flags = f
            else:
                g.set_launch(256, line_mode=m)
            g.set_spins(s0)
            g.set_temperature(200.0)
            g.step(0, 2)
            out[m] = g.get_spins()
    if built:  # blocks: the packed entries' bits
        assert np.array_equal(out[0], out[2])
    assert any(np.array_equal(out[None], out[m]) for m in (0, 2)) or "line" in enc
