"""The register-transform convolution beside pairwise exchange: during a run the dipolar refresh reads
the spins from their AoS3 gather copy, through a mesh map that need not be the identity."""
import numpy as np
import pytest

import sllg

pytestmark = pytest.mark.gpu

DIMS, MU, J, DT, STEPS = (24, 19, 7), 2.2, 3e-21, 1e-16, 7

# A step rounds each spin component by less than 8 x 2^-24 (update and normalisation); its field of at most
# 6 J / mu plus the dipolar one turns a spin by less than 0.016, so the field's own relative error (42 x
# 2^-24 for the transforms, 8 for the neighbour sums) adds less than 2^-24, and earlier errors grow by less
# than 1 + 2 x 0.016 a step.
TOL = STEPS * 9 * 1.032 ** STEPS * 2.0 ** -24


def _system(order, fill, precision):
    rng = np.random.default_rng(11)
    mesh = np.stack(np.meshgrid(*(np.arange(d) for d in DIMS), indexing="ij"), -1).reshape(-1, 3)
    if order == "shuffled":
        mesh = rng.permutation(mesh)
    mesh = mesh[:int(fill * len(mesh))]
    at = np.full(DIMS, -1)
    at[tuple(mesh.T)] = np.arange(len(mesh))
    xadj, adj = [0], []
    for p in mesh:
        for d in ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)):
            q = p + d
            if np.all(q >= 0) and np.all(q < DIMS) and at[tuple(q)] >= 0:
                adj.append(at[tuple(q)])
        xadj.append(len(adj))
    vals = np.full((1, len(adj)), J / (MU * 9.2740100783e-24))
    n = len(mesh)
    return sllg.System(n=n, species=[dict(mu=MU, lambda_=0.1)],
                       exch=dict(format=sllg.EXCH_CSR, xadj=np.array(xadj, dtype=np.uint32),
                                 adjncy=np.array(adj, dtype=np.uint32), vals=vals),
                       dip=dict(enabled=1, mesh=mesh, dim=DIMS, nk=(1, 1, 1), abc=(3e-10, 2.5e-10, 4e-10), refresh=1),
                       precision=precision, dt=DT, seed=9, update=3)


@pytest.mark.parametrize("order,fill", [("natural", 1.0), ("shuffled", 1.0), ("natural", 0.6), ("shuffled", 0.6)])
def test_refresh_from_the_gather_copy(gpu, order, fill):
    out = {}
    for name, prec, shape in [("copy", "fp32", (256, 1, 2, 1, 1, 1)), ("soa", "fp32", (256, 1, 2, 1, 0, 1)),
                              ("default", "fp32", None), ("fp64", "fp64", None)]:
        sysd = _system(order, fill, prec)
        with sllg.Context(sysd) as g:
            if shape:
                g.set_launch(*shape)
            s = np.random.default_rng(2).standard_normal((3, sysd.n))
            g.set_spins(s / np.linalg.norm(s, axis=0))
            g.step(0, STEPS - 2)
            g.step(STEPS - 2, 2)
            out[name] = (g.get_spins(), g.field())
    for a, b, c in zip(out["copy"], out["soa"], out["default"]):
        assert np.array_equal(a, b) and np.array_equal(a, c)
    assert np.abs(out["copy"][0] - out["fp64"][0]).max() <= TOL
