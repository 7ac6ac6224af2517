"""The register-transform convolution on narrow and deep meshes: the inverse transforms along z are
dealt to a plane block's 256 threads by eights, fours, pairs or single values of z, against the FP64
whole-grid transforms."""
import numpy as np
import pytest

import sllg

pytestmark = pytest.mark.gpu

# The transforms of a padded grid of at most 2^21 points take 21 radix-2 stages each way; every
# stage adds a rounding error of about 2^-24 of the largest field.
TOL = 2 * 21 * 2.0 ** -24


def _field(prec, dims, s):
    n = s.shape[1]
    mesh = np.stack(np.meshgrid(*(np.arange(d) for d in dims), indexing="ij"), -1).reshape(-1, 3)
    sysd = sllg.System(n=n, species=[dict(mu=2.2, lambda_=0.1), dict(mu=0.7, lambda_=0.1)],
                       spin_species=(np.arange(n) % 2).astype(np.uint32), precision=prec,
                       dip=dict(enabled=1, mesh=mesh, dim=dims, nk=(1, 1, 1), abc=(3e-10, 2.5e-10, 4e-10), refresh=1))
    with sllg.Context(sysd) as g:
        g.set_spins(s)
        g.step(0, 1)  # the dipolar field is refreshed at the spins given
        return g.field()


def _z_per_thread(ly, lz):
    rows = 1 << max(2, (ly - 1).bit_length())  # the padded rows a plane transforms
    return next((z for z in (8, 4, 2) if rows * -(-lz // z) >= 256), 1)


DIMS = [(16, 16, 32), (64, 8, 32), (4, 128, 32), (128, 4, 24), (4, 8, 31),  # narrow and deep
        (5, 128, 17), (5, 128, 16), (5, 128, 9), (5, 100, 8), (5, 128, 5), (5, 128, 4), (5, 70, 3), (5, 128, 2),
        (5, 64, 25), (5, 64, 24), (5, 64, 13), (5, 50, 12), (5, 64, 8), (5, 33, 7), (5, 64, 6), (5, 64, 4),
        (5, 32, 31), (5, 32, 29), (5, 32, 28), (5, 32, 16), (5, 30, 14), (5, 17, 8),
        (5, 16, 31), (5, 16, 30), (5, 8, 32), (5, 5, 2)]


def test_every_split_is_met():
    assert {_z_per_thread(y, z) for _, y, z in DIMS} == {1, 2, 4, 8}


@pytest.mark.parametrize("dims", DIMS)
def test_narrow_and_deep_meshes(gpu, dims):
    s = np.random.default_rng(sum(dims)).standard_normal((3, int(np.prod(dims))))
    s /= np.linalg.norm(s, axis=0)
    ref, got = (_field(p, dims, s) for p in ("fp64", "fp32"))
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()
