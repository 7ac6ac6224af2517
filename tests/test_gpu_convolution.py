"""The register-transform convolution (FP32, mirror-symmetric kernel, mesh up to 128 x 128 x 32)
against the FP64 whole-grid transforms."""
import numpy as np
import pytest

import sllg

pytestmark = pytest.mark.gpu

# The transforms of a padded grid of at most 2^21 points take 21 radix-2 stages each way; every
# stage adds a rounding error of about 2^-24 of the largest field.
TOL = 2 * 21 * 2.0 ** -24


def _mesh(dims, fill, rng):
    m = np.stack(np.meshgrid(*(np.arange(d) for d in dims), indexing="ij"), -1).reshape(-1, 3)
    return m if fill == 1.0 else rng.permutation(m)[:max(1, int(fill * len(m)))]


def _field(prec, mesh, dims, s, fftx, species, spec, flags=0):
    sysd = sllg.System(n=len(mesh), species=species, spin_species=spec, precision=prec, flags=flags,
                       dip=dict(enabled=1, mesh=mesh, dim=dims, nk=(1, 1, 1), abc=(3e-10, 2.5e-10, 4e-10), refresh=1),
                       fftx=fftx)
    with sllg.Context(sysd) as g:
        g.set_spins(s)
        g.step(0, 1)  # the dipolar field is refreshed at the spins given
        return g.field()


# the smallest extents, one plane along z, extents just past a power of two, the largest, padded
# extents of 16 to 256 along either axis
@pytest.mark.parametrize("dims", [(4, 4, 1), (8, 5, 2), (9, 17, 5), (17, 33, 3), (33, 65, 7), (65, 8, 32), (64, 128, 9),
                                  (128, 12, 31), (128, 128, 32)])
@pytest.mark.parametrize("fill", [1.0, 0.6])
def test_dipolar_register_transforms(gpu, dims, fill):
    rng = np.random.default_rng(sum(dims))
    mesh = _mesh(dims, fill, rng)
    s = rng.standard_normal((3, len(mesh)))
    s /= np.linalg.norm(s, axis=0)
    spec = (np.arange(len(mesh)) % 2).astype(np.uint32)
    species = [dict(mu=2.2, lambda_=0.1), dict(mu=0.7, lambda_=0.1)]
    ref, got = (_field(p, mesh, dims, s, [], species, spec) for p in ("fp64", "fp32"))
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


# symmetric tensors with the mirror images take the register transforms; an antisymmetric part
# or a missing image keeps the general kernel: both give the FP64 field
@pytest.mark.parametrize("kind", ["isotropic", "mirror", "dmi", "one_sided"])
@pytest.mark.parametrize("dims", [(5, 9, 3), (16, 8, 4)])
def test_fft_exchange_kernel_classes(gpu, kind, dims):
    rng = np.random.default_rng(3)
    J = np.eye(3) * 3e-21
    vecs = [(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]
    fftx = [(0, 0, v, J) for v in vecs]
    if kind == "mirror":  # next neighbours in the xy plane with an off-diagonal xy part
        for x in (1, -1):
            for y in (1, -1):
                O = np.zeros((3, 3))
                O[0, 1] = O[1, 0] = x * y * 4e-22
                fftx.append((0, 0, (x, y, 0), J * 0.2 + O))
    elif kind == "dmi":
        D = np.zeros((3, 3))
        D[0, 1], D[1, 0] = 5e-22, -5e-22
        fftx += [(0, 0, (1, 0, 0), D), (0, 0, (-1, 0, 0), -D)]
    elif kind == "one_sided":
        fftx.append((0, 0, (1, 1, 0), J * 0.1))
    mesh = _mesh(dims, 0.8, rng)
    s = rng.standard_normal((3, len(mesh)))
    s /= np.linalg.norm(s, axis=0)
    species = [dict(mu=2.2, lambda_=0.1)]
    ref, got = (_field(p, mesh, dims, s, fftx, species, None) for p in ("fp64", "fp32"))
    # the field is taken at the spins after the step: FP32 spins differ by 2^-24 or so each
    assert np.abs(got - ref).max() <= (TOL + 8 * 2.0 ** -24) * np.abs(ref).max()
