"""The cosine-transform form of the fast-diagonalisation solver at every transform length, along
every axis, in both precisions; boxes whose columns do not fill a tile. The reference applies
the closed-form eigenbasis (cell-centred cosines) as dense matrices in double precision: the
numerical eigenvectors of the oracle are off by n^2 eps in the lowest modes, which is more than
these bounds from 96 cells on (in double precision).

A transform of n points of magnitude s rounds about log2(n) times: six transforms of at most
9 stages and the division are 60 roundings, so the relative error is below 100 eps of the
largest mode's. The bounds are 200 eps, which leaves the conditioning of the low modes a factor
of two."""

import numpy as np
import pytest

from helpers import PREC, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

LENGTHS = (16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512)
SHAPES = [(16, 16, n) for n in LENGTHS] + [(16, n, 24) for n in LENGTHS[1:]] + [(n, 24, 16) for n in LENGTHS[1:]]


def closed_form_solve(rhs, dx):
    """psi = V Lambda^-1 V^T rhs over the last three axes, the constant mode dropped."""
    shape = rhs.shape[-3:]
    basis, lam = [], []
    for n in shape:
        k = np.arange(n)
        v = np.sqrt(2.0 / n) * np.cos(np.pi * k[:, None] * (k[None, :] + 0.5) / n)
        v[0] /= np.sqrt(2.0)
        basis.append(v)
        lam.append(4.0 / dx**2 * np.sin(np.pi * k / (2 * n)) ** 2)
    f = np.einsum("czyx,kz,ly,mx->cklm", rhs, *basis, optimize=True)
    total = lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :]
    total[0, 0, 0] = np.inf
    return np.einsum("cklm,kz,ly,mx->czyx", f / total, *basis, optimize=True)


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("shape", SHAPES)
def test_dct_solve_matches_closed_form(dev, precision, shape):
    from sopht_amd.numeric.eulerian_grid_ops import FastDiagPoissonSolver3D

    real_t = PREC[precision]
    dx = 0.05
    rng = np.random.default_rng(sum(shape))
    rhs = rng.standard_normal((3, *shape)).astype(real_t)
    ref = closed_form_solve(rhs.astype(np.float64), dx)
    s = FastDiagPoissonSolver3D(*shape, dx=dx, real_t=real_t)
    out = to_dev(np.zeros_like(rhs), dev)
    s.vector_field_solve(out, to_dev(rhs, dev))
    # the dense products of the reference round n eps(64)
    bound = 200 * float(np.finfo(real_t).eps) + 64 * max(shape) * float(np.finfo(np.float64).eps)
    assert rel_l2(to_host(out), ref) <= bound, rel_l2(to_host(out), ref)
    # one component, in place
    one = to_dev(rhs[1], dev)
    s.solve(one, one)
    assert rel_l2(to_host(one), ref[1]) <= bound, rel_l2(to_host(one), ref[1])
