"""The ordered gather takes a cell's contributors sixteen at a time: cells with counts around
multiples of sixteen, next to each other in one wavefront, add up bit for bit as the serial
node order does, for one component and for three."""

import numpy as np
import pytest

from helpers import PREC, to_dev, to_host
from oracle import ib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("counts", [(1,), (15, 16, 17), (33, 1, 32, 31), (64, 2, 100)])
@pytest.mark.parametrize("ncomp", [1, 3])
def test_spread_counts_around_sixteen(dev, precision, counts, ncomp, rng):
    from sopht_amd.numeric.immersed_boundary_ops import EulerianLagrangianGridCommunicator3D

    real_t = PREC[precision]
    n = 24
    dx = real_t(1.0 / n)
    shift = real_t(dx / 2)
    # one cluster of nodes per count, each in one cell, five cells apart along x
    X = np.concatenate([np.array([[3.3 + 5 * i], [9.4], [11.2]]) + 0.4 * rng.random((3, k))
                        for i, k in enumerate(counts)], axis=1) * float(dx)
    X = X[:, rng.permutation(X.shape[1])]
    m = X.shape[1]
    idx, d = ib.local_eulerian_grid_support(X, dx, shift, real_t)
    w, _ = ib.cosine_weights(d, dx, real_t)
    shape = (3, n, n, n) if ncomp == 3 else (n, n, n)
    Fl = rng.standard_normal((3, m) if ncomp == 3 else m).astype(real_t)
    F0 = rng.standard_normal(shape).astype(real_t)
    ref = F0.copy()
    ib.spread(ref, Fl, w, idx)
    c = EulerianLagrangianGridCommunicator3D(dx, shift, m, 2, real_t, n_components=ncomp)
    F = to_dev(F0, dev)
    c.lagrangian_to_eulerian_grid_interpolation_kernel(F, to_dev(Fl, dev), to_dev(w, dev), to_dev(idx, dev))
    c.check_support_in_domain()
    np.testing.assert_array_equal(to_host(F), ref)
