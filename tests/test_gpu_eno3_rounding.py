"""The ENO3 flux rounds the same way whatever the fields' layout: dense fields (row vectors) and
fields whose cells are two apart along x (one column or one cell per thread) give the same bits, in
the accumulating, stepping and storing forms. Its products are fused into the sums: on smooth fields
the flux is closer to the 64-bit one than the reference's 32-bit evaluation, which rounds every
product. (A face sums terms of 5/6, 1/3 and 1/6; fusing the two larger products drops roundings of
these relative sizes, so over 10^5 cells the errors differ by far more than their scatter.)"""

import numpy as np
import pytest

from oracle import stencils as S

from helpers import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


def spne():
    from sopht_amd.numeric import eulerian_grid_ops

    return eulerian_grid_ops


def spread_out(a, dev):
    big = np.full((*a.shape[:-1], 2 * a.shape[-1]), 7.0, dtype=a.dtype)
    big[..., ::2] = a
    return to_dev(big, dev)[..., ::2]


@pytest.mark.parametrize("real_t", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("shape", [(5, 5, 5), (9, 7, 37), (36, 6, 66), (40, 12, 256)])
def test_layouts_give_the_same_bits(dev, real_t, shape):
    rng = np.random.default_rng(21)
    f, one = rng.uniform(-1, 1, (2, *shape)).astype(real_t)
    u, w = rng.uniform(-1, 1, (2, 3, *shape)).astype(real_t)
    flux = spne().gen_advection_flux_conservative_eno3_pyst_kernel_3d(real_t)
    step = spne().gen_advection_timestep_euler_forward_conservative_eno3_pyst_kernel_3d(real_t, field_type="vector")
    results = []
    for place in (to_dev, spread_out):
        out, buf, vec = place(one, dev), place(one, dev), place(w, dev)
        flux(out, place(f, dev), place(u, dev), 0.25)
        step(vec, buf, place(u, dev), 0.25)
        results.append([to_host(t) for t in (out, vec, buf)])
    for a, b in zip(*results):
        np.testing.assert_array_equal(a, b)
    stored = spne().eno3_advection_flux(to_dev(f, dev), to_dev(u, dev), 0.25)
    zero = spread_out(np.zeros_like(f), dev)
    flux(zero, spread_out(f, dev), spread_out(u, dev), 0.25)
    np.testing.assert_array_equal(to_host(stored), to_host(zero))


@pytest.mark.parametrize("seed", [1, 2, 3])
@pytest.mark.parametrize("place", [to_dev, spread_out], ids=["dense", "spread"])
def test_products_are_fused(dev, place, seed):
    shape = (40, 48, 56)
    rng = np.random.default_rng(seed)
    grid = np.meshgrid(*[np.arange(n) / 56 for n in shape], indexing="ij")

    def smooth():
        k, phase = rng.uniform(2, 9, 3), rng.uniform(0, 6)
        return (1.5 + np.sin(sum(a * g for a, g in zip(k, grid)) + phase)).astype(np.float32)

    f, u = smooth(), np.stack([smooth() for _ in range(3)])
    exact, single = np.zeros(shape), np.zeros(shape, dtype=np.float32)
    S.advection_flux_conservative_eno3(exact, f.astype(np.float64), u.astype(np.float64), 0.5)
    S.advection_flux_conservative_eno3(single, f, u, np.float32(0.5))
    assert single.dtype == np.float32
    out = place(np.zeros_like(f), dev)
    spne().gen_advection_flux_conservative_eno3_pyst_kernel_3d(np.float32)(out, place(f, dev), place(u, dev), 0.5)
    assert rel_l2(to_host(out), exact) < rel_l2(single, exact)


@pytest.mark.parametrize("ncomp", [1, 3])
@pytest.mark.parametrize("real_t,wide", [(np.float32, np.float64), (np.float64, np.longdouble)], ids=["f32", "f64"])
def test_diffusion_of_the_transport_step_rounds_once(dev, real_t, wide, ncomp):
    """At rest the transport step is phi + p lap(phi), one fused multiply-add a cell: on integers
    the Laplacian is exact, and so are the product and the sum in the wider type."""
    from sopht_amd import _lib as L

    shape = (9, 12, 37)
    p = real_t(0.1)
    phi = np.random.default_rng(31).integers(-8, 9, (ncomp, *shape)).astype(real_t)
    a = phi.astype(wide)
    ref = a.copy()
    c = a[:, 1:-1, 1:-1, 1:-1]
    lap = (a[:, 2:, 1:-1, 1:-1] + a[:, :-2, 1:-1, 1:-1] + a[:, 1:-1, 2:, 1:-1] + a[:, 1:-1, :-2, 1:-1]
           + a[:, 1:-1, 1:-1, 2:] + a[:, 1:-1, 1:-1, :-2] - 6 * c)
    ref[:, 1:-1, 1:-1, 1:-1] = c + wide(p) * lap
    t = to_dev(phi, dev)
    scratch, u = to_dev(np.zeros_like(phi), dev), to_dev(np.zeros((3, *shape), dtype=real_t), dev)

    def ptrs(v):
        return L._p3(*([x.data_ptr() for x in v] + [0] * (3 - len(v))))

    L.call("sopht_passive_transport_step_3d", L.dtype_tag(real_t), ncomp, ptrs(t), ptrs(scratch), ptrs(u), *shape, 0.5,
           float(p), L.stream_ptr())
    np.testing.assert_array_equal(to_host(t), ref.astype(real_t))
