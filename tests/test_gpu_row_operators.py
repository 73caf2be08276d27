"""The row-vector operator kernels at the sizes where they can go wrong: rows shorter than a
wavefront and longer than a workgroup, row lengths that are no multiple of the vector width
(the last vector overlaps its neighbour), single chunks of planes and several, thin boxes.

Each operator runs twice on the same values: on dense fields (row-vector kernels) and on
fields whose cells are two apart along x (one thread per cell), and both are compared with the
oracle in double precision. The bound on an operator that sums ``m`` rounded products of
magnitude ``s`` is ``2 m eps s``: each product and each addition rounds once."""

import numpy as np
import pytest

from oracle import stencils as S

from helpers import to_dev, to_host

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 4), (4, 3, 5), (5, 6, 7), (9, 20, 37), (34, 5, 66), (7, 3, 1031), (40, 12, 256)]


@pytest.fixture(params=[np.float32, np.float64], ids=["f32", "f64"])
def real_t(request):
    return request.param


def spne():
    from sopht_amd.numeric import eulerian_grid_ops

    return eulerian_grid_ops


def spread_out(a, dev):
    """The array on the device with its cells two apart along x, among cells of 7."""
    big = np.full((*a.shape[:-1], 2 * a.shape[-1]), 7.0, dtype=a.dtype)
    big[..., ::2] = a
    return to_dev(big, dev)[..., ::2]


def both(run, outputs, inputs, dev, refs, bound):
    """``run(outputs, inputs)`` on dense and on spread-out fields against ``refs``."""
    for place in (lambda a: to_dev(a, dev), lambda a: spread_out(a, dev)):
        outs = [place(a) for a in outputs]
        run(outs, [place(a) for a in inputs])
        for o, r in zip(outs, refs):
            np.testing.assert_allclose(to_host(o), r, atol=bound, rtol=0)


@pytest.mark.parametrize("shape", SHAPES)
def test_stretching_steps(dev, real_t, shape):
    rng = np.random.default_rng(11)
    w = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    u = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    one = np.ones_like(w)
    p = real_t(0.3)
    w64, u64 = w.astype(np.float64), u.astype(np.float64)
    eps = float(np.finfo(real_t).eps)
    # a stage adds p (three products of 1 and a difference up to 2): at most 1.8 a stage, 9
    # roundings; three stages on values up to 1 + 1.8 + ... < 16
    flux = np.ones_like(w64)
    S.vorticity_stretching_flux(flux, w64, u64, float(p))
    kernel = spne().gen_vorticity_stretching_flux_pyst_kernel_3d(real_t)
    both(lambda o, i: kernel(o[0], i[0], i[1], p), [one], [w, u], dev, [flux], 2 * 9 * eps * 2)
    r, f = w64.copy(), np.zeros_like(w64)
    S.vorticity_stretching_timestep_euler_forward(r, u64, f, float(p))
    euler = spne().gen_vorticity_stretching_timestep_euler_forward_pyst_kernel_3d(real_t)
    both(lambda o, i: euler(o[0], i[0], o[1], p), [w, one], [u], dev, [r, f], 2 * 10 * eps * 3)
    r, f, m = w64.copy(), np.zeros_like(w64), np.zeros_like(w64)
    S.vorticity_stretching_timestep_ssprk3(r, u64, f, float(p), m)

    def ssprk3(o, i):
        spne().gen_vorticity_stretching_timestep_ssprk3_pyst_kernel_3d(real_t, o[2])(o[0], i[0], o[1], p)

    both(ssprk3, [w, one, one], [u], dev, [r, f, m], 2 * 30 * eps * 16)


def test_stretching_step_with_one_buffer_for_flux_and_midstep(dev, real_t):
    # the operands meet: the step runs as the reference's sequence of kernels
    rng = np.random.default_rng(12)
    shape = (6, 7, 9)
    w = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    u = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    w64, buf = w.astype(np.float64), np.zeros((3, *shape))

    def flux(v, p):
        S.vorticity_stretching_flux(buf, v.copy(), u.astype(np.float64), p)

    flux(w64, 0.25)
    buf += w64
    flux(buf, 0.25)
    buf += buf
    buf[...] = 0.75 * w64 + 0.25 * buf
    flux(buf, 0.125)
    buf += buf
    r = w64 / 3 + 2 * buf / 3
    wd, bd = to_dev(w, dev), to_dev(np.zeros_like(w), dev)
    spne().gen_vorticity_stretching_timestep_ssprk3_pyst_kernel_3d(real_t, bd)(wd, to_dev(u, dev), bd, real_t(0.25))
    bound = 2 * 30 * float(np.finfo(real_t).eps) * 16
    np.testing.assert_allclose(to_host(wd), r, atol=bound, rtol=0)
    np.testing.assert_allclose(to_host(bd), buf, atol=bound, rtol=0)


@pytest.mark.parametrize("shape", [(5, 5, 5), (6, 5, 6), (9, 7, 37), (36, 6, 66), (7, 5, 1031), (40, 12, 256)])
def test_eno3_flux_and_step(dev, real_t, shape):
    rng = np.random.default_rng(13)
    f = rng.uniform(-1, 1, shape).astype(real_t)
    u = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    one = np.ones_like(f)
    p = real_t(0.25)
    f64, u64 = f.astype(np.float64), u.astype(np.float64)
    # six faces of at most 4/3 each, four roundings a face and one an addition
    bound = 2 * 6 * 5 * float(np.finfo(real_t).eps) * 2
    ref = np.ones(shape)
    S.advection_flux_conservative_eno3(ref, f64, u64, float(p))
    kernel = spne().gen_advection_flux_conservative_eno3_pyst_kernel_3d(real_t)
    both(lambda o, i: kernel(o[0], i[0], i[1], p), [one], [f, u], dev, [ref], bound)
    flux = np.zeros(shape)
    S.advection_flux_conservative_eno3(flux, f64, u64, -float(p))
    step = spne().gen_advection_timestep_euler_forward_conservative_eno3_pyst_kernel_3d(real_t)
    both(lambda o, i: step(o[0], o[1], i[0], p), [f, one], [u], dev, [f64 + flux, flux], bound)
    w = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    fluxes = np.zeros((3, *shape))
    for c in range(3):
        S.advection_flux_conservative_eno3(fluxes[c], w[c].astype(np.float64), u64, -float(p))
    step3 = spne().gen_advection_timestep_euler_forward_conservative_eno3_pyst_kernel_3d(real_t, field_type="vector")
    both(lambda o, i: step3(o[0], o[1], i[0], p), [w, one], [u], dev, [w.astype(np.float64) + fluxes, fluxes[2]], bound)
    flux = spne().eno3_advection_flux(to_dev(f, dev), to_dev(u, dev), float(p))
    np.testing.assert_allclose(to_host(flux), ref - 1, atol=bound, rtol=0)


@pytest.mark.parametrize("shape", [(5, 5, 5), (6, 5, 6), (9, 7, 37), (36, 6, 66), (7, 5, 1031), (40, 12, 256)])
def test_eno3_adjoint(dev, real_t, shape):
    rng = np.random.default_rng(14)
    f = rng.uniform(-1, 1, shape).astype(real_t)
    u = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    a = rng.uniform(-1, 1, shape).astype(real_t)
    p = 0.25
    # four weighted differences of at most 2 along each axis, then three products: about
    # 12 roundings of values up to 3
    bound = 2 * 12 * float(np.finfo(real_t).eps) * 3
    fr, ur = np.zeros(shape), np.zeros((3, *shape))
    S.advection_flux_conservative_eno3_adjoint(fr, ur, *(x.astype(np.float64) for x in (a, f, u)), p)
    kernel = spne().gen_advection_flux_conservative_eno3_adjoint_kernel_3d(real_t)
    both(lambda o, i: kernel(o[0], o[1], i[0], i[1], i[2], p), [np.ones_like(f), np.ones_like(u)], [a, f, u], dev,
         [1 + fr, 1 + ur], bound)
    both(lambda o, i: kernel(None, o[0], i[0], i[1], i[2], p), [np.ones_like(u)], [a, f, u], dev, [1 + ur], bound)
    fd, ud = to_dev(f, dev).requires_grad_(), to_dev(u, dev).requires_grad_()
    flux = spne().eno3_advection_flux(fd, ud, p)
    flux.backward(to_dev(a, dev))
    np.testing.assert_allclose(to_host(fd.grad), fr, atol=bound, rtol=0)
    np.testing.assert_allclose(to_host(ud.grad), ur, atol=bound, rtol=0)
