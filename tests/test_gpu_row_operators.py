"""The row-vector operator kernels at the sizes where they can go wrong: rows shorter than a
wavefront and longer than a workgroup, row lengths that are no multiple of the vector width
(the last vector reads past the row's end), single chunks of planes and several, thin boxes.

Each operator runs on the same values in several layouts: dense fields, blocks inside larger
arrays, blocks that end where their array ends, and fields whose planes are the faster axis
(row-vector kernels; the pointwise operators take them cell by cell where they are not dense), and
fields whose cells are two apart along x (one thread per cell). What lies around a block is NaN, so
that a value read there and used would show, and must be as it was afterwards. Every result is
compared with the oracle in double precision. The bound on an operator that sums ``m`` rounded products of
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


def among(a, dev, front, back, planes_faster=False):
    """The array as a block on the device, `front` and `back` cells from the ends of each axis of a
    larger array (z, y, x) of NaN; optionally with the rows of a plane nz rows apart. Returns the
    larger array too."""
    b = np.swapaxes(a, -3, -2) if planes_faster else a
    big = np.full((*b.shape[:-3], *(n + f + k for n, f, k in zip(b.shape[-3:], front, back))), np.nan, dtype=a.dtype)
    cut = (..., *(slice(f, f + n) for n, f in zip(b.shape[-3:], front)))
    big[cut] = b
    t = to_dev(big, dev)
    view = t[cut]
    return (view.transpose(-3, -2) if planes_faster else view), t


LAYOUTS = {
    "dense": lambda a, dev: (to_dev(a, dev), None),
    "spread out": lambda a, dev: (spread_out(a, dev), None),
    "block": lambda a, dev: among(a, dev, (1, 2, 3), (1, 1, 2)),
    "block at the end": lambda a, dev: among(a, dev, (1, 1, 1), (0, 0, 0)),
    "planes faster": lambda a, dev: among(a, dev, (0, 0, 0), (0, 0, 0), True),
    "block, planes faster": lambda a, dev: among(a, dev, (2, 1, 1), (0, 0, 0), True),
}


def both(run, outputs, inputs, dev, refs, bound):
    """``run(outputs, inputs)`` in every layout against ``refs``."""
    for name, place in LAYOUTS.items():
        outs, arrays = zip(*(place(a, dev) for a in outputs))
        ins = [place(a, dev) for a in inputs]
        run(list(outs), [v for v, _ in ins])
        for o, t, r in zip(outs, arrays, refs):
            np.testing.assert_allclose(to_host(o), r, atol=bound, rtol=0, err_msg=name)
            if t is not None:  # around the block nothing was written
                o.fill_(float("nan"))
                assert t.isnan().all(), name


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


@pytest.mark.parametrize("shape", [(3, 3, 4), (9, 20, 37), (34, 5, 66)])
def test_stretching_flux_in_place_of_the_vorticity(dev, real_t, shape):
    # either kernel reads the vorticity at the cells it writes only
    rng = np.random.default_rng(18)
    w, u = rng.uniform(-1, 1, (2, 3, *shape)).astype(real_t)
    flux = np.zeros((3, *shape))
    S.vorticity_stretching_flux(flux, w.astype(np.float64), u.astype(np.float64), 0.25)
    kernel = spne().gen_vorticity_stretching_flux_pyst_kernel_3d(real_t)
    both(lambda o, i: kernel(o[0], o[0], i[0], 0.25), [w], [u], dev, [flux], 2 * 9 * float(np.finfo(real_t).eps) * 2)


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


@pytest.mark.parametrize("reset", [True, False])
@pytest.mark.parametrize("shape", SHAPES)
def test_curl_laplacian_divergence(dev, real_t, shape, reset):
    rng = np.random.default_rng(15)
    f = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    f64 = f.astype(np.float64)
    p = real_t(0.25)
    eps = float(np.finfo(real_t).eps)
    start = np.full_like(f, 0.5)
    ref = start.astype(np.float64)
    S.curl(ref, f64, 0.25, reset_ghost_zone=reset)
    curl = spne().gen_curl_pyst_kernel_3d(real_t, reset_ghost_zone=reset)
    both(lambda o, i: curl(o[0], i[0], p), [start], [f], dev, [ref], 2 * 4 * eps * 4)
    ref = start.astype(np.float64)
    S.update_vorticity_from_velocity_forcing(ref, f64, 0.25)
    update = spne().gen_update_vorticity_from_velocity_forcing_pyst_kernel_3d(real_t)
    both(lambda o, i: update(o[0], i[0], p), [start], [f], dev, [ref], 2 * 5 * eps * 4)
    ref = start.astype(np.float64)
    for c in range(3):
        S.diffusion_flux(ref[c], f64[c], 0.25, reset_ghost_zone=reset)
    flux = spne().gen_diffusion_flux_pyst_kernel_3d(real_t, field_type="vector", reset_ghost_zone=reset)
    both(lambda o, i: flux(o[0], i[0], p), [start], [f], dev, [ref], 2 * 8 * eps * 12)
    scalar = spne().gen_diffusion_flux_pyst_kernel_3d(real_t, reset_ghost_zone=reset)
    both(lambda o, i: scalar(o[0], i[0], p), [start[0]], [f[0]], dev, [ref[0]], 2 * 8 * eps * 12)
    ref = start[0].astype(np.float64)
    S.divergence(ref, f64, 0.25, reset_ghost_zone=reset)
    div = spne().gen_divergence_pyst_kernel_3d(real_t, reset_ghost_zone=reset)
    both(lambda o, i: div(o[0], i[0], p), [start[0]], [f], dev, [ref], 2 * 6 * eps * 6)


@pytest.mark.parametrize("shape", SHAPES + [(1, 1, 3), (2, 5, 9)])
def test_vector_forms_of_scalar_operators(dev, real_t, shape):
    rng = np.random.default_rng(16)
    a, b = (rng.uniform(-1, 1, (3, *shape)).astype(real_t) for _ in range(2))
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    eps = float(np.finfo(real_t).eps)
    one = np.ones_like(a)
    add = spne().gen_add_fixed_val_pyst_kernel_3d(real_t, field_type="vector")
    vals = (0.5, -0.25, 2.0)
    col = np.array(vals).reshape(3, 1, 1, 1)
    both(lambda o, i: add(o[0], i[0], vals), [one], [a], dev, [a64 + col], 2 * eps * 3)
    fix = spne().gen_set_fixed_val_pyst_kernel_3d(real_t, field_type="vector")
    both(lambda o, i: fix(o[0], vals), [one], [], dev, [one * col], 0.0)
    total = spne().gen_elementwise_sum_pyst_kernel_3d(real_t, field_type="vector")
    both(lambda o, i: total(o[0], o[0], i[0]), [a], [b], dev, [a64 + b64], 2 * eps * 2)
    saxpby = spne().gen_elementwise_saxpby_pyst_kernel_3d(real_t, field_type="vector")
    both(lambda o, i: saxpby(o[0], i[0], i[1], 0.75, 0.25), [one], [a, b], dev, [0.75 * a64 + 0.25 * b64], 2 * 3 * eps)
    cross = spne().gen_elementwise_cross_product_pyst_kernel_3d(real_t)
    both(lambda o, i: cross(o[0], i[0], i[1]), [one], [a, b], dev, [np.cross(a64, b64, axis=0)], 2 * 3 * eps * 2)
    step = spne().gen_diffusion_timestep_euler_forward_pyst_kernel_3d(real_t, field_type="vector")
    refs, flux = a64.copy(), np.zeros(shape)
    for c in range(3):
        S.diffusion_timestep_euler_forward(refs[c], flux, 0.125)
    both(lambda o, i: step(o[0], o[1], real_t(0.125)), [a, one[0]], [], dev, [refs, flux], 2 * 9 * eps * 12)
    # three tensors instead of one
    parts = [to_dev(a[c], dev) for c in range(3)]
    step(parts, to_dev(one[0], dev), real_t(0.125))
    for c in range(3):
        np.testing.assert_allclose(to_host(parts[c]), refs[c], atol=2 * 9 * eps * 12, rtol=0)


@pytest.mark.parametrize("width,shape", [(2, (4, 4, 4)), (2, (5, 9, 37)), (4, (8, 12, 9))])
def test_penalised_vector_equals_its_components(dev, real_t, width, shape):
    rng = np.random.default_rng(17)
    a = rng.uniform(-1, 1, (3, *shape)).astype(real_t)
    grid = np.meshgrid(*[(np.arange(n) + 0.5) * 0.1 for n in shape], indexing="ij")
    args = (width, 0.1, grid[2], grid[1], grid[0], real_t)
    whole, parts = to_dev(a, dev), to_dev(a, dev)
    spne().gen_penalise_field_boundary_pyst_kernel_3d(*args, field_type="vector")(whole)
    one = spne().gen_penalise_field_boundary_pyst_kernel_3d(*args)
    for c in range(3):
        one(parts[c])
    np.testing.assert_array_equal(to_host(whole), to_host(parts))
