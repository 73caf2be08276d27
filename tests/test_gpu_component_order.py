"""Vector operators on components that share memory: windows of one tensor a component apart, and
one component repeated by a zero stride. The reference loops over the components, so each sees what
the ones before it wrote; the same loop in numpy is the oracle. The fields are large enough for many
workgroups, and hold small integers with prefactors of powers of two, so every result is exact."""

import numpy as np
import pytest

from helpers import to_dev, to_host

pytestmark = pytest.mark.gpu

SHAPE = (12, 40, 66)


@pytest.fixture(params=[np.float32, np.float64], ids=["f32", "f64"])
def real_t(request):
    return request.param


def spne():
    from sopht_amd.numeric import eulerian_grid_ops

    return eulerian_grid_ops


def integers(seed, real_t, comps=4):
    return np.random.default_rng(seed).integers(-8, 9, (comps, *SHAPE)).astype(real_t)


WINDOWS = [(slice(0, 3), slice(1, 4)), (slice(1, 4), slice(0, 3))]


@pytest.mark.parametrize("out,src", WINDOWS)
def test_windows_of_one_tensor(dev, real_t, out, src):
    vals = (1.0, -2.0, 3.0)
    kernels = {
        "sum": (spne().gen_elementwise_sum_pyst_kernel_3d(real_t, field_type="vector"),
                lambda k, o, i: k(o, i, i), lambda c, i: i + i),
        "saxpby": (spne().gen_elementwise_saxpby_pyst_kernel_3d(real_t, field_type="vector"),
                   lambda k, o, i: k(o, i, o, 2.0, 0.5), None),
        "add_fixed": (spne().gen_add_fixed_val_pyst_kernel_3d(real_t, field_type="vector"),
                      lambda k, o, i: k(o, i, vals), lambda c, i: i + real_t(vals[c])),
    }
    for name, (kernel, call, one) in kernels.items():
        a = integers(3, real_t)
        t = to_dev(a, dev)
        call(kernel, t[out], t[src])
        o, i = a[out], a[src]
        for c in range(3):
            o[c] = one(c, i[c]) if one else 2 * i[c] + o[c] / 2
        np.testing.assert_array_equal(to_host(t), a, err_msg=name)


@pytest.mark.parametrize("reset", [True, False])
@pytest.mark.parametrize("out,src", WINDOWS)
def test_diffusion_flux_on_windows(dev, real_t, out, src, reset):
    a = integers(4, real_t)
    t = to_dev(a, dev)
    spne().gen_diffusion_flux_pyst_kernel_3d(real_t, field_type="vector", reset_ghost_zone=reset)(t[out], t[src], 0.5)
    o, i = a[out], a[src]
    for c in range(3):
        f = i[c].copy()
        lap = -6 * f[1:-1, 1:-1, 1:-1]
        for axis in range(3):
            for shift in (slice(2, None), slice(None, -2)):
                sl = [slice(1, -1)] * 3
                sl[axis] = shift
                lap = lap + f[tuple(sl)]
        if reset:
            o[c] = 0
        o[c][1:-1, 1:-1, 1:-1] = lap / 2
    np.testing.assert_array_equal(to_host(t), a)


def test_repeated_component(dev, real_t):
    add = spne().gen_elementwise_sum_pyst_kernel_3d(real_t, field_type="vector")
    a = integers(5, real_t, 3)
    t = to_dev(a, dev)
    add(t, t, t[0].expand(3, *SHAPE))
    for c in range(3):
        a[c] += a[0]
    np.testing.assert_array_equal(to_host(t), a)
    # one field as all three outputs: the last component's value stays
    one = to_dev(integers(6, real_t, 1), dev)
    spne().gen_set_fixed_val_pyst_kernel_3d(real_t, field_type="vector")(one[0].expand(3, *SHAPE), (1.0, 2.0, 4.0))
    assert (to_host(one) == 4).all()
    base = integers(7, real_t, 1)
    one = to_dev(base, dev)
    thrice = one[0].expand(3, *SHAPE)
    spne().gen_add_fixed_val_pyst_kernel_3d(real_t, field_type="vector")(thrice, thrice, (1.0, 2.0, 4.0))
    np.testing.assert_array_equal(to_host(one), base + 7)


def test_penalised_field_repeated(dev, real_t):
    base = integers(8, real_t, 1)
    grid = np.meshgrid(*[(np.arange(n) + 0.5) * 0.1 for n in SHAPE], indexing="ij")
    args = (2, 0.1, grid[2], grid[1], grid[0], real_t)
    whole, ref = to_dev(base, dev), to_dev(base, dev)
    spne().gen_penalise_field_boundary_pyst_kernel_3d(*args, field_type="vector")(whole[0].expand(3, *SHAPE))
    one = spne().gen_penalise_field_boundary_pyst_kernel_3d(*args)
    for _ in range(3):
        one(ref[0])
    np.testing.assert_array_equal(to_host(whole), to_host(ref))
