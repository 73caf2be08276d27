"""The three-pass Poisson schedule for x and y lengths that differ, and in FP64 (up to 384-point
x and y lines): every pair and every FP64 z length against the FP64 oracle, and the adding form
(the adjoint's solve) through a flow's adjoint step."""

import numpy as np
import pytest

from helpers import rel_l2, rel_linf, to_dev, to_host
from oracle import poisson as OP

pytestmark = pytest.mark.gpu

LENGTHS = (48, 64, 96, 128, 192, 256)


@pytest.mark.parametrize("real_t,ny,nx", [(np.float32, a, b) for a in LENGTHS for b in LENGTHS if a != b] +
                         [(np.float64, a, b) for a in LENGTHS[:-1] for b in LENGTHS[:-1]])
def test_lengths_match_oracle(dev, real_t, ny, nx):
    from sopht_amd.numeric.eulerian_grid_ops import UnboundedPoissonSolverPYFFTW3D

    nz = 4 if ny * nx > 20000 else 6
    shape = (nz, ny, nx)
    rng = np.random.default_rng(ny + nx)
    rhs = rng.standard_normal((3, *shape)).astype(real_t)
    s = UnboundedPoissonSolverPYFFTW3D(*shape, x_range=1.3, real_t=real_t)
    assert s.fft_schedule["passes"] == 3
    out = to_dev(np.zeros_like(rhs), dev)
    s.vector_field_solve(out, to_dev(rhs, dev))
    ref = np.zeros((3, *shape))
    OP.UnboundedPoissonSolver3D(*shape, x_range=1.3, real_t=np.float64).vector_field_solve(ref, rhs.astype(np.float64))
    # the bounds of the equal-length and the five-pass tests
    got = to_host(out)
    bound = 2e-5 if real_t is np.float32 else 1e-10
    assert rel_l2(got, ref) <= bound, rel_l2(got, ref)
    assert rel_linf(got, ref) <= 5 * bound, rel_linf(got, ref)


@pytest.mark.parametrize("nz", (8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256))
def test_fp64_z_lengths_match_oracle(dev, nz):
    from sopht_amd.numeric.eulerian_grid_ops import UnboundedPoissonSolverPYFFTW3D

    shape = (nz, 48, 64)
    rhs = np.random.default_rng(nz).standard_normal((3, *shape))
    s = UnboundedPoissonSolverPYFFTW3D(*shape, x_range=1.3, real_t=np.float64)
    assert s.fft_schedule["passes"] == 3
    out = to_dev(np.zeros_like(rhs), dev)
    s.vector_field_solve(out, to_dev(rhs, dev))
    ref = np.zeros((3, *shape))
    OP.UnboundedPoissonSolver3D(*shape, x_range=1.3, real_t=np.float64).vector_field_solve(ref, rhs)
    got = to_host(out)
    assert rel_l2(got, ref) <= 1e-10, rel_l2(got, ref)
    assert rel_linf(got, ref) <= 5e-10, rel_linf(got, ref)


def test_fp64_lines_of_512_points_take_five_passes(dev):
    from sopht_amd.numeric.eulerian_grid_ops import UnboundedPoissonSolverPYFFTW3D

    for ny, nx, passes in ((48, 256, 5), (256, 48, 5), (48, 48, 3)):
        assert UnboundedPoissonSolverPYFFTW3D(4, ny, nx, real_t=np.float64).fft_schedule["passes"] == passes


def test_unequal_lengths_add(dev):
    """The adding form of the last pass, through the adjoint step of a flow with unequal lengths:
    <A x, y> = <x, A^T y> for the linear velocity recovery without the free stream."""
    import torch

    from sopht_amd import simulator as sps

    shape = (24, 48, 96)
    kw = dict(kinematic_viscosity=1e-2, real_t=np.float32, with_forcing=True)
    flow = sps.UnboundedNavierStokesFlowSimulator3D(grid_size=shape, x_range=1.0, **kw)
    from sopht_amd import _lib as L

    assert L.schedule("sopht_ns3d_poisson_schedule", flow._plan)[0] == 3
    gen = torch.Generator(device=dev).manual_seed(5)
    w, ubar = (torch.randn((3, *shape), dtype=torch.float32, device=dev, generator=gen) for _ in range(2))
    u = torch.zeros_like(w)
    zero = torch.zeros_like(w)
    wo, uo = torch.empty_like(w), torch.empty_like(w)
    dt = 1e-3
    # from rest the step is linear in the vorticity up to its advection, which u = 0 leaves out
    flow.trajectory_step(w, u, zero, wo, uo, dt)
    lhs = float((uo.double() * ubar.double()).sum())
    wbar, ub, work = torch.zeros_like(w), ubar.clone(), torch.empty_like(w)
    L.call("sopht_ns3d_adjoint_step", flow._plan, L.ptr(w), L.ptr(u), dt, L.ptr(wbar), L.ptr(ub), L.ptr(work),
           L.stream_ptr())
    rhs = float((wbar.double() * w.double()).sum())
    scale = float(torch.linalg.vector_norm(uo.double()) * torch.linalg.vector_norm(ubar.double()))
    assert abs(lhs - rhs) <= 1e-4 * scale, (lhs, rhs, scale)
