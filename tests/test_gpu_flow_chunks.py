"""The first sweep's choice of planes per work item: whatever the plan picks gives the same bits
as 16-plane scalar items, and the forcing it marks is zeroed everywhere, also where the second
sweep's items span several of the first one's."""

import numpy as np
import pytest

from helpers import PREC, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("shape,chunk", [((32, 32, 32), None), ((64, 64, 64), None), ((96, 96, 96), None),
                                         ((64, 64, 128), None), ((48, 96, 64), 2), ((64, 24, 96), 4),
                                         ((192, 128, 128), 2), ((24, 12, 6), None)])
def test_s1_items_give_the_same_bits(dev, shape, chunk, precision, rng, monkeypatch):
    import torch

    from sopht_amd import _lib as L
    from sopht_amd import simulator as sps

    real_t = PREC[precision]
    sims = []
    for scalar in (False, True):
        if scalar:
            monkeypatch.delenv("SOPHT_S1_CHUNK", raising=False)
            monkeypatch.setenv("SOPHT_S1_SCALAR", "1")
        elif chunk:
            monkeypatch.setenv("SOPHT_S1_CHUNK", str(chunk))
        sims.append(sps.UnboundedNavierStokesFlowSimulator3D(
            grid_size=shape, x_range=1.0, kinematic_viscosity=1e-2, real_t=real_t, with_forcing=True,
            with_free_stream_flow=True))
    monkeypatch.delenv("SOPHT_S1_SCALAR")
    if chunk:
        assert L.schedule("sopht_ns3d_s1_schedule", sims[0]._plan)[:2] == (1, chunk)
    w0, u0 = (rng.standard_normal((3, *shape)).astype(real_t) for _ in range(2))
    F0 = np.zeros((3, *shape), dtype=real_t)
    nz, ny, nx = shape
    F0[:, nz // 2 - 1, ny // 2, nx // 2] = 3.0  # one cell, in the middle of a run of planes
    F0[:, nz - 2, 1, 1] = -2.0
    for g in sims:
        g.vorticity_field.copy_(to_dev(w0, dev))
        g.velocity_field.copy_(to_dev(u0, dev))
        g.eul_grid_forcing_field.copy_(to_dev(F0, dev))
        g.time_step(dt=1e-2, free_stream_velocity=np.array([1.0, 0.5, -0.25]))
    for name in ("vorticity_field", "velocity_field", "stream_func_field"):
        assert torch.equal(getattr(sims[0], name), getattr(sims[1], name)), name
    for g in sims:
        assert np.all(to_host(g.eul_grid_forcing_field) == 0)
