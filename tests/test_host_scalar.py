"""The velocity maximum that a kernel stores into pinned memory and the host reads: looked at for a
short while, then waited for with a synchronisation; a value that never comes is an error, and a
copied simulator reads a word of its own."""

import copy
import time

import numpy as np
import pytest

from sopht_amd import _lib as L


class Queue:
    """Stands for the stream: its synchronisation lets the pending store arrive."""

    def __init__(self, scalar, value):
        self.scalar, self.value, self.waits = scalar, value, 0

    def synchronize(self):
        self.waits += 1
        if self.value is not None:
            self.scalar._view[()] = self.value


def on_the_host(monkeypatch, value):
    """A scalar in ordinary memory, and the queue that its value arrives through."""
    import torch

    s = L.HostScalar(torch.float64, pinned=False)
    q = Queue(s, value)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: q)
    return s, q


def test_a_value_that_is_there_is_not_waited_for(monkeypatch):
    s, q = on_the_host(monkeypatch, None)
    s.arm()
    for v in (0.0, 2.5, np.nan):
        s._view[()] = v
        np.testing.assert_equal(float(s.read()), v)
    assert q.waits == 0


def test_a_late_value_is_waited_for(monkeypatch):
    s, q = on_the_host(monkeypatch, 1.25)
    s.arm()
    start = time.perf_counter()
    assert s.read() == 1.25
    assert q.waits == 1
    assert time.perf_counter() - start < 0.05  # looks for 2 ms; the rest is for a busy machine


def test_a_value_that_never_comes_raises(monkeypatch):
    s, q = on_the_host(monkeypatch, None)
    s.arm()
    with pytest.raises(RuntimeError, match="has not run"):
        s.read()
    assert q.waits == 1


def test_waiting_leaves_the_interpreter_to_other_threads(monkeypatch):
    import threading

    s, q = on_the_host(monkeypatch, 3.0)
    monkeypatch.setattr(L.HostScalar, "_LOOK_S", 0.2)
    s.arm()

    def store():
        time.sleep(0.01)
        s._view[()] = 1.5

    other = threading.Thread(target=store)
    other.start()  # its store ends the look
    assert s.read() == 1.5
    other.join()
    assert q.waits == 0


def flow(real_t=np.float32, n=32):
    import torch

    from sopht_amd import simulator as sps

    f = sps.UnboundedNavierStokesFlowSimulator3D(grid_size=(n, n, n), x_range=1.0, kinematic_viscosity=1e-3,
                                                 real_t=real_t)
    gen = torch.Generator(device="cuda").manual_seed(3)
    f.vorticity_field.normal_(generator=gen)
    f.velocity_field.normal_(generator=gen)
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("look", [0.0, 2e-3])
def test_time_step_limit_does_not_depend_on_how_it_is_read(dev, monkeypatch, look):
    import torch

    f = flow()
    expected = None
    monkeypatch.setattr(L.HostScalar, "_LOOK_S", look)
    side = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), side):
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            dt = f.compute_stable_timestep()
            u = f.velocity_field.double().abs().sum(0).max().item()
            assert dt == pytest.approx(f.compute_stable_timestep(), rel=0)
            assert f._max_out.read() == pytest.approx(u, rel=1e-6)
        expected = dt if expected is None else expected
        assert dt == expected


@pytest.mark.gpu
def test_maximum_follows_queued_steps(dev):
    import torch

    a, b = flow(np.float64), flow(np.float64)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for _ in range(20):  # more than the look lasts
        a.time_step(1e-3)
    expected = a.compute_stable_timestep()
    with torch.cuda.stream(side):
        for _ in range(20):
            b.time_step(1e-3)
        assert b.compute_stable_timestep() == expected
    torch.cuda.current_stream().wait_stream(side)


@pytest.mark.gpu
def test_copied_simulator_reads_its_own_word(dev):
    from sopht_amd import simulator as sps

    a = sps.PassiveTransportFlowSimulator(kinematic_viscosity=1e-3, grid_dim=3, grid_size=(16, 16, 16), x_range=1.0,
                                          field_type="scalar", real_t=np.float32)
    a.velocity_field.normal_()
    b = copy.deepcopy(a)
    assert b._vmax._t.is_pinned() and b._vmax._t.data_ptr() != a._vmax._t.data_ptr()
    assert a.compute_stable_timestep() == b.compute_stable_timestep()
    b.velocity_field.mul_(2)
    assert b.compute_stable_timestep() < a.compute_stable_timestep()
