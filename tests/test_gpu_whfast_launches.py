"""Several WHFast steps in one launch (driver.cpp): the same bodies, time, step
count and status as stepping one by one, which a heartbeat forces."""
import ctypes
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sim(gpu, coordinates, safe, corrector):
    rng = np.random.default_rng(4)
    st = np.zeros((5, 11))
    st[0, 9] = 1.0
    a = np.array([1.0, 1.7, 2.9, 5.1])
    th = rng.uniform(0, 6.28, 4)
    st[1:, 0], st[1:, 1], st[1:, 2] = a * np.cos(th), a * np.sin(th), 0.01 * a
    st[1:, 3], st[1:, 4] = -np.sin(th) / np.sqrt(a), np.cos(th) / np.sqrt(a)
    st[1:, 9] = 1e-5
    sim = gpu.Sim()
    sim.set_state(st)
    w = sim.set_integrator("whfast")
    w.coordinates = gpu.WHFAST_COORDINATES[coordinates]
    w.safe_mode = safe
    w.corrector = corrector
    sim.s.dt = 0.11
    return sim


def _snapshot(sim):
    s = sim.s
    return (sim.state()[:, :10], s.t, s.dt, s.dt_last_done, s.steps_done, s.is_synchronized, s.status,
            s.did_modify_particles)


@pytest.mark.parametrize("coordinates,safe,corrector", [("jacobi", 1, 0), ("jacobi", 0, 11),
                                                        ("democraticheliocentric", 0, 0)])
@pytest.mark.parametrize("exact", [0, 1])
def test_launches_equal_single_steps(gpu, coordinates, safe, corrector, exact):
    from rebound_amd import _abi
    got = []
    for single in (False, True):
        sim = _sim(gpu, coordinates, safe, corrector)
        sim.s.exact_finish_time = exact
        beat = _abi.HEARTBEAT(lambda r: None)
        if single:
            sim.s.heartbeat = beat
        snaps = []
        sim.steps(1)
        snaps.append(_snapshot(sim))
        sim.steps(2)
        snaps.append(_snapshot(sim))
        for tmax in (0.44, 13.7, 13.7, 140.05, 100.0):      # forward, no time, over 1000 steps, back
            sim.integrate(tmax)
            snaps.append(_snapshot(sim))
        sim.particles()["vx"][2] *= 1.0001                  # host edit between calls
        sim.s.did_modify_particles = 1
        sim.steps(1003)
        snaps.append(_snapshot(sim))
        got.append(snaps)
        sim.free()
    for a, b in zip(*got):
        assert np.array_equal(a[0], b[0]) and a[1:] == b[1:]


def test_refused_launch_counts_as_steps(gpu):
    sim = _sim(gpu, "jacobi", 1, 0)
    w = ctypes.cast(sim.s.integrator.state, ctypes.POINTER(gpu.WHFastState)).contents
    w.coordinates = gpu.WHFAST_COORDINATES["barycentric"]
    with pytest.raises(gpu.RebError):
        sim.steps(5)
    assert sim.s.steps_done == 5 and sim.s.t == 0.0
    sim.free()


def test_stop_is_seen_soon(gpu):
    """A launch holds about 20 ms of steps: with 64 planets, the lazy kernel and the
    17th-order corrector in safe mode a step takes 0.12 s, and a launch holds one."""
    st = np.zeros((65, 11))
    st[0, 9] = 1.0
    a, f = 1.0 + 0.2 * np.arange(64), 2.4 * np.arange(64)
    st[1:, 0], st[1:, 1] = a * np.cos(f), a * np.sin(f)
    st[1:, 3], st[1:, 4] = -np.sin(f) / np.sqrt(a), np.cos(f) / np.sqrt(a)
    st[1:, 9] = 1e-9
    sim = gpu.Sim()
    sim.set_state(st)
    w = sim.set_integrator("whfast")
    w.kernel, w.corrector, w.safe_mode = 3, 17, 1
    sim.s.dt = 0.05
    t = threading.Thread(target=lambda: sim.lib.reb_simulation_integrate(sim.ptr, float("inf")))
    t.start()
    t0 = time.time()
    while sim.s.steps_done < 2 and time.time() - t0 < 20:
        time.sleep(0.001)
    assert sim.s.steps_done >= 2
    sim.lib.reb_simulation_stop(sim.ptr)
    t.join(10)
    assert not t.is_alive() and sim.s.steps_done < 20
    sim.free()
