"""The leapfrog's opening drift taken by the previous step's reduction (gravity.hip,
kick_store): the same bits as steps that a heartbeat keeps apart, at each kernel that
finishes the accelerations, and after an integration that stops or pauses between two
steps, where the drift is taken back."""
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sim(gpu, n, precision, gravity):
    rng = np.random.default_rng(n)
    st = np.zeros((n, 11))
    st[:, :3] = rng.normal(size=(n, 3))
    st[:, 3:6] = 0.3 * rng.normal(size=(n, 3))
    st[:, 9] = 1.0 / n
    sim = gpu.Sim()
    sim.set_state(st)
    sim.set_integrator("leapfrog")
    sim.s.gravity = gpu.GRAVITY[gravity]
    sim.precision = precision
    sim.s.softening = 0.05
    sim.s.dt = 0.01
    return sim


def _snapshot(sim):
    s = sim.s
    return sim.state()[:, :10], (s.t, s.dt, s.dt_last_done, s.steps_done, s.status)


@pytest.mark.parametrize("n,precision,gravity", [
    (1, "fp64", "basic"), (257, "fp64", "basic"), (300, "split", "basic"), (300, "fp64", "compensated"),
    (65, "exact", "basic"), (65, "exact", "compensated"), (8192, "fp64", "basic"), (8500, "fp64", "compensated")])
def test_drift_ahead_equals_single_steps(gpu, n, precision, gravity):
    from rebound_amd import _abi
    got = []
    for single in (False, True):
        sim = _sim(gpu, n, precision, gravity)
        beat = _abi.HEARTBEAT(lambda r: None)
        if single:
            sim.s.heartbeat = beat
        snaps = []
        sim.steps(4)
        snaps.append(_snapshot(sim))
        for exact, tmax in ((1, 0.085), (0, 0.123), (1, 0.123), (1, 0.05)):
            sim.s.exact_finish_time = exact
            sim.s.dt = abs(sim.s.dt) if tmax > sim.s.t else -abs(sim.s.dt)
            sim.integrate(tmax)
            snaps.append(_snapshot(sim))
        sim.particles()["vx"][0] *= 1.0001                  # host edit between calls
        sim.steps(1)
        sim.steps(3)
        snaps.append(_snapshot(sim))
        got.append(snaps)
        sim.free()
    for a, b in zip(*got):
        assert np.array_equal(a[0], b[0]) and a[1] == b[1]


@pytest.mark.parametrize("pause", [False, True])
def test_stop_between_steps(gpu, pause):
    sim = _sim(gpu, 200, "fp64", "basic")
    t = threading.Thread(target=lambda: sim.lib.reb_simulation_integrate(sim.ptr, float("inf")))
    t.start()
    while sim.s.steps_done < 5:
        time.sleep(0.001)
    if pause:
        sim.s.status = -3
        time.sleep(0.05)
        steps = sim.s.steps_done
        time.sleep(0.05)
        assert sim.s.steps_done == steps
    sim.lib.reb_simulation_stop(sim.ptr)
    t.join(30)
    assert not t.is_alive()
    ref = _sim(gpu, 200, "fp64", "basic")
    ref.steps(sim.s.steps_done)
    assert np.array_equal(sim.state()[:, :10], ref.state()[:, :10]) and sim.s.t == ref.s.t
    sim.free()
    ref.free()
