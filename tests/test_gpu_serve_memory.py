"""N-body jobs of the pair-symmetric force under a memory budget that holds them only
with less workspace than they take alone (serve.hip, nbody_memory): what is charged
is what is allocated, within the budget, and the result keeps its bits."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    hip = ctypes.CDLL("libamdhip64.so", mode=ctypes.RTLD_GLOBAL)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _bodies(n):
    rng = np.random.default_rng(n)
    st = np.zeros((n, 11))
    st[:, :3] = rng.normal(size=(n, 3))
    st[:, 3:6] = 0.3 * rng.normal(size=(n, 3))
    st[:, 9] = 1.0 / n
    return st


def _alone(gpu, st, precision, gravity, steps):
    sim = gpu.Sim()
    sim.set_state(st)
    sim.set_integrator("leapfrog")
    sim.s.softening, sim.s.dt = 0.05, 1e-3
    sim.s.gravity = gpu.GRAVITY[gravity]
    sim.precision = precision
    sim.steps(steps)
    out = sim.state()[:, :9]
    sim.free()
    return out


def _serve(gpu, st, precision, gravity, budget, steps):
    """The result, the charge, and the most device memory seen in use."""
    srv = gpu.Server(memory_budget=budget)
    before = _free_memory()
    jid = srv.submit_nbody(st, softening=0.05, dt=1e-3, steps=steps, precision=precision,
                           gravity=gravity)
    least = before
    while srv.status(jid) in ("pending", "running"):
        least = min(least, _free_memory())
        time.sleep(0.0005)
    assert srv.wait(jid, 120) == "done", srv.job_error(jid)
    got = srv.result(jid)[0][:, :9]
    charged = srv.stats()["peak_bytes"]
    srv.close()
    return got, charged, before - least


@pytest.mark.parametrize("n,precision,gravity,part_mb,same", [
    (8192, "fp64", "basic", 7.5, True),          # all tasks at once, without the drift taken ahead
    (24000, "fp64", "basic", 25.1, True),        # five launches
    (24001, "split", "basic", 16.4, True),       # one round of the chip a launch
    (24000, "fp64", "compensated", 24.0, True),
    (40000, "fp64", "compensated", 26.0, False)])  # only the one-sided force fits
def test_job_in_less_memory(gpu, n, precision, gravity, part_mb, same):
    st = _bodies(n)
    steps = 150
    cap = 1 << (n - 1).bit_length()
    state = 88 * cap + 16 * n + 4096
    want = _alone(gpu, st, precision, gravity, steps)
    _, whole, _ = _serve(gpu, st, precision, gravity, 0, steps)       # and loads every kernel
    budget = state + int(part_mb * 2**20)
    assert budget < whole
    got, charged, used = _serve(gpu, st, precision, gravity, budget, steps)
    assert charged <= budget
    # allocations in pages of 2 MB: the body arrays, the partial sums, the scratch
    assert charged - state // 2 <= used <= charged + (6 << 20)
    if same:
        assert np.array_equal(got, want)
    else:
        # another order of the sums: 1e-15 of an acceleration a step, over 150 steps
        assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()


def test_refused_without_room(gpu):
    st = _bodies(24000)
    srv = gpu.Server(memory_budget=88 * 32768 + 16 * 24000 + 4096 + (15 << 20))
    with pytest.raises(gpu.RebError, match="exceeds the memory budget"):
        srv.submit_nbody(st, softening=0.05, steps=1)
    with pytest.raises(gpu.RebError, match="exceeds the memory budget"):
        srv.submit_nbody(st, softening=0.05, steps=1, gravity="compensated")
    srv.close()
