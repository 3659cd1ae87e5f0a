"""The workspace that the direct-force paths of one simulation share (gravity.hip):
the pair-symmetric path between calls of the one-sided path, which writes its
partial sums over the same memory.  Every call gives the bits of a fresh simulation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bodies(n):
    rng = np.random.default_rng(n)
    st = np.zeros((n, 11))
    st[:, :3] = rng.normal(size=(n, 3)) * [1.0, 2.0, 0.5]
    st[:, 9] = rng.uniform(0.1, 2.0, n) / n
    return st


def _sim(gpu, st, mode):
    sim = gpu.Sim()
    sim.add_plummer(len(st))
    sim.particles().view("f8").reshape(len(st), 14)[:, :11] = st
    sim.s.softening = 0.01
    if mode == "compensated":
        sim.s.gravity = gpu.GRAVITY["compensated"]
    else:
        sim.precision = mode
    return sim


@pytest.mark.parametrize("mode", ["fp64", "compensated", "split"])
@pytest.mark.parametrize("n", [8192, 10007, 16384])
def test_alternating_paths(gpu, n, mode):
    st = _bodies(n)
    active = [n // 2, gpu.SIZE_MAX]
    want = []
    for na in active:
        fresh = _sim(gpu, st, mode)
        fresh.s.N_active = na
        want.append(fresh.update_acceleration())
        fresh.free()
    sim = _sim(gpu, st, mode)
    for k in (0, 1, 0, 1, 1, 0, 1):
        sim.s.N_active = active[k]
        assert np.array_equal(sim.update_acceleration(), want[k]), k
    # ignored terms take the one-sided path as well
    sim.s.gravity_ignore_terms = 1
    sim.update_acceleration()
    sim.s.gravity_ignore_terms = 0
    assert np.array_equal(sim.update_acceleration(), want[1])
    sim.free()
