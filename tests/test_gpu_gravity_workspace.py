"""The workspace that the direct-force paths of one simulation share (gravity.hip):
the pair-symmetric path between calls of the one-sided path, which writes its
partial sums over the same memory.  Every call gives the bits of a fresh simulation."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bodies(n):
    rng = np.random.default_rng(n)
    st = np.zeros((n, 11))
    st[:, :3] = rng.normal(size=(n, 3)) * [1.0, 2.0, 0.5]
    st[:, 9] = rng.uniform(0.1, 2.0, n) / n
    return st


def _free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    hip = ctypes.CDLL("libamdhip64.so", mode=ctypes.RTLD_GLOBAL)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


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


@pytest.mark.parametrize("n,mode", [(110000, "compensated"), (153001, "fp64")])
def test_large_sums_in_bounded_memory(gpu, n, mode):
    """Beyond 512 MB of partial sums the tasks run in several launches: the
    tolerance of test_gpu_direct_split.py on sampled rows, against sums in extended
    precision (a sequential FP64 sum over this many bodies is itself off by
    sqrt(n) 2^-53 = 4e-14 of its terms); momentum; and device memory of the 512 MB, 48
    doubles per body and the allocator's rounding."""
    st = _bodies(n)
    sim = _sim(gpu, st, mode)
    sim.s.N_active = 64                                 # the body arrays first
    sim.update_acceleration()
    sim.s.N_active = gpu.SIZE_MAX
    free = _free_memory()
    acc = sim.update_acceleration()
    assert free - _free_memory() <= (512 << 20) + 384 * n + (4 << 20)
    for i in np.unique(np.concatenate([np.random.default_rng(1).integers(0, n, 64), [0, 1023, 1024, n - 2, n - 1]])):
        d = st[:, :3].astype(np.longdouble) - st[i, :3]
        r2 = (d * d).sum(1) + np.longdouble(0.01) ** 2
        terms = st[:, 9:10] * d / (r2 * np.sqrt(r2))[:, None]
        scale = np.sqrt((terms * terms).sum(1)).sum()
        assert np.sqrt(((acc[i] - terms.sum(0)) ** 2).sum()) <= 1e-14 * scale
    m = st[:, 9:10]
    assert np.abs((m * acc).sum(0)).max() <= 1e-13 * (m * np.abs(acc)).sum()
    sim.free()
