"""The parallel energy (gravity.hip, k_energy_tiles) at the edges of its 256-body
tiles, where workgroups take several tiles (from 129 tiles), with test particles,
and for bodies whose distances overflow or vanish.  Up to 700 bodies against sums in
extended precision: the terms are good to one rounding each and the sums are
compensated, which leaves the roundings of the kinetic and potential totals and
of their sum, 4 * 2^-53 of the larger one's magnitude.  Larger ones against the
oracle's sequential sum, whose own rounding is below n^2 2^-53 / 2, about sqrt of that
for random signs (1e-12 is used in test_gpu_gravity.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bodies(n, seed):
    rng = np.random.default_rng(seed)
    st = np.zeros((n, 11))
    st[:, :3] = rng.normal(size=(n, 3))
    st[:, 3:6] = rng.normal(size=(n, 3)) * 0.3
    st[:, 9] = rng.uniform(0.5, 2.0, n) / n
    return st


def _sim(gpu, st, N_active=None, tp=0):
    n = len(st)
    sim = gpu.Sim()
    sim.add_plummer(n)
    sim.particles().view("f8").reshape(n, 14)[:, :11] = st
    if N_active is not None:
        sim.s.N_active = N_active
        sim.s.testparticle_type = tp
    return sim


def _long(st, N_active, N_interact):
    x, v, m = (st[:, a].astype(np.longdouble) for a in (slice(0, 3), slice(3, 6), 9))
    kin = (0.5 * m * (v * v).sum(1))[:N_interact].sum()
    pot = np.longdouble(0)
    for i in range(N_active):
        d = x[i] - x[i + 1:N_interact]
        if len(d):
            pot -= (m[i] * m[i + 1:N_interact] / np.sqrt((d * d).sum(1))).sum()
    return kin, pot


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 511, 700])
@pytest.mark.parametrize("active,tp", [(1.0, 0), (0.6, 0), (0.6, 1)])
def test_tile_edges(gpu, n, active, tp):
    st = _bodies(n, n)
    NA = max(1, int(active * n))
    sim = _sim(gpu, st, NA if active < 1 else None, tp)
    kin, pot = _long(st, NA if active < 1 else n, n if (tp or active == 1) else NA)
    assert abs(sim.energy() - (kin + pot)) <= 4 * 2.0 ** -53 * max(kin, -pot)
    sim.free()


def test_several_tiles_per_workgroup(gpu, orc):
    st = _bodies(33100, 3)
    sim = _sim(gpu, st)
    e = orc.energy(st)
    assert abs(sim.energy() - e) <= 1e-12 * abs(e)
    sim.free()


def test_overflow_and_coincidence(gpu):
    st = _bodies(300, 5)
    st[7, 0] = 1e200                       # its pairs' r^2 overflow: no potential, as 1/inf
    st[7, 3:6] = 0.0
    keep = np.arange(300) != 7
    kin, pot = _long(st[keep], 299, 299)
    sim = _sim(gpu, st)
    assert abs(sim.energy() - (kin + pot)) <= 4 * 2.0 ** -53 * max(kin, -pot)
    sim.free()
    st[:, :3][8] = st[:, :3][9]            # coincident bodies: not finite
    sim = _sim(gpu, st)
    assert not np.isfinite(sim.energy())
    sim.free()


@pytest.mark.parametrize("n,i,j", [(2, 0, 1), (256, 254, 255), (257, 0, 256), (600, 3, 511), (600, 100, 101)])
def test_distance_below_the_normal_range(gpu, n, i, j):
    """A pair whose squared distance is subnormal, also as the last source of a tile:
    finite, with the value of FP64 arithmetic (the square keeps few bits, so the
    reference forms it the same way)."""
    st = _bodies(n, n)
    st[i, :3] = 0.0
    st[j, :3] = [1e-160, 0.0, 0.0]
    st[[i, j], 9] = 1e-78                          # the pair's term: about 1e4
    kin, pot = _long(np.delete(st, [i, j], 0), n - 2, n - 2)
    near = 1e-78 * 1e-78 / np.sqrt(1e-160 * 1e-160)
    sim = _sim(gpu, st)
    assert abs(sim.energy() - float(kin + pot) + near) <= 8 * 2.0 ** -53 * max(kin, -pot, near)
    sim.free()
