"""The one-lane-per-planet WHFast kernels (whfast_lane.hip) at the planet counts
where their unrolled loops and lane groups change shape: one planet, loop
remainders of one to three, a group of exactly half and of a whole wavefront,
and wavefronts with idle lanes, in both coordinate systems, with and without
safe mode and correctors.  Bitwise against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PLANETS = [1, 2, 3, 4, 5, 8, 9, 31, 32, 33, 63, 64]


def _system(amd, K, seed):
    """Star and K planets on nearly circular orbits, one of them planar (z = 0)."""
    rng = np.random.default_rng(seed)
    st = np.zeros((K + 1, 11))
    st[0, 9] = 1.0
    a = 1.45 ** np.arange(K) if K < 20 else 1.0 + 0.3 * np.arange(K)
    th = rng.uniform(0, 2 * np.pi, K)
    st[1:, 0], st[1:, 1] = a * np.cos(th), a * np.sin(th)
    st[1:, 2] = rng.normal(0, 0.01, K) * (np.arange(K) > 0)
    v = np.sqrt(1 / a) * rng.uniform(0.97, 1.03, K)
    st[1:, 3], st[1:, 4] = -v * np.sin(th), v * np.cos(th)
    st[1:, 9] = rng.uniform(1e-8, 1e-5, K)
    return st


@pytest.mark.parametrize("coordinates,safe,corrector",
                         [("democraticheliocentric", 0, 0), ("democraticheliocentric", 1, 0), ("jacobi", 0, 0),
                          ("jacobi", 1, 0), ("jacobi", 0, 7)])
def test_planet_counts_bitwise(gpu, orc, coordinates, safe, corrector):
    jac = coordinates == "jacobi"
    systems = [_system(gpu, K, 100 * K + s) for K in PLANETS for s in range(3)]
    nb = np.array([len(s) for s in systems])
    dt = 0.2 + 0.01 * np.arange(len(systems))
    ens = gpu.Ensemble(nb, np.concatenate(systems), dt, safe_mode=safe, coordinates=coordinates, corrector=corrector)
    ens.steps(7)
    ens.steps(4)
    st = ens.state()
    for q, init in enumerate(systems):
        s = init.copy()
        if jac:
            r = orc.whfast_jacobi(s, 1.0, dt[q], 7, safe, corrector=corrector)
        else:
            r = orc.whfast_dh(s, 1.0, dt[q], 7, safe)
        r = (orc.whfast_jacobi(r[0], 1.0, dt[q], 4, safe, corrector=corrector, pj=r[1], is_sync=1, did_modify=0)
             if jac else orc.whfast_dh(r[0], 1.0, dt[q], 4, safe, ph=r[1], is_sync=1, did_modify=0))
        got = ens.system(q, st)
        assert np.array_equal(got[:, :6], r[0][:, :6]), (len(init) - 1, q)
    ens.free()
