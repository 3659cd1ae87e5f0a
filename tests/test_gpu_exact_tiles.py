"""EXACT direct forces at the edges of the kernel's tiles (8 targets x 64 sources,
sources loaded two tiles ahead), with test particles of both types, ignored terms, and at scales
where the short square root and division give way to the compiler's.  Bitwise
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bodies(n, scale, seed):
    rng = np.random.default_rng(seed)
    st = np.zeros((n, 11))
    st[:, :3] = rng.normal(size=(n, 3)) * scale
    st[:, 9] = rng.uniform(0.5, 2.0, n)
    return st


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65, 127, 128, 129, 193, 260])
@pytest.mark.parametrize("gravity", ["basic", "compensated"])
@pytest.mark.parametrize("active,tp,ignore", [(1.0, 0, 0), (1.0, 0, 1), (1.0, 0, 2), (0.6, 0, 0), (0.6, 1, 0),
                                              (0.6, 1, 2)])
def test_tiles(gpu, orc, n, gravity, active, tp, ignore):
    for scale, soft in ((1.0, 0.01), (1.0, 0.0), (1e31, 0.0), (1e-31, 0.0)):
        st = _bodies(n, scale, n)
        NA = max(1, int(active * n))
        sim = gpu.Sim()
        sim.set_state(st)
        sim.s.softening = soft * scale
        sim.precision = "exact"
        sim.s.gravity = gpu.GRAVITY[gravity]
        if active < 1:
            sim.s.N_active = NA
            sim.s.testparticle_type = tp
        sim.s.gravity_ignore_terms = ignore
        acc = sim.update_acceleration()
        f = orc.gravity_basic if gravity == "basic" else orc.gravity_compensated
        ref = f(st, soft=soft * scale, N_active=NA if active < 1 else None, tp_type=tp if active < 1 else 0,
                ignore=ignore)
        assert np.array_equal(acc, ref), (scale, soft)
        sim.free()
