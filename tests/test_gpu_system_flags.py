"""Status bits per system of an ensemble (reb_amd_ensemble_flags): planet counts
that do not divide the wavefront, so that systems lie side by side in it at odd
offsets.  Only the innermost planet of every third system moves more than an orbit per
step (bit 2); it is the system's last lane or its first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["first", "last"])
@pytest.mark.parametrize("planets", [1, 2, 3, 5, 6, 7, 8, 11, 33, 64])
@pytest.mark.parametrize("options", [
    dict(), dict(coordinates="jacobi"), dict(gravity="compensated"), dict(coordinates="jacobi", safe_mode=1),
    dict(coordinates="jacobi", corrector=11), dict(coordinates="jacobi", kernel=3)],
    ids=["dh", "jacobi", "comp", "safe", "corrector", "lazy"])
def test_long_step_flag_stays_with_its_system(gpu, planets, where, options):
    nsys = 2 * (64 // planets) + 3
    N = planets + 1
    st = np.zeros((nsys, N, 11))
    st[:, 0, 9] = 1.0
    a = 4.0 + np.arange(planets)
    f = 2.4 * np.arange(planets)
    for s in range(nsys):
        r = a.copy()
        if s % 3 == 1:
            r[0 if where == "first" else -1] = 0.05     # period 0.07
        v = np.sqrt(1.0 / r)
        st[s, 1:, 0], st[s, 1:, 1] = r * np.cos(f), r * np.sin(f)
        st[s, 1:, 3], st[s, 1:, 4] = -v * np.sin(f), v * np.cos(f)
        st[s, 1:, 9] = 1e-9
    ens = gpu.Ensemble([N] * nsys, st.reshape(-1, 11), 0.2, **options)
    want = np.array([s % 3 == 1 for s in range(nsys)])
    for _ in range(2):                                  # the second launch starts from the first one's bits
        ens.steps(3)
        assert np.array_equal((ens.flags() & 2) != 0, want)
    ens.free()
