"""The pair-symmetric direct force with its tasks cut into several workgroups
(gravity.hip, sym_split): body counts on both sides of a superblock boundary, with
one body or all but one in the last superblock, where the split changes.  Against
the oracle's per-target sums on sampled rows, the tolerances of
test_gpu_gravity.py: FP64 and COMPENSATED 1e-14 of sum_j |a_ij|, split precision 4e-7 of it (the
FP32 reciprocal square root cubed, one pair dominating)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bodies(n, seed):
    rng = np.random.default_rng(seed)
    st = np.zeros((n, 11))
    st[:, :3] = rng.normal(size=(n, 3)) * [1.0, 2.0, 0.5]
    st[:, 3:6] = rng.normal(size=(n, 3))
    st[:, 9] = rng.uniform(0.1, 2.0, n) / n
    return st


@pytest.mark.parametrize("n", [8193, 9215, 13312, 16385, 20480, 23000, 33793, 47104])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-14), ("compensated", 1e-14), ("split", 4e-7)])
def test_split_tasks(gpu, orc, n, precision, tol):
    st = _bodies(n, n)
    sim = gpu.Sim()
    sim.add_plummer(n)
    sim.particles().view("f8").reshape(n, 14)[:, :11] = st
    sim.s.softening = 0.01
    if precision == "compensated":
        sim.s.gravity = gpu.GRAVITY["compensated"]
    else:
        sim.precision = precision
    acc = sim.update_acceleration()
    rows = np.unique(np.concatenate([np.random.default_rng(1).integers(0, n, 96), [0, 1023, 1024, n - 2, n - 1]]))
    ref = orc.gravity_rows(st, rows, soft=0.01)
    scale = np.zeros(len(rows))
    for k, i in enumerate(rows):
        d = st[i, :3] - st[:, :3]
        r2 = (d * d).sum(1)
        scale[k] = (st[:, 9] * np.sqrt(r2) / (r2 + 1e-4) ** 1.5).sum()
    assert (np.sqrt(((acc[rows] - ref) ** 2).sum(1)) / scale).max() <= tol
    m = st[:, 9:10]
    assert np.abs((m * acc).sum(0)).max() <= (1e-6 if precision == "split" else 1e-13) * (m * np.abs(acc)).sum()
    sim.free()
