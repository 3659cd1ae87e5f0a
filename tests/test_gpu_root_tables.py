"""The tree walks over the table of root boxes (tree.hip): root boxes that are
empty, hold one body (leaves) or few, 1 to 300 of them (the collision filter's table
holds 256), counts around the groups of four and 64, wavefronts of every width, and
operands outside the short square root's range.  Bitwise against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sim(gpu, st, root_size, nr, ghosts, theta2, soft):
    n = len(st)
    sim = gpu.Sim()
    sim.add_plummer(n)
    sim.particles().view("f8").reshape(n, 14)[:, :11] = st
    s = sim.s
    s.root_size = root_size
    s.N_root_x, s.N_root_y, s.N_root_z = nr
    s.boundary = gpu.BOUNDARY["periodic"]
    s.N_ghost_x, s.N_ghost_y = ghosts
    s.gravity = gpu.GRAVITY["tree"]
    s.opening_angle2 = theta2
    s.softening = soft
    s.G = 0.7
    return sim


def _bodies(n, box, seed, cluster=0.0):
    rng = np.random.default_rng(seed)
    st = np.zeros((n, 11))
    st[:, :3] = rng.uniform(-0.5, 0.5, (n, 3)) * box
    k = int(cluster * n)
    st[:k, :3] = st[0, :3] * 0.9 + rng.normal(0, 1e-3, (k, 3)) * np.min(box)
    st[:, 3:6] = rng.normal(size=(n, 3))
    st[:, 9] = rng.uniform(0.5, 2, n)
    st[:, 10] = rng.uniform(0.2, 1.0, n) * 0.25 * (np.prod(box) / n) ** (1 / 3)
    return st


def _offsets(box, ghosts):
    return np.array([[i * box[0], j * box[1], 0.0] for i in range(-ghosts[0], ghosts[0] + 1)
                     for j in range(-ghosts[1], ghosts[1] + 1)])


@pytest.mark.parametrize("nr,n,cluster", [((1, 1, 1), 5, 0), ((1, 1, 1), 3000, 0.3), ((2, 1, 1), 700, 0),
                                          ((5, 1, 1), 64, 0), ((8, 8, 1), 40, 0), ((13, 5, 1), 9000, 0.2),
                                          ((20, 15, 1), 2000, 0.5), ((3, 2, 2), 20000, 0)])
@pytest.mark.parametrize("scale,soft", [(1.0, 0.05), (1e35, 0.0), (1e-35, 0.0)])
def test_gravity(gpu, orc, nr, n, cluster, scale, soft):
    if n > 5000 and scale != 1.0:
        n = 5000
    box = np.array(nr) * 2.0 * scale
    st = _bodies(n, box, n, cluster)
    sim = _sim(gpu, st, 2.0 * scale, nr, (1, 1), 0.3, soft)
    acc = sim.update_acceleration()
    ref = orc.tree_gravity(st, 2.0 * scale, nr, 0.7, soft, 0.3, _offsets(box, (1, 1)))
    ref = ref[0] if isinstance(ref, tuple) else ref
    assert np.array_equal(acc, ref)
    sim.free()


@pytest.mark.parametrize("nr,n,cluster", [((1, 1, 1), 50, 0), ((5, 1, 1), 64, 0), ((8, 8, 1), 40, 0),
                                          ((13, 5, 1), 6000, 0.1), ((20, 15, 1), 2000, 0.2)])
@pytest.mark.parametrize("negative", [False, True])
def test_collisions(gpu, orc, nr, n, cluster, negative):
    box = np.array(nr) * 2.0
    st = _bodies(n, box, n + 1, cluster)
    if negative:
        st[::7, 10] *= -3.0                # the reference squares the summed reach
    sim = _sim(gpu, st, 2.0, nr, (1, 1), 0.3, 0.05)
    s = sim.s
    s.gravity = gpu.GRAVITY["none"]
    s.collision = gpu.COLLISION["tree"]
    found = []
    from rebound_amd import _abi
    keep = _abi.RESOLVE(lambda r, c: found.append((c.p1, c.p2)) or 0)
    s.collision_resolve = keep
    sim.set_integrator("leapfrog")
    s.dt = 0.0
    sim.steps(1)
    gb6 = np.hstack([_offsets(box, (1, 1)), np.zeros((9, 3))])
    ref = orc.collisions_tree(st, 2.0, nr, gb6)
    ref = ref[0] if isinstance(ref, tuple) else ref
    want = sorted((int(a), int(b)) for a, b in np.asarray(ref)[:, :2])
    assert sorted(found) == want
    sim.free()


def test_gravity_at_the_filling_cells(gpu, orc):
    """The records that fill the table to fours lie at (2^66, 0, 0): the image of a
    body at the origin of a box of that size is exactly there, without softening."""
    size, nr = 2.0 ** 60, (64, 1, 1)
    st = _bodies(200, np.full(3, 2.0 ** 55), 3)
    st[7, :3] = 0.0
    sim = _sim(gpu, st, size, nr, (1, 0), 1.5, 0.0)
    acc = sim.update_acceleration()
    ref, _ = orc.tree_gravity(st, size, nr, 0.7, 0.0, 1.5, _offsets((64 * size, size), (1, 0)))
    assert np.isfinite(ref).all() and np.array_equal(acc, ref)
    sim.free()


@pytest.mark.parametrize("theta2", [0.0, np.inf, np.nan])
@pytest.mark.parametrize("soft", [0.0, 0.05])
def test_gravity_angle_limits(gpu, orc, theta2, soft):
    """Opening angles for which theta^2 r^2 is infinite or no number, with root boxes of
    one body: the body itself stays left out, in every image."""
    nr = (6, 5, 1)
    box = np.array(nr) * 2.0
    st = _bodies(40, box, 5, 0.2)
    sim = _sim(gpu, st, 2.0, nr, (1, 1), theta2, soft)
    acc = sim.update_acceleration()
    ref, _ = orc.tree_gravity(st, 2.0, nr, 0.7, soft, theta2, _offsets(box, (1, 1)))
    assert np.isfinite(ref).all() and np.array_equal(acc, ref)
    sim.free()


@pytest.mark.parametrize("nr,n", [((32, 32, 1), 1500), ((33, 31, 1), 12000), ((128, 128, 1), 900),
                                  ((129, 128, 1), 900), ((1000, 1000, 1), 300), ((1, 20000, 1), 2)])
def test_large_root_grids(gpu, orc, nr, n):
    """Root grids of one and more batches of the compaction (1024 boxes), listed by box
    and (more boxes than bodies) by body; the device memory of a tree does not grow with
    empty boxes."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so", mode=ctypes.RTLD_GLOBAL)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_memory():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    box = np.array(nr) * 2.0
    st = _bodies(n, box, n)
    st[:, 10] *= 0.3
    sim = _sim(gpu, st, 2.0, nr, (1, 0), 0.4, 0.05)
    before = free_memory()
    acc = sim.update_acceleration()
    assert before - free_memory() <= (64 << 20)
    ref, _ = orc.tree_gravity(st, 2.0, nr, 0.7, 0.05, 0.4, _offsets(box, (1, 0)))
    assert np.array_equal(acc, ref)
    s = sim.s
    s.gravity = gpu.GRAVITY["none"]
    s.collision = gpu.COLLISION["tree"]
    found = []
    from rebound_amd import _abi
    keep = _abi.RESOLVE(lambda r, c: found.append((c.p1, c.p2)) or 0)
    s.collision_resolve = keep
    sim.set_integrator("leapfrog")
    s.dt = 0.0
    sim.steps(1)
    gb6 = np.hstack([_offsets(box, (1, 0)), np.zeros((3, 3))])
    ref = orc.collisions_tree(st, 2.0, nr, gb6)
    ref = ref[0] if isinstance(ref, tuple) else ref
    assert sorted(found) == sorted((int(a), int(b)) for a, b in np.asarray(ref)[:, :2])
    sim.free()
