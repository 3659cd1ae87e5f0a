"""The workloads this repository's speed is measured on, through its public
entry points: leapfrog N-body simulations, direct forces on device arrays, the
WHFast integrator on one planetary system, batched ensembles and MEGNO maps,
and shearing sheets with tree gravity and collisions.

A case is a plain dict; `kind` selects the path and the other keys its size and
options.  Sizes are those of bench.py, of the tests, or lie between them:

  leapfrog   Plummer spheres of 64 .. 65536 bodies (bench.py: 1024 and 65536,
             its serving mix 256 .. 8192), every precision and gravity that
             the direct force has, alone or followed by the energy a user
             monitors
  direct     the force on device arrays a caller already holds, all bodies
             active or with test particles
  whfast     one simulation of a star and its planets through
             reb_simulation_integrate, as most programs use REBOUND
  ensemble   up to 16384 systems of 2 .. 8 planets (bench.py's ensemble), in
             both coordinate systems, with or without MEGNO
  sheet      planetary-ring patches of up to 200000 hard spheres (bench.py's
             sheet and smaller ones of the same optical depth)
"""
import ctypes
import math

import numpy as np
import torch

import rebound_amd as amd

F8 = torch.float64
STATE_COLS = 14                # doubles per struct reb_particle
AREA_PER_BODY = 1360.0 ** 2 / 200000   # box area per ring body of bench.py's sheet


def listed():
    return [
        # a small cluster: launches and transfers, not pairs, set its time (lower end of the serving mix)
        dict(name="leapfrog_256", kind="leapfrog", n=256, gravity="basic", precision="fp64", steps=100, energy=False),
        # the small benchmark configuration in the mode that reproduces REBOUND's bits
        dict(name="leapfrog_1024_exact", kind="leapfrog", n=1024, gravity="basic", precision="exact", steps=100,
             energy=False),
        # an ordinary cluster run of a ragged size, with the energy check a user makes between outputs
        dict(name="leapfrog_10007_energy", kind="leapfrog", n=10007, gravity="basic", precision="fp64", steps=20,
             energy=True),
        # compensated summation, chosen for long runs with small energy errors
        dict(name="leapfrog_24000_compensated", kind="leapfrog", n=24000, gravity="compensated", precision="fp64",
             steps=10, energy=False),
        # the headline configuration: the largest direct sum
        dict(name="leapfrog_65536", kind="leapfrog", n=65536, gravity="basic", precision="fp64", steps=10,
             energy=False),
        # a caller with its own device arrays: massive bodies and test particles, split precision
        dict(name="direct_30011_split", kind="direct", n=30011, n_active=20011, gravity="basic", precision="split"),
        # one solar-system-like simulation in REBOUND's default WHFast settings
        dict(name="whfast_8_planets", kind="whfast", planets=8, coordinates="jacobi", safe_mode=1, corrector=0,
             steps=400),
        # the ensemble benchmark
        dict(name="ensemble_16384_dh", kind="ensemble", systems=16384, kmin=2, kmax=8,
             coordinates="democraticheliocentric", safe_mode=0, megno=False, steps=1000),
        # an ensemble in the reference's default coordinates
        dict(name="ensemble_6000_jacobi", kind="ensemble", systems=6000, kmin=2, kmax=8, coordinates="jacobi",
             safe_mode=0, megno=False, steps=400),
        # the MEGNO-map benchmark
        dict(name="megno_16384", kind="ensemble", systems=16384, kmin=2, kmax=8, coordinates="jacobi", safe_mode=1,
             megno=True, steps=100),
        # the ring benchmark, and a small patch of it
        dict(name="sheet_200000", kind="sheet", n=200000, n_root=10, steps=2),
        dict(name="sheet_12007", kind="sheet", n=12007, n_root=4, steps=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["leapfrog", "leapfrog", "leapfrog", "direct", "whfast", "ensemble", "ensemble", "sheet"])
    if kind == "leapfrog":
        gravity, precision = rng.choice([("basic", "fp64"), ("basic", "fp64"), ("compensated", "fp64"),
                                         ("basic", "split"), ("basic", "exact")])
        n = _log_int(rng, 64, 65536 if precision != "exact" else 32768)
        most = 65536.0 ** 2 * 10 / (4 if precision == "exact" else 2)
        steps = max(1, min(rng.randint(20, 120), int(most / float(n) ** 2)))
        energy = precision != "exact" and rng.random() < 0.3
        return dict(kind=kind, n=n, gravity=gravity, precision=precision, steps=steps, energy=energy)
    if kind == "direct":
        gravity, precision = rng.choice([("basic", "fp64"), ("compensated", "fp64"), ("basic", "split")])
        n = _log_int(rng, 256, 65536)
        n_active = n if rng.random() < 0.5 else rng.randint(n // 4, n)
        return dict(kind=kind, n=n, n_active=n_active, gravity=gravity, precision=precision)
    if kind == "whfast":
        jac = rng.random() < 0.6
        return dict(kind=kind, planets=rng.randint(1, 12), coordinates="jacobi" if jac else "democraticheliocentric",
                    safe_mode=rng.randint(0, 1), corrector=rng.choice([0, 0, 11]) if jac else 0,
                    steps=rng.randint(100, 400))
    if kind == "ensemble":
        jac = rng.random() < 0.6
        megno = jac and rng.random() < 0.4
        systems = _log_int(rng, 100, 16384)
        kmin = rng.randint(1, 4)
        return dict(kind=kind, systems=systems, kmin=kmin, kmax=rng.randint(kmin, 8),
                    coordinates="jacobi" if jac else "democraticheliocentric",
                    safe_mode=1 if megno else rng.randint(0, 1), megno=megno,
                    steps=rng.randint(50, 100) if megno else rng.randint(100, 300))
    return dict(kind="sheet", n=_log_int(rng, 1500, 150000), n_root=rng.randint(2, 10), steps=1)


# ------------------------------------------------------------------ inputs
def _plummer(n, seed):
    """(n, 11) x y z vx vy vz ax ay az m r of an equal-mass Plummer sphere
    (Aarseth, Henon & Wielen 1974), total mass 1, at rest."""
    rng = np.random.default_rng(seed)
    r = 1.0 / np.sqrt(rng.uniform(1e-6, 0.999, n) ** (-2.0 / 3.0) - 1.0)
    q = np.empty(n)
    todo = np.arange(n)
    while todo.size:
        c, y = rng.uniform(0, 1, todo.size), rng.uniform(0, 0.1, todo.size)
        ok = y < c * c * (1 - c * c) ** 3.5
        q[todo[ok]] = c[ok]
        todo = todo[~ok]
    v = q * math.sqrt(2.0) * (1 + r * r) ** -0.25

    def on_sphere(length):
        z = rng.uniform(-1, 1, n)
        phi = rng.uniform(0, 2 * math.pi, n)
        s = np.sqrt(1 - z * z)
        return length[:, None] * np.stack([s * np.cos(phi), s * np.sin(phi), z], 1)

    st = np.zeros((n, 11))
    st[:, 0:3] = on_sphere(r)
    st[:, 3:6] = on_sphere(v)
    st[:, 0:6] -= st[:, 0:6].mean(0)
    st[:, 9] = 1.0 / n
    return st


def _softening(n):
    return 0.005 if n > 16384 else 0.02


def _planets(S, kmin, kmax, seed):
    """S systems of a star (m = 1) and K planets, K uniform in kmin .. kmax (the
    same K for every seed, so that results of two seeds have one shape): inner orbit a = 1, log-uniform period ratios in [1.5, 2.5] and masses in
    [1e-7, 1e-4], eccentricities and inclinations of a few hundredths, uniform
    angles, moved to the centre of mass.  Returns (K [S], bodies
    [S, kmax + 1, 7] x y z vx vy vz m, timestep [S] = inner period / 20).
    Rows after a system's last planet are massless bodies on far orbits."""
    rng = np.random.default_rng(seed)
    K = np.random.default_rng(0).integers(kmin, kmax + 1, S)
    ratio = np.exp(rng.uniform(math.log(1.5), math.log(2.5), (S, kmax)))
    ratio[:, 0] = 1.0
    a = np.cumprod(ratio, 1) ** (2.0 / 3.0)
    m = np.exp(rng.uniform(math.log(1e-7), math.log(1e-4), (S, kmax)))
    e = np.minimum(rng.rayleigh(0.02, (S, kmax)), 0.08)
    inc = rng.rayleigh(0.01, (S, kmax))
    Om, om, f = (rng.uniform(0, 2 * math.pi, (S, kmax)) for _ in range(3))
    off = np.arange(1, kmax + 1)[None, :] > K[:, None]
    m[off] = 0.0
    a = np.where(off, 1e3 * np.arange(1, kmax + 1)[None, :], a)
    mu = 1.0 + m
    r = a * (1 - e * e) / (1 + e * np.cos(f))
    v0 = np.sqrt(mu / a / (1 - e * e))
    cO, sO, co, so, cf, sf, ci, si = (g(w) for w in (Om, om, f, inc) for g in (np.cos, np.sin))
    b = np.zeros((S, kmax + 1, 7))
    b[:, 0, 6] = 1.0
    p = b[:, 1:]
    p[..., 0] = r * (cO * (co * cf - so * sf) - sO * (so * cf + co * sf) * ci)
    p[..., 1] = r * (sO * (co * cf - so * sf) + cO * (so * cf + co * sf) * ci)
    p[..., 2] = r * (so * cf + co * sf) * si
    p[..., 3] = v0 * ((e + cf) * (-ci * co * sO - cO * so) - sf * (co * cO - ci * so * sO))
    p[..., 4] = v0 * ((e + cf) * (ci * co * cO - sO * so) - sf * (co * sO + ci * so * cO))
    p[..., 5] = v0 * ((e + cf) * co * si - sf * si * so)
    p[..., 6] = m
    b[..., 0:6] -= ((b[..., 6:7] * b[..., 0:6]).sum(1) / b[..., 6:7].sum(1))[:, None, :]
    return K, b, 2 * math.pi / np.sqrt(1.0 + m[:, 0]) / 20.0


def _used(K, kmax):
    return np.arange(kmax + 1)[None, :] <= K[:, None]


def _rows(K, b):
    """The used rows as (bodies, 11)."""
    flat = b[_used(K, b.shape[1] - 1)]
    st = np.zeros((flat.shape[0], 11))
    st[:, 0:6] = flat[:, 0:6]
    st[:, 9] = flat[:, 6]
    return st


def _deviations(nrow, seed):
    """Initial variational particles (x y z vx vy vz ax ay az m)."""
    v = np.zeros((nrow, 10))
    v[:, 0:6] = np.random.default_rng(seed + 1).normal(0, 1, (nrow, 6)) * 1e-8
    return v


def _cube(sim):
    """The bodies of a simulation as an (N, 14) view of doubles."""
    return sim.particles().view("f8").reshape(-1, STATE_COLS)


def _sim_of(st):
    """A simulation holding the bodies `st`."""
    sim = amd.Sim()
    sim.add_plummer(st.shape[0])          # allocates; every value is replaced
    _cube(sim)[:, :11] = st
    return sim


def _sheet(n, n_root, seed):
    """The ring patch of rebound_amd.shearing_sheet (bench.py's sheet), its
    bodies drawn with numpy."""
    size = math.sqrt(AREA_PER_BODY * n)
    rng = np.random.default_rng(seed)
    st = np.zeros((n, 11))
    st[:, 0:2] = rng.uniform(-size / 2, size / 2, (n, 2))
    st[:, 2] = rng.normal(0, 1, n)
    st[:, 3:6] = rng.normal(0, 3.2, (n, 3)) * [1, 1, 0.5]
    st[:, 4] -= 1.5 * st[:, 0]
    u = rng.uniform(0, 1, n)
    radius = (u * (4.0 ** -2 - 1.0) + 1.0) ** -0.5      # dN/dR ~ R^-3 in [1, 4]
    st[:, 9] = 400.0 * 4.0 / 3.0 * math.pi * radius ** 3
    st[:, 10] = radius
    sim = _sim_of(st)
    s = sim.s
    s.rand_seed = seed % (1 << 31)
    s.OMEGA = 1.0
    s.G = 1.546 / 400.0
    s.softening = 0.1
    s.dt = 1e-3 * 2.0 * math.pi
    s.root_size = size / n_root
    s.N_root_x = s.N_root_y = n_root
    s.N_root_z = 1
    s.N_ghost_x = s.N_ghost_y = 2
    s.boundary = amd.BOUNDARY["shear"]
    s.gravity = amd.GRAVITY["tree"]
    s.opening_angle2 = 0.25
    sim.set_integrator("sei")
    amd.lib().reb_amd_set_coefficient_of_restitution(sim.ptr, 0.5)
    s.collision = amd.COLLISION["tree"]
    s.collision_resolve = ctypes.cast(amd.lib().reb_collision_resolve_hardsphere, type(s.collision_resolve))
    return sim


def prepare(case, seed):
    kind = case["kind"]
    if kind == "leapfrog":
        sim = _sim_of(_plummer(case["n"], seed))
        sim.set_integrator("leapfrog")
        sim.s.softening = _softening(case["n"])
        sim.s.dt = 5e-4
        sim.s.gravity = amd.GRAVITY[case["gravity"]]
        sim.precision = case["precision"]
        return {"case": case, "sim": sim}
    if kind == "direct":
        n = case["n"]
        st = torch.from_numpy(_plummer(n, seed)).cuda()
        cols = [st[:, k].contiguous() for k in (0, 1, 2, 9)]
        acc = [torch.zeros(n, dtype=F8, device="cuda") for _ in range(3)]
        L = amd.lib()
        ws = torch.empty(L.reb_amd_gravity_workspace_bytes(n, amd.PRECISION[case["precision"]]), dtype=torch.uint8,
                         device="cuda")
        return {"case": case, "cols": cols, "acc": acc, "ws": ws, "L": L}
    if kind == "whfast":
        K, b, dt = _planets(1, case["planets"], case["planets"], seed)
        sim = _sim_of(_rows(K, b))
        w = sim.set_integrator("whfast")
        w.coordinates = amd.WHFAST_COORDINATES[case["coordinates"]]
        w.safe_mode = case["safe_mode"]
        w.corrector = case["corrector"]
        sim.s.dt = float(dt[0])
        return {"case": case, "sim": sim}
    if kind == "ensemble":
        K, b, dt = _planets(case["systems"], case["kmin"], case["kmax"], seed)
        rows = _rows(K, b)
        ens = amd.Ensemble(K + 1, rows, dt, safe_mode=case["safe_mode"], coordinates=case["coordinates"])
        if case["megno"]:
            ens.init_megno(_deviations(rows.shape[0], seed))
        return {"case": case, "ens": ens}
    return {"case": case, "sim": _sheet(case["n"], case["n_root"], seed)}


# ------------------------------------------------------------------ one pass
def _whfast_tmax(t, case, dt):
    # output times are no multiple of the step: the last step is a shortened one
    return t + (case["steps"] - 0.5) * dt


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "direct":
        n, L = case["n"], state["L"]
        rc = L.reb_amd_gravity_direct(*[c.data_ptr() for c in state["cols"]], *[a.data_ptr() for a in state["acc"]], n,
                                      case["n_active"], 0, 0, 1.0, _softening(n), amd.PRECISION[case["precision"]],
                                      int(case["gravity"] == "compensated"), state["ws"].data_ptr(),
                                      torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError("reb_amd_gravity_direct: %d" % rc)
        return state["acc"]
    if kind == "ensemble":
        ens = state["ens"]
        ens.steps(case["steps"])
        st = ens.state()
        out = {"x": st[:, 0:3], "v": st[:, 3:6], "a": st[:, 6:9]}
        if case["megno"]:
            out["megno"], out["lyapunov"] = ens.megno()
            var = ens.var_state()
            out["dx"], out["dv"] = var[:, 0:3], var[:, 3:6]
        return out
    sim = state["sim"]
    out = {}
    if kind == "whfast":
        sim.integrate(_whfast_tmax(sim.s.t, case, sim.s.dt))
    else:
        sim.steps(case["steps"])
        if case.get("energy"):
            out["energy"] = sim.energy()
        if kind == "sheet":
            out["collisions"], out["pressure"] = int(sim.s.collisions_log_n), float(sim.s.collisions_plog)
    st = _cube(sim)[:, :9].copy()         # the simulation may be gone when the result is read
    out.update(x=st[:, 0:3], v=st[:, 3:6], a=st[:, 6:9])
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("leapfrog", "direct"):
        n = float(case["n"])
        na = float(case.get("n_active", n))
        # an unordered pair of massive bodies: 27 operations (the serial loop
        # of REBOUND's gravity.c:195-214); a test particle and a source: 20
        force = 27.0 * na * (na - 1) / 2 + 20.0 * (n - na) * na
        if kind == "direct":
            return {"bytes": 8.0 * 7 * n, "flops": force}
        energy = 11.0 * n * (n - 1) / 2 if case["energy"] else 0.0
        return {"bytes": 8.0 * 2 * 11 * n, "flops": force * case["steps"] + energy}
    if kind == "sheet":
        # a body sums about 115 cells or bodies for each of the 25 periodic
        # images at this opening angle, 20 operations each
        n = float(case["n"])
        return {"bytes": 8.0 * 2 * 11 * n, "flops": 20.0 * 115 * 25 * n * case["steps"]}
    if kind == "whfast":
        S, K = 1.0, float(case["planets"])
    else:
        S, K = float(case["systems"]), 0.5 * (case["kmin"] + case["kmax"])
    # Kepler solve, planet-planet terms and coordinate sums per planet
    per = 180.0 * K + 20.0 * K * (K - 1) + 30.0 * K
    if case.get("megno"):
        per *= 3.0
    return {"bytes": 8.0 * S * (K + 1) * 20, "flops": S * per * case["steps"]}


def tolerance(case):
    # Everything but the fast modes of the direct force reproduces REBOUND's
    # own order of operations bit for bit.
    if case["kind"] not in ("leapfrog", "direct") or case["precision"] == "exact":
        return "exact"
    # Split precision: r^-1 in FP32 (2^-23); its rounding differs from pair to
    # pair, so the sums agree to about 3e-8 (measured against exact()).
    if case["precision"] == "split":
        return {"rel": 1.2e-7, "max": 5e-6}
    # FP64 sums in another order: the sequential sums of the exact mode are
    # within 5e-15 of exact() up to 32768 bodies.
    return {"rel": 2e-14, "max": 2e-12}


# ------------------------------------------------------------------ plain 64-bit results
def _acc(x, m, soft2, na):
    """Accelerations of all bodies from the first `na` (test particles feel only)."""
    n = x.shape[0]
    out = torch.empty_like(x)
    rows = max(1, (1 << 24) // max(na, 1))
    for b in range(0, n, rows):
        d = [x[b:b + rows, k, None] - x[None, :na, k] for k in range(3)]
        r2 = d[0] * d[0]
        r2.add_(d[1] * d[1]).add_(d[2] * d[2]).add_(soft2)
        w = r2.sqrt_().pow_(3).reciprocal_().mul_(m[None, :na])
        for k in range(3):
            out[b:b + rows, k] = -(d[k].mul_(w)).sum(1)
    return out


def _energy(x, v, m):
    n = x.shape[0]
    e = 0.5 * (m * (v * v).sum(1)).sum()
    rows = max(1, (1 << 24) // n)
    for b in range(0, n, rows):
        d2 = torch.zeros(min(rows, n - b), n, dtype=F8, device=x.device)
        for k in range(3):
            d = x[b:b + rows, k, None] - x[None, :, k]
            d2.add_(d * d)
        d2[d2 == 0] = math.inf
        e = e - 0.5 * (m[b:b + rows, None] * m[None, :] / d2.sqrt_()).sum()
    return float(e)


def _kepler(q, v, mu, h):
    """Two-body motion over h on bound orbits (f and g functions, Newton's
    method on Kepler's equation in the eccentric-anomaly difference)."""
    r0 = (q * q).sum(-1).sqrt()
    a = 1.0 / (2.0 / r0 - (v * v).sum(-1) / mu)
    n = (mu / a ** 3).sqrt()
    ec = 1.0 - r0 / a
    es = (q * v).sum(-1) / (mu * a).sqrt()
    E = n * h
    for _ in range(8):
        s, c = E.sin(), E.cos()
        E = E - (E - ec * s + es * (1 - c) - n * h) / (1 - ec * c + es * s)
    s, c1 = E.sin(), 2 * (E / 2).sin() ** 2
    r = a * (1 - ec * (1 - c1) + es * s)
    f, g = 1 - a / r0 * c1, h - (E - s) / n
    fd, gd = -(mu * a).sqrt() / (r * r0) * s, 1 - a / r * c1
    return f[..., None] * q + g[..., None] * v, fd[..., None] * q + gd[..., None] * v


def _pairs(x, m, skip):
    """Accelerations between the bodies of each system; skip(i, j) leaves a pair out."""
    N = x.shape[1]
    keep = torch.tensor([[0.0 if i == j or skip(i, j) else 1.0 for j in range(N)] for i in range(N)], dtype=F8,
                        device=x.device)
    d = x[:, :, None, :] - x[:, None, :, :]
    r2 = (d * d).sum(-1) + (1 - keep)
    return -(d * (keep * m[:, None, :] / (r2 * r2.sqrt()))[..., None]).sum(2)


def _to_jacobi(x, m):
    out = [None] * x.shape[1]
    eta, s = m[:, 0:1], m[:, 0:1] * x[:, 0]
    for k in range(1, x.shape[1]):
        out[k] = x[:, k] - s / eta
        s, eta = s + m[:, k:k + 1] * x[:, k], eta + m[:, k:k + 1]
    out[0] = s / eta
    return torch.stack(out, 1)


def _from_jacobi(q, m):
    out = [None] * q.shape[1]
    com, eta = q[:, 0], m.sum(1, keepdim=True)
    for k in range(q.shape[1] - 1, 0, -1):
        com = com - m[:, k:k + 1] / eta * q[:, k]
        eta = eta - m[:, k:k + 1]
        out[k] = com + q[:, k]
    out[0] = com
    return torch.stack(out, 1)


def _wh_jacobi(x, v, m, h):
    """One Wisdom-Holman step in Jacobi coordinates: (x, v, accelerations of the kick)."""
    eta = m.cumsum(1)
    q, p = _to_jacobi(x, m), _to_jacobi(v, m)
    hh = 0.5 * h

    def drift(q, p):
        qk, pk = _kepler(q[:, 1:], p[:, 1:], eta[:, 1:], hh[:, None])
        return torch.cat([q[:, :1] + hh[:, None, None] * p[:, :1], qk], 1), torch.cat([p[:, :1], pk], 1)

    q, p = drift(q, p)
    acc = _pairs(_from_jacobi(q, m), m, lambda i, j: i + j == 1)
    k = _to_jacobi(acc, m)[:, 1:]
    far = q[:, 2:]
    r2 = (far * far).sum(-1, keepdim=True)
    k = torch.cat([k[:, :1], k[:, 1:] + eta[:, 2:, None] * far / (r2 * r2.sqrt())], 1)
    q, p = drift(q, torch.cat([p[:, :1], p[:, 1:] + h[:, None, None] * k], 1))
    return _from_jacobi(q, m), _from_jacobi(p, m), acc


def _wh_dh(x, v, m, h):
    """The same in democratic heliocentric coordinates."""
    M, m0 = m.sum(1)[:, None], m[:, 0:1]
    com, vcom = (m[..., None] * x).sum(1) / M, (m[..., None] * v).sum(1) / M
    q, p = x[:, 1:] - x[:, :1], v[:, 1:] - vcom[:, None]
    mp = m[:, 1:]
    hh = 0.5 * h[:, None]

    def jump(q, p):
        return q + hh[..., None] * ((mp[..., None] * p).sum(1) / m0)[:, None]

    q, p = _kepler(q, p, m0, hh)
    q = jump(q, p)
    acc = _pairs(q, mp, lambda i, j: False)
    p = p + h[:, None, None] * acc
    q = jump(q, p)
    q, p = _kepler(q, p, m0, hh)
    com = com + h[:, None] * vcom
    x0 = com - (mp[..., None] * q).sum(1) / M
    v0 = vcom - (mp[..., None] * p).sum(1) / m0
    return (torch.cat([x0[:, None], q + x0[:, None]], 1), torch.cat([v0[:, None], p + vcom[:, None]], 1),
            torch.cat([torch.zeros_like(acc[:, :1]), acc], 1))


def _exact_planets(case, seed):
    S = case.get("systems", 1)
    kmin, kmax = (case["planets"],) * 2 if case["kind"] == "whfast" else (case["kmin"], case["kmax"])
    K, b, dt = _planets(S, kmin, kmax, seed)
    used = _used(K, kmax)
    b = torch.from_numpy(b).cuda()
    x, v, m = b[..., 0:3], b[..., 3:6], b[..., 6]
    h = torch.from_numpy(np.broadcast_to(dt, (S,)).copy()).cuda()
    step = _wh_jacobi if case["coordinates"] == "jacobi" else _wh_dh
    if not case.get("megno"):
        for s in range(case["steps"]):
            last_half = case["kind"] == "whfast" and s == case["steps"] - 1
            x, v, a = step(x, v, m, 0.5 * h if last_half else h)
        out = {"x": x, "v": v, "a": a}
    else:
        d = np.zeros((S, kmax + 1, 6))
        d[used] = _deviations(int(used.sum()), seed)[:, 0:6]
        d = torch.from_numpy(d).cuda()
        dx, dv = d[..., 0:3], d[..., 3:6]
        live = torch.from_numpy(used).cuda()[..., None].double()
        Ys = Yss = var = cov = mt = mY = torch.zeros(S, dtype=F8, device="cuda")
        for s in range(case["steps"]):
            (x, v, a), (dx, dv, _) = torch.func.jvp(lambda X, V: step(X, V, m, h), (x, v), (dx, dv))
            dx, dv = dx * live, dv * live
            _, da = torch.func.jvp(lambda X: _pairs(X, m, lambda i, j: False), (x,), (dx,))
            t, n = h * (s + 1), s + 1.0
            dd = ((dx * dv + dv * da) * live).sum((1, 2)) / (dx * dx + dv * dv).sum((1, 2))
            Ys = Ys + 2 * h * t * dd
            Yss = Yss + Ys / t * h
            Y = Yss / t
            mt = mt + (t - mt) / n
            mY = mY + (Y - mY) / n
            cov = cov + (n - 1) / n * (t - mt) * (Y - mY)
            var = var + (n - 1) / n * (t - mt) ** 2
        out = {"x": x, "v": v, "a": a, "dx": dx, "dv": dv}
    used = torch.from_numpy(used).cuda()
    out = {k: w[used].cpu().numpy() for k, w in out.items()}
    if case.get("megno"):
        out["megno"], out["lyapunov"] = Y.cpu().numpy(), (cov / var).cpu().numpy()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "sheet":
        # the colliding pairs are resolved one after another in a random
        # order, each from the velocities the last one left: no formula
        return None
    if kind in ("whfast", "ensemble"):
        if case.get("corrector"):
            return None
        return _exact_planets(case, seed)
    n = case["n"]
    st = torch.from_numpy(_plummer(n, seed)).cuda()
    x, v, m = st[:, 0:3].clone(), st[:, 3:6].clone(), st[:, 9].contiguous()
    soft2 = _softening(n) ** 2
    if kind == "direct":
        return list(_acc(x, m, soft2, case["n_active"]).t().contiguous())
    h = 5e-4
    for _ in range(case["steps"]):
        x = x + 0.5 * h * v
        a = _acc(x, m, soft2, n)
        v = v + h * a
        x = x + 0.5 * h * v
    out = {"x": x.cpu().numpy(), "v": v.cpu().numpy(), "a": a.cpu().numpy()}
    if case["energy"]:
        out["energy"] = _energy(x, v, m)
    return out
