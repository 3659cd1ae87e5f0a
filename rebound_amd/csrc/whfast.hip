// WHFast on the GPU: the "whfast" integrator plugin of one simulation, the
// batched Kepler solver, the energies of many systems, and the launch that chooses
// between the lane kernels (whfast_lane.hip) and the general ones
// (whfast_general.hip).
//
// Reference: integrator_whfast.c:876-947 (init), :1051-1259 (synchronize, step),
// :241-427 (Kepler solver).
#include <cmath>
#include <cstring>

#include "internal.h"
#include "whfast_device.h"
#include "whfast_kepler.h"

namespace rbamd {

// ---------------------------------------------------------------- batch Kepler
__global__ void k_kepler_batch(double* __restrict__ s6, const double* __restrict__ mu,
                               const double* __restrict__ dt, int n, int* __restrict__ flags) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double* s = s6 + 6 * (size_t)i;
    double x = s[0], y = s[1], z = s[2], vx = s[3], vy = s[4], vz = s[5];
    const int f = kepler_solver(x, y, z, vx, vy, vz, mu[i], dt[i]);
    s[0] = x;
    s[1] = y;
    s[2] = z;
    s[3] = vx;
    s[4] = vy;
    s[5] = vz;
    if (f && flags) atomicOr(flags, f);
}

// Energy of each system in the reference's order (tools.c:108-162):
// kinetic over bodies, then potential over pairs (i<j), one thread per system.
__global__ void k_system_energy(WHParams P, double* __restrict__ out, int nsys) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsys) return;
    const WHSys S = P.sys[s];
    const size_t st = P.stride;
    const double* B = P.body;
    const int N = S.N;
    const int NA = S.Nact_grav;
    const int NI = S.tp_type == 0 ? NA : N;
    double e_kin = 0., e_pot = 0.;
    for (int i = 0; i < NI; i++) {
        const size_t b = (size_t)S.body0 + i;
        const double vx = B[3 * st + b], vy = B[4 * st + b], vz = B[5 * st + b], m = B[9 * st + b];
        e_kin += 0.5 * m * (vx * vx + vy * vy + vz * vz);
    }
    for (int i = 0; i < NA; i++) {
        const size_t bi = (size_t)S.body0 + i;
        for (int j = i + 1; j < NI; j++) {
            const size_t bj = (size_t)S.body0 + j;
            const double dx = B[bi] - B[bj];
            const double dy = B[st + bi] - B[st + bj];
            const double dz = B[2 * st + bi] - B[2 * st + bj];
            e_pot -= S.G * B[9 * st + bj] * B[9 * st + bi] / sqrt(dx * dx + dy * dy + dz * dz);
        }
    }
    out[s] = e_kin + e_pot;
}

__global__ void k_reset_counter(unsigned int* c) { *c = 0u; }

int whfast_launch(const WHParams& P, hipStream_t st) {
    hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(1), 0, st, P.counter);
    if (whfast_lane_takes(P))
        whfast_lane_launch(P, st);
    else
        whfast_general_launch(P, st);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int whfast_energy_launch(const WHParams& P, double* out, int nsys, hipStream_t st) {
    hipLaunchKernelGGL(k_system_energy, dim3((nsys + 63) / 64), dim3(64), 0, st, P, out, nsys);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// Lanes per system with K planets: one per planet, so a wavefront packs
// floor(64 / K) systems of one planet count.
int whfast_group_size(int K) { return K < 1 ? 1 : (K > 64 ? 64 : K); }

// Persistent workgroups (one wavefront each) that fit on the device at once.
int whfast_max_resident(int device) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1)
        cus = 256;
    return whfast_lane_per_cu() * cus;
}

// ---------------------------------------------------------------- per-simulation plugin
struct WHFastDevice {
    DevBuf ph;       // 7 * cap doubles (p_h SoA, same stride as the particle block)
    DevBuf meta;     // WHSys, WHTask, order, flags, counter
    DevBuf var;      // variational sets: pv and jv (10 * N_var doubles each), set offsets, MEGNO value
    size_t cap = 0;
};

void whfast_release(struct reb_simulation* r) {
    DeviceState* d = dev_of(r);
    if (d->whfast) {
        d->whfast->ph.release();
        d->whfast->meta.release();
        d->whfast->var.release();
        delete d->whfast;
        d->whfast = nullptr;
    }
}

// integrator_whfast.c:876-947, restricted to what this engine implements.
static bool whfast_check(struct reb_simulation* r, struct reb_integrator_whfast_state* s) {
    if (r->N_var) {
        // integrator_whfast.c:877-910
        if (s->coordinates != REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI) {
            reb_simulation_error(r, "Variational particles are only compatible with Jacobi coordinates.");
            return false;
        }
        if (s->kernel != REB_INTEGRATOR_WHFAST_KERNEL_DEFAULT) {
            reb_simulation_error(r, "Variational particles are only compatible with the standard kernel.");
            return false;
        }
        if (s->corrector2) {
            reb_simulation_error(r, "Variational particles not compatible with 2nd corrector.");
            return false;
        }
        if (s->safe_mode == 0 && r->calculate_megno) {
            reb_simulation_error(r, "MEGNO is not compatible with WHFast's safe_mode=0.");
            return false;
        }
        if (s->N_allocated_var != r->N_var) {
            s->p_jh_var = (struct reb_particle*)realloc(s->p_jh_var, sizeof(struct reb_particle) * r->N_var);
            for (size_t i = s->N_allocated_var; i < r->N_var; i++) memset(&s->p_jh_var[i], 0, sizeof(struct reb_particle));
            s->N_allocated_var = r->N_var;
        }
        for (size_t v = 0; v < r->N_var_config; v++) {
            const struct reb_variational_configuration& vc = r->var_config[v];
            if (vc.order != 1) {
                reb_simulation_error(r, "WHFast only supports first order variational equations.");
                return false;
            }
            if (vc.testparticle >= 0) {
                reb_simulation_error(r, "Test particle variations not supported with WHFast. Use IAS15.");
                return false;
            }
            // the kernel reads entries index .. index + N - 1 of the set
            if (vc.index < 0 || (size_t)vc.index + r->N > r->N_var) {
                reb_simulation_error(r, "A set of variational particles does not match the number of bodies.");
                return false;
            }
        }
        // simulation.c:673-682: variational accelerations of BASIC gravity only
        if (r->gravity != REB_GRAVITY_BASIC) {
            reb_simulation_error(r, "Variational gravity calculation not implemented in selected gravity module. Please use REB_GRAVITY_BASIC.");
            return false;
        }
    }
    if (s->coordinates != REB_INTEGRATOR_WHFAST_COORDINATES_DEMOCRATICHELIOCENTRIC &&
        s->coordinates != REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI) {
        reb_simulation_error(r, "This engine implements WHFast in Jacobi and democratic heliocentric coordinates.");
        return false;
    }
    if (s->kernel != REB_INTEGRATOR_WHFAST_KERNEL_DEFAULT && s->coordinates != REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI) {
        reb_simulation_error(r, "Non-standard kernel requires Jacobi coordinates.");
        return false;
    }
    if (s->kernel > 3) {
        reb_simulation_error(r, "Kernel method must be 0 (default), 1 (exact modified kick), 2 (composition kernel), or 3 (lazy implementer's modified kick). ");
        return false;
    }
    if (s->corrector != 0 && s->coordinates != REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI) {
        reb_simulation_error(r, "Symplectic correctors are only compatible with Jacobi and Barycentric coordinates.");
        return false;
    }
    if (s->corrector != 0 && s->corrector != 3 && s->corrector != 5 && s->corrector != 7 && s->corrector != 11 &&
        s->corrector != 17) {
        reb_simulation_error(r, "First symplectic correctors are only available in the following orders: 0, 3, 5, 7, 11, 17.");
        return false;
    }
    if (s->corrector2 != 0 && s->coordinates != REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI) {
        // the reference's second corrector runs the Jacobi operators whatever the coordinates
        reb_simulation_error(r, "The second symplectic corrector is supported with Jacobi coordinates only.");
        return false;
    }
    if (s->keep_unsynchronized == 1 && s->safe_mode == 1)
        reb_simulation_error(r, "whfast->keep_unsynchronized == 1 is not compatible with safe_mode. Must set whfast->safe_mode = 0.");
    if (s->keep_unsynchronized) {
        reb_simulation_error(r, "keep_unsynchronized is not supported by this engine.");
        return false;
    }
    const bool jac = s->coordinates == REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI;
    // integrator_whfast.c:929-939: the modified-kick and lazy kernels switch
    // the simulation to the Jacobi gravity
    if (s->kernel == 1 || s->kernel == 3) r->gravity = REB_GRAVITY_JACOBI;
    if (r->gravity != REB_GRAVITY_BASIC && r->gravity != REB_GRAVITY_COMPENSATED &&
        !(jac && r->gravity == REB_GRAVITY_JACOBI)) {
        reb_simulation_error(r, "WHFast on this engine evaluates the interaction with BASIC or COMPENSATED gravity "
                                "(or the Jacobi gravity in Jacobi coordinates).");
        return false;
    }
    if (r->additional_forces || dev_of(r)->dev_forces) {
        // the interaction runs inside the group kernel, which has no host callbacks
        reb_simulation_error(r, "additional_forces and device forces are not supported with WHFast on this engine.");
        return false;
    }
    if (r->N < 1) return false;
    if (r->N - 1 > 64) {
        reb_simulation_error(r, "WHFast on this engine handles up to 64 bodies besides the central one per simulation.");
        return false;
    }
    if (r->N_ghost_x || r->N_ghost_y || r->N_ghost_z) {
        reb_simulation_error(r, "Ghost boxes are not supported with WHFast.");
        return false;
    }
    if (s->kernel != 1 && s->kernel != 3)
        r->gravity_ignore_terms = jac ? REB_GRAVITY_IGNORE_TERMS_BETWEEN_0_AND_1 : REB_GRAVITY_IGNORE_TERMS_INVOLVING_0;
    if (s->N_allocated != r->N) {
        s->N_allocated = r->N;
        s->p_jh = (struct reb_particle*)realloc(s->p_jh, sizeof(struct reb_particle) * r->N);
        memset(s->p_jh, 0, sizeof(struct reb_particle) * r->N);
        r->did_modify_particles = 1;
    }
    return true;
}

static bool whfast_prepare(struct reb_simulation* r, WHParams& P) {
    DeviceState* d = dev_of(r);
    if (!ensure_device(r)) return false;
    if (!d->whfast) d->whfast = new WHFastDevice();
    WHFastDevice* w = d->whfast;
    if (w->cap != d->cap) {
        const bool fresh = w->cap == 0;
        if (!w->ph.ensure(sizeof(double) * 7 * d->cap)) return false;
        if (!RB_HIP(r, hipMemsetAsync(w->ph.p, 0, sizeof(double) * 7 * d->cap, d->stream))) return false;
        w->cap = d->cap;
        auto* s = (struct reb_integrator_whfast_state*)r->integrator.state;
        if (fresh && s && s->p_jh && s->N_allocated == r->N && r->N > 0 && !r->did_modify_particles) {
            // The integrator state holds p_jh of its own (a simulation read
            // from a binary file): continue from it, as the reference does.
            std::vector<double> h(7 * (size_t)r->N);
            for (size_t i = 0; i < r->N; i++) {
                const struct reb_particle& q = s->p_jh[i];
                const double f[7] = {q.x, q.y, q.z, q.vx, q.vy, q.vz, q.m};
                for (int k = 0; k < 7; k++) h[(size_t)k * r->N + i] = f[k];
            }
            for (int k = 0; k < 7; k++)
                if (!RB_HIP(r, hipMemcpyAsync(w->ph.as<double>() + (size_t)k * d->cap, h.data() + (size_t)k * r->N,
                                              sizeof(double) * r->N, hipMemcpyHostToDevice, d->stream)))
                    return false;
            if (!stream_sync(r)) return false;
        } else {
            r->did_modify_particles = 1;
        }
    }
    const size_t meta_bytes = sizeof(WHSys) + sizeof(WHTask) + 2 * sizeof(int) + 2 * sizeof(unsigned int) + 64;
    if (!w->meta.ensure(meta_bytes)) return false;
    char* base = w->meta.as<char>();
    WHSys sys;
    sys.body0 = 0;
    sys.N = (int)r->N;
    const size_t NA = (r->N_active == SIZE_MAX || r->testparticle_type == 1) ? r->N : r->N_active;
    sys.Nact = (int)NA;
    sys.Nact_grav = (int)((r->N_active == SIZE_MAX) ? r->N : r->N_active);
    sys.tp_type = r->testparticle_type;
    sys.steps = -1;
    sys.req = 0;
    sys.pad = 0;
    sys.G = r->G;
    sys.dt = r->dt;
    WHTask task{whfast_group_size((int)r->N - 1), 0, 1};
    struct Meta {
        WHSys sys;
        WHTask task;
        int order;
        unsigned int flags;
        unsigned int counter;
    } h;
    h.sys = sys;
    h.task = task;
    h.order = 0;
    h.flags = r->is_synchronized ? 1u : 0u;
    h.counter = 0;
    // Small, per-call metadata; the copy is ordered on the stream before the launch.
    static thread_local Meta staging;
    if (!stream_sync(r)) return false;
    staging = h;
    if (!RB_HIP(r, hipMemcpyAsync(base, &staging, sizeof(Meta), hipMemcpyHostToDevice, d->stream))) return false;
    Meta* dm = reinterpret_cast<Meta*>(base);
    P.sys = &dm->sys;
    P.tasks = &dm->task;
    P.order = &dm->order;
    P.flags = &dm->flags;
    P.counter = &dm->counter;
    P.ntasks = 1;
    P.grid = 1;
    P.body = d->soa.as<double>();
    P.ph = w->ph.as<double>();
    P.stride = d->cap;
    P.G = r->G;
    P.soft2 = r->softening * r->softening;
    P.compensated = r->gravity == REB_GRAVITY_COMPENSATED ? 1 : 0;
    P.all_active = sys.Nact == sys.N && sys.Nact_grav == sys.N;
    return true;
}

static bool whfast_finish(struct reb_simulation* r, struct reb_integrator_whfast_state* s, const WHParams& P) {
    DeviceState* d = dev_of(r);
    unsigned int flags = 0;
    if (!RB_HIP(r, hipMemcpyAsync(&flags, P.flags, sizeof(flags), hipMemcpyDeviceToHost, d->stream))) return false;
    if (!stream_sync(r)) return false;
    r->is_synchronized = flags & 1u;
    if ((flags & 2u) && !(r->messages_timestep_warning & 1)) {
        r->messages_timestep_warning |= 1;
        reb_simulation_warning(r, "Possible convergence issue. Timestep in Kepler solver is larger than one orbital period.");
    }
    if ((flags & 4u) && s->recalculate_coordinates_but_not_synchronized_warning == 0) {
        reb_simulation_warning(r, "Particles were modified while simulation was not synchronized.");
        s->recalculate_coordinates_but_not_synchronized_warning++;
    }
    mark_device_newer(r);
    return true;
}

// Refresh the public p_jh copy (heliocentric state) from the device.
static void whfast_mirror_pjh(struct reb_simulation* r, struct reb_integrator_whfast_state* s) {
    DeviceState* d = dev_of(r);
    if (!d->whfast || !s->p_jh || r->N == 0) return;
    std::vector<double> h(7 * r->N);
    for (int f = 0; f < 7; f++)
        (void)hipMemcpyAsync(h.data() + f * r->N, d->whfast->ph.as<double>() + (size_t)f * d->cap,
                             sizeof(double) * r->N, hipMemcpyDeviceToHost, d->stream);
    (void)hipStreamSynchronize(d->stream);
    for (size_t i = 0; i < r->N; i++) {
        s->p_jh[i].x = h[0 * r->N + i];
        s->p_jh[i].y = h[1 * r->N + i];
        s->p_jh[i].z = h[2 * r->N + i];
        s->p_jh[i].vx = h[3 * r->N + i];
        s->p_jh[i].vy = h[4 * r->N + i];
        s->p_jh[i].vz = h[5 * r->N + i];
        s->p_jh[i].m = h[6 * r->N + i];
    }
}

// The host copy of p_jh made current (before a binary snapshot is written).
void whfast_refresh_host(struct reb_simulation* r) {
    auto* s = (struct reb_integrator_whfast_state*)r->integrator.state;
    DeviceState* d = dev_of(r);
    if (!s || !d->whfast || !d->whfast->cap) return;
    whfast_mirror_pjh(r, s);
}

// The variational sets go to the device before each launch and come back
// after it (r->particles_var and the integrator's p_jh_var stay the host's:
// the sets are small and the plugin steps once per launch).  Layout: pv then
// jv, 10 fields of N_var doubles each (x y z vx vy vz ax ay az m), then the
// sets' offsets and the MEGNO value.
static bool var_upload(struct reb_simulation* r, struct reb_integrator_whfast_state* s, WHParams& P) {
    DeviceState* d = dev_of(r);
    WHFastDevice* w = d->whfast;
    const size_t nv = r->N_var;
    const size_t nd = 20 * nv + 1 + (r->N_var_config + 1) / 2;
    if (!w->var.ensure(sizeof(double) * nd)) {
        reb_simulation_error(r, "Out of device memory for the variational particles.");
        return false;
    }
    std::vector<double> h(nd, 0.);
    auto pack = [&](const struct reb_particle* q, double* o) {
        for (size_t i = 0; i < nv; i++) {
            const double f[10] = {q[i].x, q[i].y, q[i].z, q[i].vx, q[i].vy, q[i].vz, q[i].ax, q[i].ay, q[i].az, q[i].m};
            for (int k = 0; k < 10; k++) o[(size_t)k * nv + i] = f[k];
        }
    };
    pack(r->particles_var, h.data());
    pack(s->p_jh_var, h.data() + 10 * nv);
    int* vi = reinterpret_cast<int*>(h.data() + 20 * nv + 1);
    for (size_t v = 0; v < r->N_var_config; v++) vi[v] = r->var_config[v].index;
    if (!RB_HIP(r, hipMemcpyAsync(w->var.p, h.data(), sizeof(double) * nd, hipMemcpyHostToDevice, d->stream)))
        return false;
    double* base = w->var.as<double>();
    P.nvar = (int)r->N_var_config;
    P.var_index = reinterpret_cast<const int*>(base + 20 * nv + 1);
    P.pv = base;
    P.jv = base + 10 * nv;
    P.vstride = nv;
    P.megno = r->calculate_megno ? 1 : 0;
    P.megno_out = base + 20 * nv;
    return stream_sync(r);
}

static bool var_download(struct reb_simulation* r, struct reb_integrator_whfast_state* s, double* megno_dd) {
    DeviceState* d = dev_of(r);
    const size_t nv = r->N_var;
    std::vector<double> h(20 * nv + 1);
    if (!RB_HIP(r, hipMemcpyAsync(h.data(), d->whfast->var.p, sizeof(double) * h.size(), hipMemcpyDeviceToHost,
                                  d->stream)) ||
        !stream_sync(r))
        return false;
    auto unpack = [&](const double* o, struct reb_particle* q) {
        for (size_t i = 0; i < nv; i++) {
            q[i].x = o[0 * nv + i]; q[i].y = o[1 * nv + i]; q[i].z = o[2 * nv + i];
            q[i].vx = o[3 * nv + i]; q[i].vy = o[4 * nv + i]; q[i].vz = o[5 * nv + i];
            q[i].ax = o[6 * nv + i]; q[i].ay = o[7 * nv + i]; q[i].az = o[8 * nv + i];
            q[i].m = o[9 * nv + i];
        }
    };
    unpack(h.data(), r->particles_var);
    unpack(h.data() + 10 * nv, s->p_jh_var);
    *megno_dd = h[20 * nv];
    return true;
}

// n steps in one launch (n == 1 for the per-step plugin call).
bool whfast_run(struct reb_simulation* r, struct reb_integrator_whfast_state* s, long nsteps, int sync_at_end,
                double* megno_dd = nullptr) {
    if (!whfast_check(r, s)) return false;
    WHParams P;
    if (!whfast_prepare(r, P)) return false;
    if (r->N_var && !var_upload(r, s, P)) return false;
    P.nsteps = nsteps;
    P.safe_mode = s->safe_mode ? 1 : 0;
    P.did_modify = r->did_modify_particles ? 1 : 0;
    P.sync_at_end = sync_at_end;
    P.coords = s->coordinates == REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI ? WH_JACOBI : WH_DH;
    P.corrector = (int)s->corrector;
    P.corrector2 = s->corrector2 ? 1 : 0;
    P.kernel = (int)s->kernel;
    P.jacgrav = r->gravity == REB_GRAVITY_JACOBI ? 1 : 0;
    if (whfast_launch(P, dev_of(r)->stream)) return RB_HIP(r, hipGetLastError());
    if (!whfast_finish(r, s, P)) return false;
    double dd = 0.;
    if (r->N_var && !var_download(r, s, &dd)) return false;
    if (megno_dd) *megno_dd = dd;
    return true;
}

void whfast_step_device(struct reb_simulation* r, struct reb_integrator_whfast_state* s) {
    double dd = 0.;
    if (!whfast_run(r, s, 1, 0, &dd)) return;
    r->t += r->dt / 2.;
    r->t += r->dt / 2.;
    r->dt_last_done = r->dt;
    if (r->calculate_megno && r->N_var) {
        // integrator_whfast.c:1250-1258 (the device formed deltad/delta2);
        // the reference leaves gravity_ignore_terms at INVOLVING_0 afterwards
        r->gravity_ignore_terms = REB_GRAVITY_IGNORE_TERMS_INVOLVING_0;
        const double dY = r->dt * 2. * (r->t - r->megno_initial_t) * dd;
        megno_update(r, dY, r->dt);
    }
}

// Steps of one simulation that a launch may hold: about 20 ms of them and at most
// 1000, so that an interrupt or reb_simulation_stop is seen soon.  A step's time is
// its kicks (a plain step counts two, with its drifts and transforms) times one kick's,
// fitted to measured steps (us; 1, 8 and 64 planets): safe mode 4.2, 7.7, 38.8 (the
// fit 5.6, 9.8, 43); composition kernel 13, 26, 105 (17, 29, 130); corrector 17 in safe mode
// 175, 370, 1409 (185, 323, 1432); test particles 20, 28, 84 (21, 28, 84); lazy kernel 17,
// 101, 3981 (21, 84, 4116), with corrector 17 in safe mode 0.9, 3.7, 124 ms (0.7, 2.8, 136).
size_t whfast_launch_steps(const struct reb_simulation* r, const struct reb_integrator_whfast_state* s) {
    const double K = r->N > 1 ? (double)(r->N - 1) : 1.;
    const bool jacgrav = s->kernel == 1 || s->kernel == 3 || r->gravity == REB_GRAVITY_JACOBI;
    const bool all_active = r->N_active == SIZE_MAX || r->N_active == r->N;
    const double kick = jacgrav ? 10. + 0.5 * K * K : (all_active ? 2.5 + 0.3 * K : 10. + 0.5 * K);
    double kicks = s->kernel == 2 ? 6. : 2.;
    if (s->safe_mode) kicks += (s->corrector ? 4. * (s->corrector - 1.) : 0.) + (s->corrector2 ? 16. : 0.);
    const double n = 20e3 / (kicks * kick);
    return n < 1. ? 1 : (n > 1000. ? 1000 : (size_t)n);
}

// n steps without variational sets in one launch; the time advances as n calls of
// whfast_step_device would advance it.  False: nothing was done.
bool whfast_steps_device(struct reb_simulation* r, struct reb_integrator_whfast_state* s, long n) {
    if (!whfast_run(r, s, n, 0)) return false;
    for (long k = 0; k < n; k++) {
        r->t += r->dt / 2.;
        r->t += r->dt / 2.;
    }
    r->dt_last_done = r->dt;
    return true;
}

void whfast_synchronize_device(struct reb_simulation* r, struct reb_integrator_whfast_state* s) {
    if (r->is_synchronized) return;
    if (!whfast_run(r, s, 0, 1)) return;
    whfast_mirror_pjh(r, s);
}

}  // namespace rbamd

using namespace rbamd;

extern "C" {

void* rb_whfast_create(void) {
    auto* s = (struct reb_integrator_whfast_state*)calloc(1, sizeof(struct reb_integrator_whfast_state));
    s->coordinates = REB_INTEGRATOR_WHFAST_COORDINATES_JACOBI;
    s->safe_mode = 1;
    return s;
}

void rb_whfast_free(void* p) {
    auto* s = (struct reb_integrator_whfast_state*)p;
    free(s->p_jh);
    free(s->p_jh_var);
    free(s);
}

void rb_whfast_step(struct reb_simulation* r, void* state) {
    whfast_step_device(r, (struct reb_integrator_whfast_state*)state);
}

void rb_whfast_synchronize(struct reb_simulation* r, void* state) {
    auto* s = (struct reb_integrator_whfast_state*)state;
    if (!whfast_check(r, s)) return;
    whfast_synchronize_device(r, s);
}

REB_API int reb_amd_kepler_solver_batch(double* state6, const double* mu, const double* dt, size_t n) {
    if (n == 0) return 0;
    if (reb_amd_device_count() <= 0) {
        set_last_error("reb_amd_kepler_solver_batch: no HIP device");
        return 1;
    }
    double *d6 = nullptr, *dmu = nullptr, *ddt = nullptr;
    int* dflag = nullptr;
    int rc = 0;
    if (hipMalloc(&d6, sizeof(double) * 6 * n) != hipSuccess || hipMalloc(&dmu, sizeof(double) * n) != hipSuccess ||
        hipMalloc(&ddt, sizeof(double) * n) != hipSuccess || hipMalloc(&dflag, sizeof(int)) != hipSuccess) {
        rc = 2;
    } else {
        rc |= hipMemcpy(d6, state6, sizeof(double) * 6 * n, hipMemcpyHostToDevice) != hipSuccess;
        rc |= hipMemcpy(dmu, mu, sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess;
        rc |= hipMemcpy(ddt, dt, sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess;
        rc |= hipMemset(dflag, 0, sizeof(int)) != hipSuccess;
        hipLaunchKernelGGL(k_kepler_batch, dim3((n + 63) / 64), dim3(64), 0, 0, d6, dmu, ddt, (int)n, dflag);
        rc |= hipGetLastError() != hipSuccess;
        rc |= hipMemcpy(state6, d6, sizeof(double) * 6 * n, hipMemcpyDeviceToHost) != hipSuccess;
    }
    if (d6) (void)hipFree(d6);
    if (dmu) (void)hipFree(dmu);
    if (ddt) (void)hipFree(ddt);
    if (dflag) (void)hipFree(dflag);
    if (rc) set_last_error("reb_amd_kepler_solver_batch: HIP failure");
    return rc;
}

REB_API void reb_integrator_whfast_kepler_solver(struct reb_particle* const p, double mu, double dt,
                                                 const struct reb_simulation* const r) {
    double s[6] = {p->x, p->y, p->z, p->vx, p->vy, p->vz};
    if (reb_amd_kepler_solver_batch(s, &mu, &dt, 1)) {
        if (r) reb_simulation_error((struct reb_simulation*)r, "Kepler solver: no HIP device.");
        return;
    }
    p->x = s[0];
    p->y = s[1];
    p->z = s[2];
    p->vx = s[3];
    p->vy = s[4];
    p->vz = s[5];
}

}  // extern "C"
