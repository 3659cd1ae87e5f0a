// WHFast for systems whose bodies are all active: one lane per planet, the
// whole state of a system in its lanes' registers for all steps of a launch.
// Democratic heliocentric or Jacobi coordinates, the default and composition
// kernels, the symplectic correctors, BASIC or COMPENSATED gravity, and at most
// one first-order variational set (with or without MEGNO).  Test particles,
// the kernels with Jacobi gravity and several variational sets run in the
// general kernels of whfast_general.hip.
//
// Reference: integrator_whfast.c:392-490, 612-784, 1051-1259, gravity.c:215-343
// and :533-640, transformations.c:34-258 and :388-477, tools.c:1313-1380 and
// :1483-1522.  Every sum over bodies is formed by every lane of a group in the
// reference's index order from values its owners publish in LDS, with the
// reference's expressions (no contraction, IEEE sqrt and division), so the
// results are the reference's bits.
//
// What bounds it: with about one wavefront per SIMD (16384 systems are 1317
// wavefronts) the dependent chain of one step: the Kepler solve, the ordered
// scans of the transforms, the pair terms.  Hence
//  - the partial sums of the masses and their reciprocals, which the Jacobi
//    scans divide by, are constants of a launch: each lane forms its planet's
//    once and the scans multiply (a scan over 8 planets did 8 dependent
//    divisions);
//  - every drift of a step, a synchronization or a corrector runs through one
//    copy of the Kepler solver: the launch is a sequence of phases (drift, then
//    optionally a kick), so the loop fits the instruction cache and no state is
//    forced to memory by out-of-line copies (the general Jacobi instance is
//    1.1 MB of code, and its calls keep the lane's state in scratch);
//  - the pair loop runs over the other planets only (no per-pair self test), two
//    terms at a time.
// Measured against the general kernels, request and read-back of the state: 6000
// Jacobi systems of 2..8 planets, 400 steps, 14.66 -> 2.90 ms; 16384 MEGNO systems,
// 100 steps, 22.1 -> 7.5 ms; 16384 democratic heliocentric systems, 1000 steps,
// 10.5 -> 9.2 ms.
#include <cmath>
#include <type_traits>

#include "internal.h"
#include "whfast_device.h"
#include "whfast_kepler.h"

namespace rbamd {

namespace {

struct __align__(16) V4 {
    double x, y, z, w;
};
struct V3 {
    double x, y, z;
};
// A vector of a lane's state that few phases touch: in registers, or in the
// lane's column of an LDS array of three rows.
struct InRegisters {
    V3 v;
    __device__ __forceinline__ V3 get() const { return v; }
    __device__ __forceinline__ void set(const V3& q) { v = q; }
};
struct InLds {
    double (*p)[64];
    int lane;
    __device__ __forceinline__ V3 get() const { return V3{p[0][lane], p[1][lane], p[2][lane]}; }
    __device__ __forceinline__ void set(const V3& q) {
        p[0][lane] = q.x;
        p[1][lane] = q.y;
        p[2][lane] = q.z;
    }
};

__device__ __forceinline__ void kahan(double term, double& a, double& c) {
    const double yv = term - c;
    const double tv = a + yv;
    c = (tv - a) - yv;
    a = tv;
}

template <bool JAC, bool COMP, bool VAR, bool CHAIN>
__device__ __forceinline__ void lane_body(const WHParams& P) {
    static_assert(!VAR || (JAC && !COMP), "variational sets: Jacobi coordinates, BASIC gravity");
    static_assert(!CHAIN || JAC, "correctors and the composition kernel: Jacobi coordinates");
    __shared__ V4 ex[4][64];              // values the lanes publish
    __shared__ double2 fwd[64], bwd[64];  // mass scans of the Jacobi transforms (see scans())
    __shared__ double2 bwv[64];           // bwd of the variational set
    // The inertial velocities, which only synchronizations touch, and the MEGNO
    // sums wait in LDS: the registers of two wavefronts per SIMD hold the rest
    // without spills.
    __shared__ double cold[JAC ? (VAR ? 12 : 6) : 1][64];
    __shared__ double megno[VAR ? kMegnoFields : 1][64];
    __shared__ int task_id;
    const int lane = threadIdx.x;
    using Vel = std::conditional_t<JAC, InLds, InRegisters>;
    auto make_vel = [&](int row) {
        if constexpr (JAC)
            return InLds{cold + row, lane};
        else
            return InRegisters{V3{0, 0, 0}};
    };
    const size_t st = P.stride;
    for (;;) {
        if (lane == 0) task_id = (int)atomicAdd(P.counter, 1u);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(task_id);
        __syncthreads();
        if (t >= P.ntasks) break;
        const WHTask task = P.tasks[t];
        const int G = task.G;
        const int gl = lane % G;              // lane within the group
        const int ls = lane / G;              // system within the task
        const bool sys_ok = ls < task.nsys;
        // lanes without a system read the first group's slots and store nothing
        const int gbase = sys_ok ? lane - gl : 0;
        const int sidx = sys_ok ? P.order[task.sys0 + ls] : 0;
        const WHSys S = P.sys[sidx];
        // all systems of a task have one body count
        const int N = __builtin_amdgcn_readfirstlane(S.N);
        const int me = gl + 1;                // my body's index
        const bool live = sys_ok && me < N;
        const size_t b0 = (size_t)S.body0;
        const size_t bm = b0 + me;
        const double dt = S.dt, Gc = S.G;

        // ---- load
        V3 i{0, 0, 0}, a{0, 0, 0};                   // my planet, inertial
        V3 h{0, 0, 0}, hv{0, 0, 0};                  // my planet, heliocentric / Jacobi
        V3 s{0, 0, 0}, sa{0, 0, 0};                  // the star
        Vel iv = make_vel(0), sv = make_vel(3);      // their velocities
        V3 c{0, 0, 0}, cv{0, 0, 0};                  // p_jh[0] (barycentre)
        double im = 0, hm = 0, sm = 0, cm = 0;
        auto ld3 = [&](const double* base, size_t stride, int f, size_t k) {
            return V3{base[(size_t)f * stride + k], base[(size_t)(f + 1) * stride + k],
                      base[(size_t)(f + 2) * stride + k]};
        };
        auto st3 = [&](double* base, size_t stride, int f, size_t k, const V3& v) {
            base[(size_t)f * stride + k] = v.x;
            base[(size_t)(f + 1) * stride + k] = v.y;
            base[(size_t)(f + 2) * stride + k] = v.z;
        };
        if (sys_ok) {
            s = ld3(P.body, st, 0, b0);
            sv.set(ld3(P.body, st, 3, b0));
            if (JAC && !VAR) sa = ld3(P.body, st, 6, b0);
            sm = P.body[9 * st + b0];
            c = ld3(P.ph, st, 0, b0);
            cv = ld3(P.ph, st, 3, b0);
            cm = P.ph[6 * st + b0];
        }
        if (live) {
            i = ld3(P.body, st, 0, bm);
            iv.set(ld3(P.body, st, 3, bm));
            if (!VAR) a = ld3(P.body, st, 6, bm);
            im = P.body[9 * st + bm];
            h = ld3(P.ph, st, 0, bm);
            hv = ld3(P.ph, st, 3, bm);
            hm = JAC ? P.ph[6 * st + bm] : im;
        }
        const size_t vs = VAR ? P.vstride : 0;
        const size_t vb0 = VAR ? b0 + (size_t)P.var_index[0] : 0, vbm = vb0 + me;
        // variational set: my planet's, the star's and the barycentre's.  The
        // accelerations of a launch with one go to memory where they are formed.
        V3 di{0, 0, 0}, da{0, 0, 0}, ds{0, 0, 0}, dsa{0, 0, 0};
        V3 dh{0, 0, 0}, dhv{0, 0, 0}, dc{0, 0, 0}, dcv{0, 0, 0};
        double dm = 0, dsm = 0, dhm = 0, dcm = 0;
        Vel div = make_vel(VAR ? 6 : 0), dsv = make_vel(VAR ? 9 : 0);
        if (VAR && sys_ok) {
            ds = ld3(P.pv, vs, 0, vb0);
            dsv.set(ld3(P.pv, vs, 3, vb0));
            dsm = P.pv[9 * vs + vb0];
            dc = ld3(P.jv, vs, 0, vb0);
            dcv = ld3(P.jv, vs, 3, vb0);
            dcm = P.jv[9 * vs + vb0];
        }
        if (VAR && live) {
            di = ld3(P.pv, vs, 0, vbm);
            div.set(ld3(P.pv, vs, 3, vbm));
            dm = P.pv[9 * vs + vbm];
            dh = ld3(P.jv, vs, 0, vbm);
            dhv = ld3(P.jv, vs, 3, vbm);
            dhm = P.jv[9 * vs + vbm];
        }
        // MEGNO of the system (every lane of its group holds it)
        if (VAR && P.megno == 2 && sys_ok)
            for (int f = 0; f < kMegnoFields; f++) megno[f][lane] = P.megno_sys[(size_t)sidx * kMegnoFields + f];
        const unsigned int flags0 = sys_ok ? P.flags[sidx] : 1u;
        int sync = flags0 & 1u;
        int warn = (flags0 >> 1) & 15u;
        const long my_steps = !sys_ok ? 0 : (S.steps >= 0 && S.steps < P.nsteps ? (long)S.steps : P.nsteps);
        const bool safe = P.safe_mode || (sys_ok && (S.req & 4));

        // ------------------------------------------------ exchange through LDS
        auto publish = [&](int k, const V3& v, double w) { ex[k][lane] = V4{v.x, v.y, v.z, w}; };
        // f(k, its lane) for the group's planets k = 1 .. N-1 in order; the LDS
        // reads of four planets are issued together
        auto ascending = [&](auto&& f) {
            int k = 1, q = gbase;
            for (; k + 3 < N; k += 4, q += 4) {
                f(k, q);
                f(k + 1, q + 1);
                f(k + 2, q + 2);
                f(k + 3, q + 3);
            }
            if (k + 1 < N) {
                f(k, q);
                f(k + 1, q + 1);
                k += 2;
                q += 2;
            }
            if (k < N) f(k, q);
        };
        auto descending = [&](auto&& f) {
            int k = N - 1, q = gbase + N - 2;
            for (; k > 3; k -= 4, q -= 4) {
                f(k, q);
                f(k - 1, q - 1);
                f(k - 2, q - 2);
                f(k - 3, q - 3);
            }
            if (k > 1) {
                f(k, q);
                f(k - 1, q - 1);
                k -= 2;
                q -= 2;
            }
            if (k > 0) f(k, q);
        };

        // ------------------------------------------------ mass scans (Jacobi)
        // fwd[k] = {1/eta_{k-1}, eta_k/eta_{k-1} as eta_k * (1/eta_{k-1})} with
        // eta_k = m_0 + ... + m_k added in index order (transformations.c:34-81);
        // bwd[k] = {1/eta, eta - m_k} of the downward scan that starts from the
        // total mass of p_jh[0] (transformations.c:178-226).  The same values the
        // scans would form at every call: masses do not change in a launch.
        double eta_me = 0., eta_fwd_me = 0., eta_end = 0., eta_end_i = 0.;
        double cm_scan = 0., star_i = 0.;      // the downward scan's start and 1/(its end)
        double dcm_scan = 0., dstar_i = 0.;
        auto down_scan = [&](double top, double2* out, double& endi) {
            __syncthreads();
            publish(0, V3{0., 0., 0.}, im);
            __syncthreads();
            double e = top, eb = 0., ea = 0.;
            descending([&](int k, int q) {
                if (k == me) eb = e;
                e -= ex[0][q].w;
                if (k == me) ea = e;
            });
            out[lane] = make_double2(1. / eb, ea);
            endi = 1. / e;
            __syncthreads();
        };
        if (JAC) {
            // the Kepler and interaction masses start from p_jh's
            // (integrator_whfast.c:595-605, :446-451)
            publish(0, V3{0., 0., 0.}, hm);
            publish(1, V3{0., 0., 0.}, im);
            __syncthreads();
            double eh = sm, e = sm, eb = 0.;
            ascending([&](int k, int q) {
                if (k <= me) eh += ex[0][q].w;
                if (k == me) eb = e;
                e += ex[1][q].w;
                if (k == me) eta_fwd_me = e;
            });
            eta_me = eh;
            eta_end = e;
            eta_end_i = 1. / e;
            const double ei = 1. / eb;
            fwd[lane] = make_double2(ei, eta_fwd_me * ei);
            __syncthreads();
            cm_scan = cm;
            down_scan(cm, bwd, star_i);
            if (VAR) {
                dcm_scan = dcm;
                down_scan(dcm, bwv, dstar_i);
            }
        }

        // ------------------------------------------------ coordinate transforms
        // transformations.c:34-81 (Jacobi) of one set of vectors: X of the star and
        // x of the planets (published in row R) to mine, out, and the sum's
        // barycentre, com.
        auto scan_up = [&](int R, const V3& X, V3& out, V3* com) {
            V3 u{sm * X.x, sm * X.y, sm * X.z};
            ascending([&](int k, int q) {
                const V4 o = ex[R][q];
                const double2 f = fwd[q];
                const V3 j{o.x - u.x * f.x, o.y - u.y * f.x, o.z - u.z * f.x};
                if (k == me) out = j;
                u.x = u.x * f.y + o.w * j.x;
                u.y = u.y * f.y + o.w * j.y;
                u.z = u.z * f.y + o.w * j.z;
            });
            if (com) *com = V3{u.x * eta_end_i, u.y * eta_end_i, u.z * eta_end_i};
        };
        // transformations.c:178-258: the planets' Jacobi vectors (row R, masses in
        // .w) and the barycentre's to mine, out, and the star's.
        auto scan_down = [&](int R, const V3& C, double top, const double2* tab, double endi, V3& out, V3& star) {
            V3 u{C.x * top, C.y * top, C.z * top};
            descending([&](int k, int q) {
                const V4 o = ex[R][q];
                const double2 f = tab[q];
                u.x = (u.x - o.w * o.x) * f.x;
                u.y = (u.y - o.w * o.y) * f.x;
                u.z = (u.z - o.w * o.z) * f.x;
                if (k == me) out = V3{o.x + u.x, o.y + u.y, o.z + u.z};
                u.x *= f.y;
                u.y *= f.y;
                u.z *= f.y;
            });
            star = V3{u.x * endi, u.y * endi, u.z * endi};
        };
        auto from_inertial = [&](bool en) {
            __syncthreads();
            if constexpr (JAC) {
                publish(0, i, im);
                publish(1, iv.get(), im);
                if (VAR) {
                    publish(2, di, im);
                    publish(3, div.get(), im);
                }
                __syncthreads();
                V3 nh{0, 0, 0}, nhv{0, 0, 0}, nc, ncv;
                scan_up(0, s, nh, &nc);
                scan_up(1, sv.get(), nhv, &ncv);
                if (en) {
                    h = nh; hv = nhv; c = nc; cv = ncv;
                    cm = eta_end;
                    hm = im;
                    eta_me = eta_fwd_me;
                }
                if constexpr (VAR) {
                    V3 ndh{0, 0, 0}, ndhv{0, 0, 0}, ndc, ndcv;
                    scan_up(2, ds, ndh, &ndc);
                    scan_up(3, dsv.get(), ndhv, &ndcv);
                    if (en) {
                        dh = ndh; dhv = ndhv; dc = ndc; dcv = ndcv;
                        dhm = dm;
                        dcm = eta_end;
                    }
                }
            } else {
                // transformations.c:388-424
                publish(0, V3{i.x * im, i.y * im, i.z * im}, im);
                const V3 v = iv.get(), vstar = sv.get();
                publish(1, V3{v.x * im, v.y * im, v.z * im}, 0.);
                __syncthreads();
                V3 x0{0., 0., 0.}, v0{0., 0., 0.};
                double m0 = 0.;
                x0.x += s.x * sm; x0.y += s.y * sm; x0.z += s.z * sm;
                v0.x += vstar.x * sm; v0.y += vstar.y * sm; v0.z += vstar.z * sm;
                m0 += sm;
                ascending([&](int k, int q) {
                    const V4 o = ex[0][q], ov = ex[1][q];
                    x0.x += o.x; x0.y += o.y; x0.z += o.z;
                    v0.x += ov.x; v0.y += ov.y; v0.z += ov.z;
                    m0 += o.w;
                });
                if (en) {
                    c = V3{x0.x / m0, x0.y / m0, x0.z / m0};
                    cv = V3{v0.x / m0, v0.y / m0, v0.z / m0};
                    cm = m0;
                    h = V3{i.x - s.x, i.y - s.y, i.z - s.z};
                    hv = V3{v.x - cv.x, v.y - cv.y, v.z - cv.z};
                    hm = im;
                }
            }
        };
        // Positions of the systems with `en`, and velocities of those with `vel`
        // (transformations.c:178-258; DH :426-477).
        auto to_inertial = [&](bool en, bool vel) {
            const bool any_vel = __any(vel);
            if constexpr (JAC) {
                if (__any(!(cm == cm_scan))) {
                    cm_scan = cm;
                    down_scan(cm, bwd, star_i);
                }
                if constexpr (VAR) {
                    if (__any(!(dcm == dcm_scan))) {
                        dcm_scan = dcm;
                        down_scan(dcm, bwv, dstar_i);
                    }
                }
                __syncthreads();
                publish(0, h, im);
                if (VAR) publish(2, dh, im);
                if (any_vel) {
                    publish(1, hv, im);
                    if (VAR) publish(3, dhv, im);
                }
                __syncthreads();
                V3 n{0, 0, 0}, ns;
                scan_down(0, c, cm, bwd, star_i, n, ns);
                if (en) {
                    s = ns;
                    if (live) i = n;
                }
                if constexpr (VAR) {
                    scan_down(2, dc, dcm, bwv, dstar_i, n, ns);
                    if (en) {
                        ds = ns;
                        if (live) di = n;
                    }
                }
                if (any_vel) {
                    scan_down(1, cv, cm, bwd, star_i, n, ns);
                    if (en && vel) {
                        sv.set(ns);
                        if (live) iv.set(n);
                    }
                    if constexpr (VAR) {
                        scan_down(3, dcv, dcm, bwv, dstar_i, n, ns);
                        if (en && vel) {
                            dsv.set(ns);
                            if (live) div.set(n);
                        }
                    }
                }
            } else {
                const double mtot = cm, m0 = sm;
                __syncthreads();
                publish(0, V3{h.x * hm / mtot, h.y * hm / mtot, h.z * hm / mtot}, 0.);
                if (any_vel) publish(1, V3{hv.x * hm / m0, hv.y * hm / m0, hv.z * hm / m0}, 0.);
                __syncthreads();
                V3 x0{0., 0., 0.};
                ascending([&](int k, int q) {
                    const V4 o = ex[0][q];
                    x0.x += o.x; x0.y += o.y; x0.z += o.z;
                });
                if (en) {
                    im = hm;
                    s = V3{c.x - x0.x, c.y - x0.y, c.z - x0.z};
                    i = V3{h.x + s.x, h.y + s.y, h.z + s.z};
                }
                if (any_vel) {
                    V3 v0{0., 0., 0.};
                    ascending([&](int k, int q) {
                        const V4 o = ex[1][q];
                        v0.x += o.x; v0.y += o.y; v0.z += o.z;
                    });
                    if (en && vel) {
                        iv.set(V3{hv.x + cv.x, hv.y + cv.y, hv.z + cv.z});
                        sv.set(V3{cv.x - v0.x, cv.y - v0.y, cv.z - v0.z});
                    }
                }
            }
        };

        // ------------------------------------------------ operators of a step
        // integrator_whfast.c:589-636 (mu = G m0, Jacobi G eta_k) and the
        // variational drift :392-427
        auto kepler = [&](double hh, bool en) {
            if (!en || !live) return;
            const double mu = JAC ? eta_me * Gc : sm * Gc;
            if constexpr (VAR) {
                KepOut ko;
                warn |= kepler_solver(h.x, h.y, h.z, hv.x, hv.y, hv.z, mu, hh, &ko);
                kepler_var(ko, dh.x, dh.y, dh.z, dhv.x, dhv.y, dhv.z);
            } else {
                warn |= kepler_solver(h.x, h.y, h.z, hv.x, hv.y, hv.z, mu, hh);
            }
        };
        // integrator_whfast.c:638-672
        auto com = [&](double hh, bool en) {
            if (!en) return;
            c.x += hh * cv.x; c.y += hh * cv.y; c.z += hh * cv.z;
            if (VAR) {
                dc.x = dc.x + hh * dcv.x; dc.y = dc.y + hh * dcv.y; dc.z = dc.z + hh * dcv.z;
            }
        };
        // integrator_whfast.c:537-554 (DH)
        auto jump = [&](double hh, bool en) {
            __syncthreads();
            publish(0, V3{hm * hv.x, hm * hv.y, hm * hv.z}, 0.);
            __syncthreads();
            V3 q{0, 0, 0};
            ascending([&](int k, int at) {
                const V4 o = ex[0][at];
                q.x += o.x; q.y += o.y; q.z += o.z;
            });
            if (live && en) {
                h.x += hh * (q.x / sm);
                h.y += hh * (q.y / sm);
                h.z += hh * (q.z / sm);
            }
        };
        // -G/r^3 (BASIC, gravity.c:222-230) or -G/(r^2 r) (COMPENSATED, :315-341)
        // of a pair; times the source's mass and the displacement it is the term.
        auto pair_factor = [&](const V3& d) {
            if (COMP) {
                const double r2 = d.x * d.x + d.y * d.y + d.z * d.z + P.soft2;
                const double rr = sqrt(r2);
                return -(Gc / (r2 * rr));
            }
            const double r = sqrt(d.x * d.x + d.y * d.y + d.z * d.z + P.soft2);
            return -Gc / (r * r * r);
        };
        struct Sum {
            V3 a{0., 0., 0.}, k{0., 0., 0.};
        };
        auto add = [&](Sum& A, double f, const V3& d) {
            if (COMP) {
                kahan(f * d.x, A.a.x, A.k.x);
                kahan(f * d.y, A.a.y, A.k.y);
                kahan(f * d.z, A.a.z, A.k.z);
            } else {
                A.a.x += f * d.x;
                A.a.y += f * d.y;
                A.a.z += f * d.z;
            }
        };
        // Accelerations with gravity_ignore_terms INVOLVING_0 (DH: planets only)
        // or BETWEEN_0_AND_1 (Jacobi).  The star's term of a planet and the planet's of
        // the star share their factor (the displacement only changes sign).
        auto gravity = [&](bool en) {
            __syncthreads();
            publish(0, i, im);
            Sum A;
            if constexpr (JAC) {
                const V3 d{i.x - s.x, i.y - s.y, i.z - s.z};
                V3 ts{0., 0., 0.};
                if (live && me >= 2) {
                    const double f = pair_factor(d);
                    const double fs = f * im;
                    ts = V3{fs * -d.x, fs * -d.y, fs * -d.z};
                    add(A, f * sm, d);
                }
                publish(1, ts, 0.);
            }
            __syncthreads();
            if constexpr (JAC) {
                Sum B;
                for (int k = 2; k < N; k++) {
                    const V4 o = ex[1][gbase + k - 1];
                    if (COMP) {
                        kahan(o.x, B.a.x, B.k.x);
                        kahan(o.y, B.a.y, B.k.y);
                        kahan(o.z, B.a.z, B.k.z);
                    } else {
                        B.a.x += o.x;
                        B.a.y += o.y;
                        B.a.z += o.z;
                    }
                }
                if (en) {
                    sa = B.a;
                    if (VAR && gl == 0 && sys_ok) st3(P.body, st, 6, b0, sa);
                }
            }
            // the other planets in ascending order: entry n of 0 .. N-3 is planet
            // n+1, from my own on the one after it
            auto other = [&](int n) { return gbase + n + (n >= gl ? 1 : 0); };
            int n = 0;
            for (; n + 2 <= N - 2; n += 2) {
                const V4 o0 = ex[0][other(n)], o1 = ex[0][other(n + 1)];
                const V3 d0{i.x - o0.x, i.y - o0.y, i.z - o0.z};
                const V3 d1{i.x - o1.x, i.y - o1.y, i.z - o1.z};
                const double f0 = pair_factor(d0) * o0.w;
                const double f1 = pair_factor(d1) * o1.w;
                add(A, f0, d0);
                add(A, f1, d1);
            }
            if (n < N - 2) {
                const V4 o0 = ex[0][other(n)];
                const V3 d0{i.x - o0.x, i.y - o0.y, i.z - o0.z};
                add(A, pair_factor(d0) * o0.w, d0);
            }
            if (live && en) {
                a = A.a;
                if (VAR) st3(P.body, st, 6, bm, a);
            }
        };
        // gravity.c:533-640, first order, every body varied, the pairs (0,1) left
        // out when first == 2 (the step) and not when first == 1 (MEGNO).  Body
        // k's sum holds its terms with j < k, then those with i > k; a term enters
        // both bodies with opposite signs, so written with the displacement from
        // the other body it is added in either role.
        auto var_gravity = [&](bool en, int first) {
            __syncthreads();
            publish(0, i, im);
            publish(1, di, dm);
            // coefficients of one pair: the tidal tensor applied to dd, and r^-3
            auto tide = [&](const V3& d, const V3& dd, V3& t, double& r3inv) {
                const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
                const double r = sqrt(r2);
                r3inv = 1. / (r2 * r);
                const double r5inv = 3. * r3inv / r2;
                const double xx = d.x * d.x * r5inv - r3inv;
                const double yy = d.y * d.y * r5inv - r3inv;
                const double zz = d.z * d.z * r5inv - r3inv;
                const double xy = d.x * d.y * r5inv;
                const double xz = d.x * d.z * r5inv;
                const double yz = d.y * d.z * r5inv;
                t.x = dd.x * xx + dd.y * xy + dd.z * xz;
                t.y = dd.x * xy + dd.y * yy + dd.z * yz;
                t.z = dd.x * xz + dd.y * yz + dd.z * zz;
            };
            auto term = [&](double m, double dmass, const V3& d, const V3& t, double r3inv) {
                const double Gm = Gc * m, dGm = Gc * dmass;
                return V3{Gm * t.x - dGm * r3inv * d.x, Gm * t.y - dGm * r3inv * d.y,
                          Gm * t.z - dGm * r3inv * d.z};
            };
            V3 A{0., 0., 0.}, t;
            double r3;
            V3 ts{0., 0., 0.};
            if (live && me >= first) {
                const V3 d{i.x - s.x, i.y - s.y, i.z - s.z}, dd{di.x - ds.x, di.y - ds.y, di.z - ds.z};
                tide(d, dd, t, r3);
                const V3 q = term(sm, dsm, d, t, r3);
                A.x += q.x; A.y += q.y; A.z += q.z;
                ts = term(im, dm, d, t, r3);
            }
            publish(2, ts, 0.);
            __syncthreads();
            V3 B{0., 0., 0.};
            for (int k = first; k < N; k++) {
                const V4 o = ex[2][gbase + k - 1];
                B.x -= o.x; B.y -= o.y; B.z -= o.z;
            }
            auto other = [&](int n) { return gbase + n + (n >= gl ? 1 : 0); };
            auto pair = [&](int at, V3& q) {
                const V4 o = ex[0][at], od = ex[1][at];
                const V3 d{i.x - o.x, i.y - o.y, i.z - o.z}, dd{di.x - od.x, di.y - od.y, di.z - od.z};
                V3 tt;
                double r3i;
                tide(d, dd, tt, r3i);
                q = term(o.w, od.w, d, tt, r3i);
            };
            int n = 0;
            for (; n + 2 <= N - 2; n += 2) {
                V3 q0, q1;
                pair(other(n), q0);
                pair(other(n + 1), q1);
                A.x += q0.x; A.y += q0.y; A.z += q0.z;
                A.x += q1.x; A.y += q1.y; A.z += q1.z;
            }
            if (n < N - 2) {
                V3 q0;
                pair(other(n), q0);
                A.x += q0.x; A.y += q0.y; A.z += q0.z;
            }
            if (!en) return;
            dsa = B;
            if (gl == 0 && sys_ok) st3(P.pv, vs, 6, vb0, B);
            if (live) {
                da = A;
                st3(P.pv, vs, 6, vbm, A);
            }
        };
        // integrator_whfast.c:494-501 (DH), :439-490 (Jacobi: accelerations to Jacobi
        // form, transformations.c:147-176, the kick, then the Kepler term of the
        // interior bodies, for the bodies and the variational set)
        auto interaction = [&](double hh, bool en) {
            if constexpr (JAC) {
                __syncthreads();
                publish(0, a, im);
                if (VAR) publish(1, da, im);
                __syncthreads();
                V3 ja{0., 0., 0.}, jd{0., 0., 0.}, dcom{0., 0., 0.};
                scan_up(0, sa, ja, nullptr);
                if constexpr (VAR) scan_up(1, dsa, jd, &dcom);
                if (!en) return;
                if (VAR && gl == 0 && sys_ok) st3(P.jv, vs, 6, vb0, dcom);
                if (!live) return;
                double rj2i = 0., prefac1 = 0., rj3iM = 0.;
                if (me > 1) {
                    rj2i = 1. / (h.x * h.x + h.y * h.y + h.z * h.z);
                    const double rji = sqrt(rj2i);
                    rj3iM = rji * rj2i * Gc * eta_me;
                    prefac1 = hh * rj3iM;
                }
                if constexpr (VAR) {
                    st3(P.jv, vs, 6, vbm, jd);
                    if (me > 1) {
                        const double rj5M = rj3iM * rj2i;
                        const double rdr = dh.x * h.x + dh.y * h.y + dh.z * h.z;
                        const double prefac2 = -hh * 3. * rdr * rj5M;
                        dhv.x += prefac1 * dh.x + prefac2 * h.x;
                        dhv.y += prefac1 * dh.y + prefac2 * h.y;
                        dhv.z += prefac1 * dh.z + prefac2 * h.z;
                    }
                    dhv.x += hh * jd.x;
                    dhv.y += hh * jd.y;
                    dhv.z += hh * jd.z;
                }
                hv.x += hh * ja.x;
                hv.y += hh * ja.y;
                hv.z += hh * ja.z;
                if (me > 1) {
                    hv.x += prefac1 * h.x;
                    hv.y += prefac1 * h.y;
                    hv.z += prefac1 * h.z;
                }
            } else {
                if (!live || !en) return;
                hv.x += hh * a.x;
                hv.y += hh * a.y;
                hv.z += hh * a.z;
            }
        };
        // integrator_whfast.c:1250-1258 and tools.c:1483-1522: the variational
        // accelerations with every term, the ordered sums over the bodies, and the
        // system's MEGNO sums (time advanced as the reference's two half steps).
        auto megno_step = [&](bool en) {
            var_gravity(en, 1);
            auto prod = [&](const V3& x, const V3& v, const V3& acc, V3& p, V3& q, V3& xx, V3& vv) {
                p = V3{v.x * x.x, v.y * x.y, v.z * x.z};
                q = V3{acc.x * v.x, acc.y * v.y, acc.z * v.z};
                xx = V3{x.x * x.x, x.y * x.y, x.z * x.z};
                vv = V3{v.x * v.x, v.y * v.y, v.z * v.z};
            };
            V3 p, q, xx, vv;
            prod(di, div.get(), da, p, q, xx, vv);
            __syncthreads();
            publish(0, p, 0.);
            publish(1, q, 0.);
            publish(2, xx, 0.);
            publish(3, vv, 0.);
            __syncthreads();
            double deltad = 0., delta2 = 0.;
            auto fold = [&](double p0, double p1, double p2, double q0, double q1, double q2, double x0, double x1,
                            double x2, double v0, double v1, double v2) {
                deltad += p0; deltad += p1; deltad += p2;
                deltad += q0; deltad += q1; deltad += q2;
                delta2 += x0; delta2 += x1; delta2 += x2;
                delta2 += v0; delta2 += v1; delta2 += v2;
            };
            prod(ds, dsv.get(), dsa, p, q, xx, vv);
            fold(p.x, p.y, p.z, q.x, q.y, q.z, xx.x, xx.y, xx.z, vv.x, vv.y, vv.z);
            ascending([&](int k, int at) {
                const V4 o0 = ex[0][at], o1 = ex[1][at], o2 = ex[2][at], o3 = ex[3][at];
                fold(o0.x, o0.y, o0.z, o1.x, o1.y, o1.z, o2.x, o2.y, o2.z, o3.x, o3.y, o3.z);
            });
            const double dd = deltad / delta2;
            if (!en) return;
            if (P.megno == 1) {
                if (gl == 0) *P.megno_out = dd;
                return;
            }
            double M[kMegnoFields];
            for (int f = 0; f < kMegnoFields; f++) M[f] = megno[f][lane];
            double tt = M[0];
            tt += dt / 2.;
            tt += dt / 2.;
            const double t0 = M[1];
            const double n = M[8] + 1.;
            M[2] += dt * 2. * (tt - t0) * dd;
            const double Y = M[2] / (tt - t0);
            M[3] += Y * dt;
            const double d_t = tt - t0 - M[6];
            M[6] += d_t / n;
            const double meg = tt == t0 ? 0. : M[3] / (tt - t0);
            const double d_Y = meg - M[7];
            M[7] += d_Y / n;
            M[4] += (n - 1.) / n * (tt - t0 - M[6]) * (meg - M[7]);
            M[5] += (n - 1.) / n * (tt - t0 - M[6]) * (tt - t0 - M[6]);
            M[0] = tt;
            M[8] = n;
            for (int f = 0; f < kMegnoFields; f++) megno[f][lane] = M[f];
        };
        // tools.c:1313-1380 on a batched set: divided by its largest coordinate
        // once that exceeds 1e100
        auto var_rescale = [&](bool en) {
            auto grow = [](double scale, double v) {
                const double w = fabs(v);
                return w > scale ? w : scale;
            };
            auto largest = [&](const V3& x, const V3& v) {
                return grow(grow(grow(grow(grow(grow(0., x.x), x.y), x.z), v.x), v.y), v.z);
            };
            V3 pv = div.get(), ps = dsv.get();
            const double own = live ? largest(di, pv) : 0.;
            const double star = largest(ds, ps);
            if (!__any(own > 1e100 || star > 1e100)) return;
            __syncthreads();
            publish(0, V3{0., 0., 0.}, own);
            __syncthreads();
            double scale = star;
            ascending([&](int k, int at) { scale = grow(scale, ex[0][at].w); });
            if (!en || !(scale > 1e100)) return;
            auto divide = [&](V3& v) {
                v.x = v.x / scale; v.y = v.y / scale; v.z = v.z / scale;
            };
            divide(di);
            divide(pv);
            divide(ds);
            divide(ps);
            div.set(pv);
            dsv.set(ps);
        };

        // ------------------------------------------------ the launch as phases
        // integrator_whfast.c:1051-1259.
        bool modified = P.did_modify || (sys_ok && (S.req & 2));
        bool act = false, want = false, sen = false;
        long n = 0;
        auto kick = [&](double hh, bool en, bool vel) {
            if (!JAC) jump(dt / 2., en);
            // the inertial velocities of a step are visible only after the
            // system's last one (or are replaced by a synchronization)
            to_inertial(en, vel);
            if constexpr (VAR) var_gravity(en, 2);
            gravity(en);
            interaction(hh, en);
            if (!JAC) jump(dt / 2., en);
        };
        if constexpr (!CHAIN) {
            // A phase is a drift, then a step's kick or the end of a synchronization:
            // before a step whose bodies were modified (PRE), after one in safe
            // mode (POST), or at the launch's end.
            enum { STEP, PRE, POST, END };
            int mode = STEP;
            for (bool begun = false;; begun = true) {
                if (begun) {
                    const bool stepping = mode == STEP;
                    const bool en = stepping ? act : sen;
                    const double hd = stepping && !sync ? dt : dt / 2.;
                    kepler(hd, en);
                    com(hd, en);
                    if (stepping) {
                        kick(dt, act, act && n == my_steps - 1);
                        if (act) sync = 0;
                        want = sen = act && safe;
                        if (__any(want)) {
                            mode = POST;
                            continue;
                        }
                    } else {
                        to_inertial(sen, sen);
                        if (want) sync = 1;
                        if (mode == END) break;
                        if (mode == PRE) {
                            from_inertial(want);
                            mode = STEP;
                            continue;
                        }
                    }
                    if (VAR && P.megno) megno_step(act);
                    if (VAR && P.megno == 2) var_rescale(act);
                    if (act) modified = false;
                    n++;
                }
                mode = STEP;
                if (n >= P.nsteps) {
                    want = sys_ok && (P.sync_at_end || (S.req & 1));
                    sen = want && !sync;
                    if (!__any(sen)) {
                        if (want) sync = 1;
                        break;
                    }
                    mode = END;
                    continue;
                }
                act = n < my_steps;
                want = act && (safe || modified);
                if (__any(want)) {
                    sen = want && !sync;
                    if (sen) warn |= 2;
                    if (__any(sen))
                        mode = PRE;
                    else
                        from_inertial(want);
                }
            }
        } else {
        // `where` is uniform: S_STEP runs the drifts and kicks of step n, S_SYNC
        // those of a synchronization; chain selects a corrector's phases in between
        // (integrator_whfast.c:653-784: a chain of Z(a, b) = drift a, kick -b, drift
        // -2a, kick b, drift a; the second corrector two U(a, b)).
        enum { S_NEXT, S_RECALC, S_CORRECT, S_CORRECT2, S_STEP, S_STEP_END, S_CLOSE, S_SYNC, S_SYNC2, S_SYNC_END, S_DONE };
        const double h_first = P.kernel == 2 ? 5. * dt / 8. : dt / 2.;
        const double h_sync = P.kernel == 2 ? 3. * dt / 8. : dt / 2.;
        int where = S_NEXT, back = S_DONE;      // back: where a synchronization returns to
        int chain = 0, at = 0, len = 0, after_chain = S_STEP;
        double inv = 1.;
        bool chain_en = false, first = false;
        int sub = 0;                             // composition kernel: kick of the step
        const CorrZ* cz = nullptr;
        // phases of a corrector for the systems with `en`, then on to `then`
        auto start_chain = [&](int which, double sign, bool en, int then) {
            chain = which;
            inv = sign;
            chain_en = en;
            after_chain = then;
            at = 0;
            if (which == 1) {
                int z = 0;
                cz = corrector_chain(P.corrector, z);
                len = 3 * z;
            } else {
                len = 20;
            }
        };
        for (;;) {
            // advance to the next drift
            bool drift = false;
            while (!drift && where != S_DONE) {
                if (chain) {
                    if (at < len) {
                        drift = true;
                        continue;
                    }
                    chain = 0;
                    where = after_chain;
                }
                switch (where) {
                    case S_NEXT: {
                        if (n >= P.nsteps) {
                            want = sys_ok && (P.sync_at_end || (S.req & 1));
                            back = S_DONE;
                            where = S_SYNC;
                            break;
                        }
                        act = n < my_steps;
                        want = act && (safe || modified);
                        if (want && !sync) warn |= 2;
                        back = S_RECALC;
                        where = __any(want && !sync) ? S_SYNC : (__any(want) ? S_RECALC : S_CORRECT);
                        break;
                    }
                    case S_RECALC: {
                        const bool rc = act && (safe || modified);
                        if (rc) sync = 1;
                        from_inertial(rc);
                        where = S_CORRECT;
                        break;
                    }
                    case S_CORRECT:
                        sub = 0;
                        where = S_STEP;
                        first = act && sync;
                        if (JAC && (P.corrector || P.corrector2) && __any(first)) {
                            if (P.corrector)
                                start_chain(1, 1., first, S_CORRECT2);
                            else
                                where = S_CORRECT2;
                        }
                        break;
                    case S_CORRECT2:
                        where = S_STEP;
                        if (P.corrector2) start_chain(2, 1., first, S_STEP);
                        break;
                    case S_STEP:
                        drift = true;
                        break;
                    case S_STEP_END: {
                        if (act) sync = 0;
                        want = act && safe;
                        back = S_CLOSE;
                        where = __any(want) ? S_SYNC : S_CLOSE;
                        break;
                    }
                    case S_CLOSE: {
                        if (VAR && P.megno) megno_step(act);
                        if (VAR && P.megno == 2) var_rescale(act);
                        if (act) modified = false;
                        n++;
                        where = S_NEXT;
                        break;
                    }
                    case S_SYNC:
                        sen = want && !sync;
                        if (__any(sen)) {
                            drift = true;
                        } else {
                            if (want) sync = 1;
                            where = back;
                        }
                        break;
                    case S_SYNC2:
                        if (P.corrector && JAC) {
                            start_chain(1, -1., sen, S_SYNC_END);
                        } else {
                            where = S_SYNC_END;
                        }
                        break;
                    case S_SYNC_END:
                        to_inertial(sen, sen);
                        if (want) sync = 1;
                        where = back;
                        break;
                    default:
                        where = S_DONE;
                        break;
                }
            }
            if (where == S_DONE && !drift) break;
            // this phase's drift and kick
            double hd = 0., hk = 0.;
            bool en = false, docom = false, dokick = false;
            if (chain == 1) {
                const CorrZ z = cz[at / 3];
                const int k = z.ka, part = at % 3;
                const double ca = (k < 0 ? -kCorrA[-k] : kCorrA[k]) * dt;
                const double cb = (z.kb * inv) * dt;
                en = chain_en;
                hd = part == 1 ? -2. * ca : ca;
                dokick = part < 2;
                hk = part == 0 ? -cb : cb;
                at++;
            } else if (chain == 2) {
                // U(a, b): a | a,+b | -a | -a,-b | a | a,-b | -a | -a,+b | a | -a
                const double sgn = at < 10 ? 0.5 : -0.5;
                const double ca = sgn * inv * dt;
                const double cb = kCorr2B * inv * dt;
                const int part = at % 10;
                const bool neg = part == 2 || part == 3 || part == 6 || part == 7 || part == 9;
                en = chain_en;
                hd = neg ? -ca : ca;
                dokick = (part & 1) && part < 9;
                hk = (part == 1 || part == 7) ? cb : -cb;
                at++;
            } else if (where == S_STEP) {
                en = act;
                docom = dokick = true;
                if (P.kernel != 2) {
                    hd = sync ? h_first : dt;
                    hk = dt;
                } else {
                    // integrator_whfast.c:1189-1218
                    hd = sub == 0 ? (sync ? h_first : dt)
                                  : (sub == 1 ? -dt / 4. : (sub == 2 ? dt / 8. : (sub == 3 ? -dt / 8. : dt / 4.)));
                    hk = sub == 2 ? dt : ((sub == 0 || sub == 3) ? -dt / 6. : dt / 6.);
                }
            } else {
                en = sen;
                hd = h_sync;
                docom = true;
            }
            kepler(hd, en);
            if (docom) com(hd, en);
            if (dokick) kick(hk, en, chain == 0 && sub == 0 && en && n == my_steps - 1);
            if (chain == 0) {
                if (where == S_STEP) {
                    if (P.kernel == 2 && sub < 4)
                        sub++;
                    else
                        where = S_STEP_END;
                } else if (where == S_SYNC) {
                    if (P.corrector2 && JAC)
                        start_chain(2, -1., sen, S_SYNC2);
                    else
                        where = S_SYNC2;
                }
            }
        }
        }
        // the system's flags: any of its lanes' warnings and solver branches
        warn = group_or(warn, lane - gl, G);

        // ---- store
        if (live) {
            st3(P.body, st, 0, bm, i);
            st3(P.body, st, 3, bm, iv.get());
            if (!VAR) st3(P.body, st, 6, bm, a);
            P.body[9 * st + bm] = im;
            st3(P.ph, st, 0, bm, h);
            st3(P.ph, st, 3, bm, hv);
            P.ph[6 * st + bm] = hm;
            if (VAR) {
                st3(P.pv, vs, 0, vbm, di);
                st3(P.pv, vs, 3, vbm, div.get());
                st3(P.jv, vs, 0, vbm, dh);
                st3(P.jv, vs, 3, vbm, dhv);
                P.jv[9 * vs + vbm] = dhm;
            }
        }
        if (sys_ok && gl == 0) {
            st3(P.body, st, 0, b0, s);
            st3(P.body, st, 3, b0, sv.get());
            if (!VAR) st3(P.body, st, 6, b0, sa);
            st3(P.ph, st, 0, b0, c);
            st3(P.ph, st, 3, b0, cv);
            P.ph[6 * st + b0] = cm;
            P.flags[sidx] = (unsigned)(sync & 1) | (unsigned)((warn & 15) << 1);
            if (VAR) {
                st3(P.pv, vs, 0, vb0, ds);
                st3(P.pv, vs, 3, vb0, dsv.get());
                st3(P.jv, vs, 0, vb0, dc);
                st3(P.jv, vs, 3, vb0, dcv);
                P.jv[9 * vs + vb0] = dcm;
                if (P.megno == 2)
                    for (int f = 0; f < kMegnoFields; f++)
                        P.megno_sys[(size_t)sidx * kMegnoFields + f] = megno[f][lane];
            }
        }
        __syncthreads();
    }
}

}  // namespace

// Two wavefronts per SIMD: all 1317 wavefronts of a 16384-system ensemble are
// resident at once.
#define RB_LANE __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
__global__ RB_LANE void k_lane_dh(WHParams P) { lane_body<false, false, false, false>(P); }
__global__ RB_LANE void k_lane_dh_comp(WHParams P) { lane_body<false, true, false, false>(P); }
__global__ RB_LANE void k_lane_jac(WHParams P) { lane_body<true, false, false, false>(P); }
__global__ RB_LANE void k_lane_var(WHParams P) { lane_body<true, false, true, false>(P); }
// with correctors or the composition kernel
__global__ RB_LANE void k_lane_jac_chain(WHParams P) { lane_body<true, false, false, true>(P); }
__global__ RB_LANE void k_lane_jac_comp(WHParams P) { lane_body<true, true, false, true>(P); }
__global__ RB_LANE void k_lane_var_chain(WHParams P) { lane_body<true, false, true, true>(P); }
#undef RB_LANE

// Whether the lane kernels take this launch.
bool whfast_lane_takes(const WHParams& P) {
    const bool jac = P.coords == WH_JACOBI;
    return P.all_active && (P.kernel == 0 || (P.kernel == 2 && jac)) && !P.jacgrav &&
           (P.nvar == 0 || (P.nvar == 1 && jac && !P.compensated && P.kernel == 0));
}

void whfast_lane_launch(const WHParams& P, hipStream_t st) {
    const bool chain = P.corrector || P.corrector2 || P.kernel == 2;
    void (*k)(WHParams);
    if (P.nvar)
        k = chain ? k_lane_var_chain : k_lane_var;
    else if (P.coords == WH_JACOBI)
        k = P.compensated ? k_lane_jac_comp : (chain ? k_lane_jac_chain : k_lane_jac);
    else
        k = P.compensated ? k_lane_dh_comp : k_lane_dh;
    hipLaunchKernelGGL(k, dim3(P.grid), dim3(64), 0, st, P);
}

// Wavefronts of the ensemble kernels that fit on one CU.
int whfast_lane_per_cu() {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_lane_dh, 64, 0) != hipSuccess || per_cu < 1) per_cu = 8;
    return per_cu;
}

}  // namespace rbamd
