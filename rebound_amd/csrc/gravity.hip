// Direct O(N^2) gravity on the GPU (reference: gravity.c:167-531) and the
// energy diagnostic (tools.c:108-162).
//
// Three precisions (rebound_amd.h):
//   EXACT  one lane per target i, sources j streamed through LDS tiles in
//          ascending order, IEEE sqrt/div and no contraction (the library is
//          built with -ffp-contract=off): every term and every partial sum is
//          the reference's OpenMP loop (gravity.c:215-232, 308-343), so the
//          result is bit-identical.
//   FP64   r^-3 from v_rsq_f64 refined to full double accuracy, fused
//          multiply-adds, each LDS tile's sum folded into the running sum
//          with Kahan compensation, and the source range split over
//          blockIdx.y so that N=65536 fills every SIMD; the partial sums are
//          added in a fixed order by a second kernel (deterministic).
//   SPLIT  displacement and r^2 in FP64, r^-1 from the FP32 reciprocal
//          square root (v_rsq_f32, about 2^-23 relative), cubed and
//          multiplied by m_j in FP64 (no FP32 exponent limit on r^-3 or m),
//          accumulation in FP64; each LDS tile's FP64 partial is folded into
//          the running sum with Kahan compensation.
//
// Data layout: structure of arrays (x, y, z, m as separate double arrays).
// Sources are staged per 256-wide tile into LDS as double4 (x, y, z, m) and
// read back as broadcasts (every lane of a wavefront reads the same entry).
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>

#include "ieee_mid.h"
#include "internal.h"

namespace rbamd {

static constexpr int kBlock = 256;     // targets per workgroup = sources per LDS tile (exact kernels)

// Shape of the fast kernels (tuning knobs, fixed at build time): targets per
// workgroup (= sources per LDS tile), unroll of the pair loop, and wavefronts
// per SIMD the register budget is sized for.
#ifndef RB_FAST_BLOCK
#define RB_FAST_BLOCK 256
#endif
#ifndef RB_FAST_UNROLL
#define RB_FAST_UNROLL 4
#endif
#ifndef RB_FAST_WAVES
#define RB_FAST_WAVES 4
#endif
#define RB_STR(x) #x
#define RB_UNROLL(n) _Pragma(RB_STR(unroll n))
static constexpr int kFast = RB_FAST_BLOCK;

struct GB3 { double x, y, z; };
// Ghost-box offsets travel by value in the kernel arguments (kernarg segment,
// read with scalar loads), so no copy or synchronisation is needed per call.
static constexpr int kMaxGB = 125;       // N_ghost up to 2 in all three axes
struct GBList {
    int n;
    GB3 g[kMaxGB];
    bool zero() const { return n == 1 && g[0].x == 0. && g[0].y == 0. && g[0].z == 0.; }
};

// Ghost-box offsets of a pass: the list of the simulation (kernel argument) or
// the single zero offset of a simulation without ghost boxes, whose kernels then
// carry no 3 KB list in their arguments and wait for no read of it.
struct GBFromList {
    GBList gl;
    __device__ int n() const { return gl.n; }
    __device__ const GB3& get(int g) const { return gl.g[g]; }
};
struct GBZero {
    __device__ int n() const { return 1; }
    __device__ GB3 get(int) const { return GB3{0., 0., 0.}; }
};

// The leapfrog's kick and closing drift, applied by the pass that finishes the
// accelerations (on == 0: nothing).  on == 2: the next step's opening drift
// follows as well (a launch of 2 to 3 us less per step), the positions between the
// two are kept in `back` (stride doubles per component) in case that step is not taken.
struct KickDrift {
    double *x, *y, *z, *vx, *vy, *vz;
    double kick, drift;
    int on;
    double* back;
    size_t stride;
};
// What it reads, fetched before the accelerations are known.
struct KickState {
    double x, y, z, vx, vy, vz;
};
__device__ __forceinline__ KickState kick_load(const KickDrift& kd, int i) {
    if (!kd.on) return KickState{};
    return KickState{kd.x[i], kd.y[i], kd.z[i], kd.vx[i], kd.vy[i], kd.vz[i]};
}
// integrator_leapfrog.c:84-93 then :72-82: v += dt*a, x += dt/2*v (twice: the
// next step's)
__device__ __forceinline__ void kick_store(const KickDrift& kd, int i, const KickState& s, double ax, double ay,
                                           double az) {
    if (!kd.on) return;
    const double vx = s.vx + kd.kick * ax;
    const double vy = s.vy + kd.kick * ay;
    const double vz = s.vz + kd.kick * az;
    kd.vx[i] = vx;
    kd.vy[i] = vy;
    kd.vz[i] = vz;
    double x = s.x + kd.drift * vx;
    double y = s.y + kd.drift * vy;
    double z = s.z + kd.drift * vz;
    if (kd.on == 2) {
        kd.back[i] = x;
        kd.back[kd.stride + i] = y;
        kd.back[2 * kd.stride + i] = z;
        x += kd.drift * vx;
        y += kd.drift * vy;
        z += kd.drift * vz;
    }
    kd.x[i] = x;
    kd.y[i] = y;
    kd.z[i] = z;
}

__device__ __forceinline__ bool skip_pair(int i, int j, int ignore) {
    if (ignore == 1 && ((j == 1 && i == 0) || (i == 1 && j == 0))) return true;
    if (ignore == 2 && (j == 0 || i == 0)) return true;
    return i == j;
}

__device__ __forceinline__ void kahan_add(double term, double& a, double& c) {
    const double yv = term - c;
    const double tv = a + yv;
    c = (tv - a) - yv;
    a = tv;
}

// ---------------------------------------------------------------- EXACT
// BASIC: gravity.c:217-231 (targets 0..N-1, sources 0..N_active-1 for every
// ghost box), then :259-276 (active targets also feel test particles when
// testparticle_type is set).  COMPENSATED: gravity.c:308-343 (active
// targets), :346-378 (test-particle targets), :379-410 (active targets feel
// test particles), no ghost boxes, Kahan sums.
//
// The terms are independent: four wavefronts of a workgroup compute them for
// TGT targets x TILE sources at a time (the reference's expressions, no
// contraction) into LDS rows, one row per (target, component), and a fifth
// wavefront adds the previous tile's rows meanwhile, one lane per row, in
// ascending source order: the reference's sequential sum, each component its own
// chain.  The rows are double-buffered, so one barrier per tile suffices.  Small N
// is bound by the chains (N dependent additions), so the summing lanes read their row
// sixteen terms ahead; the term threads load their sources two tiles ahead (staging
// them in LDS lost 15 % from 8192 bodies: fewer workgroups per CU).  A leapfrog step
// with the terms and the sums on the same wavefronts and now: 64 bodies 16.1 -> 11.3 us,
// 1024 32.3 -> 22.0, 8192 231 -> 181, 32768 3.16 -> 2.7 ms.
static constexpr int kExTermThreads = 256;
static constexpr int kExThreads = kExTermThreads + 64;

// PER pair factors of one target: -G / r^3 (BASIC, gravity.c:222-230) or
// G / (r^2 r) (COMPENSATED, :315-341), from the short IEEE sequences of
// ieee_mid.h while every operand is in their range.
template <bool COMP, int PER>
__device__ __forceinline__ void exact_factors(const double* r2, double G, bool g_mid, double* f) {
    unsigned int far = 0;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        far = max(far, mid_distance(r2[q]));
        const double r = sqrt_mid(r2[q]);
        f[q] = COMP ? div_mid(G, r2[q] * r) : div_mid(-G, r * r * r);
    }
    if (!g_mid || far >= kMidSpan) {
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const double r = sqrt(r2[q]);
            f[q] = COMP ? G / (r2[q] * r) : -G / (r * r * r);
        }
    }
}

template <bool COMP, int TGT, int TILE, class GBS>
__global__ __launch_bounds__(kExThreads) void k_exact(const double* __restrict__ x, const double* __restrict__ y,
                                                       const double* __restrict__ z, const double* __restrict__ m,
                                                       double* __restrict__ ax, double* __restrict__ ay,
                                                       double* __restrict__ az, int N, int N_active, int tp_type,
                                                       int ignore, double G, double soft2, GBS gbs) {
    constexpr int PER = TGT * TILE / kExTermThreads;   // terms per thread and tile
    constexpr int ROWS = 3 * TGT;
    constexpr int PITCH = TILE + 2;                    // row pitch (doubles): 16-byte aligned rows, spread banks
    static_assert(PER % 2 == 0 && PER * kExTermThreads == TGT * TILE && kExTermThreads % TGT == 0, "tile shape");
    static_assert(ROWS <= 64 && TILE % 32 == 0, "one summing lane per row, rows read in sixteens");
    __shared__ __align__(16) double T[2][ROWS][PITCH];
    const int tid = threadIdx.x;
    const int i0 = blockIdx.x * TGT;
    const int ngb = gbs.n();
    int buf = 0;
    if (tid < kExTermThreads) {
        // thread -> (target ti, sources tj0 .. tj0 + PER - 1 of a tile)
        const int ti = tid % TGT;
        const int tj0 = (tid / TGT) * PER;
        const int i = min(i0 + ti, N - 1);             // rows past the last target are not added
        const double xi = x[i], yi = y[i], zi = z[i];
        const bool g_mid = mid_distance(fabs(G)) < kMidSpan;
        for (int g = 0; g < ngb; g++) {
            const GB3 gb = gbs.get(g);
            for (int pass = 0; pass < (tp_type ? 2 : 1); pass++) {
                const int j0 = pass == 0 ? 0 : N_active;
                const int j1 = pass == 0 ? N_active : N;
                // this thread's sources, loaded two tiles ahead (a tile of small N
                // takes 0.3 us, less than a fetch of what the drift just wrote)
                double4 ahead[2][PER];
                auto fetch = [&](int t, double4* o) {
#pragma unroll
                    for (int q = 0; q < PER; q++) {
                        const int j = min(t + tj0 + q, j1 - 1);
                        o[q] = make_double4(x[j], y[j], z[j], m[j]);
                    }
                };
                auto tile = [&](int t, double4* o) {
                    double dx[PER], dy[PER], dz[PER], r2[PER], f[PER], cm[PER];
#pragma unroll
                    for (int q = 0; q < PER; q++) {
                        if (COMP) {
                            dx[q] = xi - o[q].x;
                            dy[q] = yi - o[q].y;
                            dz[q] = zi - o[q].z;
                        } else {
                            dx[q] = (gb.x + xi) - o[q].x;
                            dy[q] = (gb.y + yi) - o[q].y;
                            dz[q] = (gb.z + zi) - o[q].z;
                        }
                        r2[q] = dx[q] * dx[q] + dy[q] * dy[q] + dz[q] * dz[q] + soft2;
                        cm[q] = o[q].w;
                    }
                    if (t + 2 * TILE < j1) fetch(t + 2 * TILE, o);
                    exact_factors<COMP, PER>(r2, G, g_mid, f);
#pragma unroll
                    for (int q = 0; q < PER; q += 2) {
                        const double w0 = (COMP ? -f[q] : f[q]) * cm[q];
                        const double w1 = (COMP ? -f[q + 1] : f[q + 1]) * cm[q + 1];
                        double2* row = reinterpret_cast<double2*>(&T[buf][3 * ti][tj0 + q]);
                        row[0] = make_double2(w0 * dx[q], w1 * dx[q + 1]);
                        row[PITCH / 2] = make_double2(w0 * dy[q], w1 * dy[q + 1]);
                        row[PITCH] = make_double2(w0 * dz[q], w1 * dz[q + 1]);
                    }
                    // After this barrier the summers read T[buf]; the next writes
                    // to T[buf] come two tiles later, after the next barrier,
                    // which the summers reach only once this sum is done.
                    __syncthreads();
                    buf ^= 1;
                };
                if (j0 < j1) fetch(j0, ahead[0]);
                if (j0 + TILE < j1) fetch(j0 + TILE, ahead[1]);
                for (int t = j0; t < j1; t += 2 * TILE) {
                    tile(t, ahead[0]);
                    if (t + TILE < j1) tile(t + TILE, ahead[1]);
                }
            }
        }
        return;
    }
    // lanes 0 .. ROWS-1: (target si, component sc)
    const int lane = tid - kExTermThreads;
    const int si = i0 + lane / 3;
    const int sc = lane % 3;
    const bool summer = lane < ROWS && si < N;
    double acc = 0., comp = 0.;
    auto add = [&](double term) {
        if (COMP)
            kahan_add(term, acc, comp);
        else
            acc += term;
    };
    for (int g = 0; g < ngb; g++) {
        for (int pass = 0; pass < (tp_type ? 2 : 1); pass++) {
            const int j0 = pass == 0 ? 0 : N_active;
            const int j1 = pass == 0 ? N_active : N;
            // the second pass only reaches active targets
            const bool mine = summer && !(pass == 1 && si >= N_active);
            auto skipped = [&](int j) {
                if (COMP || pass == 0) return skip_pair(si, j, ignore);
                return (ignore == 1 && j == 1 && si == 0) || (ignore == 2 && (j == 0 || si == 0));
            };
            for (int t = j0; t < j1; t += TILE, buf ^= 1) {
                const int n = min(TILE, j1 - t);
                __syncthreads();
                if (!mine) continue;
                const double2* row = reinterpret_cast<const double2*>(T[buf][lane]);
                // Pairs the reference leaves out: the target itself and,
                // with ignored terms, pairs with bodies 0 and 1.
                const bool self = (COMP || pass == 0) && t <= si && si < t + n;
                const bool rare = ignore != 0 && (t < 2 || si < 2);
                const bool whole = !self && !rare && n == TILE;
                double2 v[2][8];
#pragma unroll
                for (int k = 0; k < 8; k++) v[0][k] = row[k];
#pragma unroll
                for (int h = 0; h < TILE / 16; h++) {
                    if (h + 1 < TILE / 16) {
#pragma unroll
                        for (int k = 0; k < 8; k++) v[(h + 1) & 1][k] = row[8 * (h + 1) + k];
                    }
                    if (whole) {
#pragma unroll
                        for (int k = 0; k < 8; k++) {
                            add(v[h & 1][k].x);
                            add(v[h & 1][k].y);
                        }
                        continue;
                    }
#pragma unroll
                    for (int k = 0; k < 16; k++) {
                        const int at = 16 * h + k;
                        bool left_out = at >= n || (self && t + at == si);
                        if (rare) left_out = left_out || skipped(t + at);
                        const double term = k & 1 ? v[h & 1][k / 2].y : v[h & 1][k / 2].x;
                        if (COMP) {
                            const double s0 = acc, c0 = comp;
                            add(term);
                            acc = left_out ? s0 : acc;
                            comp = left_out ? c0 : comp;
                        } else {
                            // a zero changes nothing: the sum starts from +0 and is never -0
                            add(left_out ? 0. : term);
                        }
                    }
                }
            }
        }
    }
    if (summer) {
        double* out = sc == 0 ? ax : (sc == 1 ? ay : az);
        out[si] = acc;
    }
}

// ---------------------------------------------------------------- EXACT, row-wise (large N)
// One thread per target adds its terms in ascending source order; the terms
// of tiles away from the target are independent and overlap in flight.  At
// large N this beats the LDS-term kernel above, whose per-term LDS traffic
// and barriers cost more than the serial chain hides.
//
// gravity.c:217-231 (targets 0..N-1, sources 0..N_active-1 for every ghost
// box), then :259-276 (active targets also feel test particles when
// testparticle_type is set).
__global__ __launch_bounds__(kBlock) void k_basic_exact(
    const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
    const double* __restrict__ m, double* __restrict__ ax, double* __restrict__ ay, double* __restrict__ az,
    int N, int N_active, int tp_type, int ignore, double G, double soft2, GBList gl) {
    __shared__ double4 tile[kBlock];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const bool live = i < N;
    const int blk_lo = blockIdx.x * kBlock, blk_hi = blk_lo + kBlock;
    const double xi = live ? x[i] : 0., yi = live ? y[i] : 0., zi = live ? z[i] : 0.;
    double a_x = 0., a_y = 0., a_z = 0.;
    const bool g_mid = mid_distance(fabs(G)) < kMidSpan;
    for (int g = 0; g < gl.n; g++) {
        const GB3 gb = gl.g[g];
        for (int pass = 0; pass < 2; pass++) {
            int j0 = pass == 0 ? 0 : N_active;
            int j1 = pass == 0 ? N_active : N;
            if (pass == 1 && !tp_type) break;
            for (int t = j0; t < j1; t += kBlock) {
                __syncthreads();
                const int jj = t + (int)threadIdx.x;
                if (jj < j1) tile[threadIdx.x] = make_double4(x[jj], y[jj], z[jj], m[jj]);
                __syncthreads();
                const int n = min(kBlock, j1 - t);
                if (!live || (pass == 1 && i >= N_active)) continue;
                auto terms = [&](auto count, const double4* s) {
                    constexpr int PER = decltype(count)::value;
                    double dx[PER], dy[PER], dz[PER], r2[PER], f[PER];
#pragma unroll
                    for (int q = 0; q < PER; q++) {
                        dx[q] = (gb.x + xi) - s[q].x;
                        dy[q] = (gb.y + yi) - s[q].y;
                        dz[q] = (gb.z + zi) - s[q].z;
                        r2[q] = dx[q] * dx[q] + dy[q] * dy[q] + dz[q] * dz[q] + soft2;
                    }
                    exact_factors<false, PER>(r2, G, g_mid, f);
#pragma unroll
                    for (int q = 0; q < PER; q++) {
                        const double prefact = f[q] * s[q].w;
                        a_x += prefact * dx[q];
                        a_y += prefact * dy[q];
                        a_z += prefact * dz[q];
                    }
                };
                using One = std::integral_constant<int, 1>;
                using Four = std::integral_constant<int, 4>;
                // Tiles without this block's targets (and, with ignored terms,
                // without bodies 0 and 1 as sources or among the block's
                // targets) need no per-pair test: the terms are then
                // independent work the compiler can overlap, while the sums
                // still add them in ascending j.
                const bool check =
                    (pass == 0 && t < blk_hi && t + n > blk_lo) || (ignore != 0 && (t < 2 || blk_lo < 2));
                if (!check) {
                    int k = 0;
                    for (; k + 4 <= n; k += 4) terms(Four{}, tile + k);
                    for (; k < n; k++) terms(One{}, tile + k);
                    continue;
                }
                for (int k = 0; k < n; k++) {
                    const int j = t + k;
                    if (pass == 0) {
                        if (skip_pair(i, j, ignore)) continue;
                    } else {
                        if (ignore == 1 && j == 1 && i == 0) continue;
                        if (ignore == 2 && (j == 0 || i == 0)) continue;
                    }
                    terms(One{}, tile + k);
                }
            }
        }
    }
    if (live) {
        ax[i] = a_x;
        ay[i] = a_y;
        az[i] = a_z;
    }
}

// COMPENSATED, row-wise
// gravity.c:308-343 (active targets), :346-378 (test-particle targets), :379-410
// (active targets feel test particles).  No ghost boxes in the reference.

__global__ __launch_bounds__(kBlock) void k_comp_exact(
    const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
    const double* __restrict__ m, double* __restrict__ ax, double* __restrict__ ay, double* __restrict__ az,
    int N, int N_active, int tp_type, int ignore, double G, double soft2) {
    __shared__ double4 tile[kBlock];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const bool live = i < N;
    const int blk_lo = blockIdx.x * kBlock, blk_hi = blk_lo + kBlock;
    const double xi = live ? x[i] : 0., yi = live ? y[i] : 0., zi = live ? z[i] : 0.;
    double a_x = 0., a_y = 0., a_z = 0., c_x = 0., c_y = 0., c_z = 0.;
    const bool g_mid = mid_distance(fabs(G)) < kMidSpan;
    for (int pass = 0; pass < 2; pass++) {
        int j0 = pass == 0 ? 0 : N_active;
        int j1 = pass == 0 ? N_active : N;
        if (pass == 1 && !tp_type) break;
        for (int t = j0; t < j1; t += kBlock) {
            __syncthreads();
            const int jj = t + (int)threadIdx.x;
            if (jj < j1) tile[threadIdx.x] = make_double4(x[jj], y[jj], z[jj], m[jj]);
            __syncthreads();
            const int n = min(kBlock, j1 - t);
            if (!live || (pass == 1 && i >= N_active)) continue;
            auto terms = [&](auto count, const double4* s) {
                constexpr int PER = decltype(count)::value;
                double dx[PER], dy[PER], dz[PER], r2[PER], f[PER];
#pragma unroll
                for (int q = 0; q < PER; q++) {
                    dx[q] = xi - s[q].x;
                    dy[q] = yi - s[q].y;
                    dz[q] = zi - s[q].z;
                    r2[q] = dx[q] * dx[q] + dy[q] * dy[q] + dz[q] * dz[q] + soft2;
                }
                exact_factors<true, PER>(r2, G, g_mid, f);
#pragma unroll
                for (int q = 0; q < PER; q++) {
                    const double prefactj = -f[q] * s[q].w;
                    kahan_add(prefactj * dx[q], a_x, c_x);
                    kahan_add(prefactj * dy[q], a_y, c_y);
                    kahan_add(prefactj * dz[q], a_z, c_z);
                }
            };
            using One = std::integral_constant<int, 1>;
            using Four = std::integral_constant<int, 4>;
            const bool check = (t < blk_hi && t + n > blk_lo) || (ignore != 0 && (t < 2 || blk_lo < 2));
            if (!check) {
                int k = 0;
                for (; k + 4 <= n; k += 4) terms(Four{}, tile + k);
                for (; k < n; k++) terms(One{}, tile + k);
                continue;
            }
            for (int k = 0; k < n; k++) {
                const int j = t + k;
                if (skip_pair(i, j, ignore)) continue;
                terms(One{}, tile + k);
            }
        }
    }
    if (live) {
        ax[i] = a_x;
        ay[i] = a_y;
        az[i] = a_z;
    }
}

// Measured on gfx950 (leapfrog steps; the start of the lines: sums and terms on the
// same wavefront, sources one tile ahead, full-range square root and division):
// 8 targets x 64 sources beat 16 x 64 at every N (1024 bodies 23.5 us against 29.9,
// 16384 0.70 ms against 0.99; before 32.0 and 0.86), and the row-wise kernel from
// about 57000 (49152 bodies 5.7 ms against 6.4, 65536 9.9 against 8.5; before 6.6
// and 8.9).
static constexpr int kExactRowwiseN = 57344;

template <bool COMP>
static void launch_exact(hipStream_t st, const double* x, const double* y, const double* z, const double* m,
                         double* ax, double* ay, double* az, int N, int N_active, int tp_type, int ignore, double G,
                         double soft2, const GBList& gl) {
    const dim3 grid((N + 7) / 8);
    if (N >= kExactRowwiseN) {
        if (COMP)
            hipLaunchKernelGGL(k_comp_exact, dim3((N + kBlock - 1) / kBlock), dim3(kBlock), 0, st, x, y, z, m, ax,
                               ay, az, N, N_active, tp_type, ignore, G, soft2);
        else
            hipLaunchKernelGGL(k_basic_exact, dim3((N + kBlock - 1) / kBlock), dim3(kBlock), 0, st, x, y, z, m, ax,
                               ay, az, N, N_active, tp_type, ignore, G, soft2, gl);
    } else if (COMP || gl.zero()) {
        hipLaunchKernelGGL((k_exact<COMP, 8, 64, GBZero>), grid, dim3(kExThreads), 0, st, x, y, z, m, ax, ay, az, N,
                           N_active, tp_type, ignore, G, soft2, GBZero{});
    } else {
        hipLaunchKernelGGL((k_exact<false, 8, 64, GBFromList>), grid, dim3(kExThreads), 0, st, x, y, z, m, ax, ay,
                           az, N, N_active, tp_type, ignore, G, soft2, GBFromList{gl});
    }
}

// ---------------------------------------------------------------- FP64 / SPLIT / COMP-FP64
// Pair kernel of the fast modes.  Accumulates S_i = sum_j m_j r_ij^-3 d_ij over
// one chunk of sources (blockIdx.y) and writes it (and for the compensated
// variant its Kahan carry) to the partial buffer; k_reduce applies -G.
enum FastMode { FM_FP64 = 0, FM_SPLIT = 1, FM_COMP = 2 };

// r^-3 in FP64.  v_rsq_f64 is good to 2^-24 (measured on gfx950); it is
// refined through e = 1 - r2*y^2 (|e| < 2^-23):
//   r^-3 = y^3 (1 - e)^(-3/2) = y^3 (1 + 3/2 e + 15/8 e^2 + O(e^3)),
// leaving a relative error of order 2^-69, far below FP64 rounding.
// `c15` is 1.5 held in a register: a GFX9 VOP3 instruction takes at most one
// scalar or literal operand, so fma(e, 1.875, 1.5) with both constants would
// be rebuilt from two v_mov per pair.
__device__ __forceinline__ double rinv3_fp64(double r2, double c15, double c1875) {
    const double yv = __builtin_amdgcn_rsq(r2);
    const double h = yv * yv;
    const double e = fma(-r2, h, 1.0);
    const double y3 = h * yv;
    const double p = fma(e, c1875, c15);
    return fma(y3, e * p, y3);
}

// A loop-invariant constant kept in a VGPR (opaque to constant folding).
__device__ __forceinline__ double vreg_const(double v) {
    asm volatile("" : "+v"(v));
    return v;
}

// kahan_add of the product w d, unrounded: one operation less, one rounding less.
__device__ __forceinline__ void kahan_fma(double w, double d, double& a, double& c) {
    const double yv = fma(w, d, -c);
    const double tv = a + yv;
    c = (tv - a) - yv;
    a = tv;
}

template <int MODE, bool CHECK>
__device__ __forceinline__ void pair_tile(const double4* __restrict__ tile, int n,
                                          int jbase, int i, int ignore, double gx, double gy, double gz,
                                          double soft2, double& sx, double& sy, double& sz, double& cx, double& cy,
                                          double& cz, double c15, double c1875) {
    RB_UNROLL(RB_FAST_UNROLL)
    for (int k = 0; k < n; k++) {
        const double4 s = tile[k];
        const double dx = gx - s.x;
        const double dy = gy - s.y;
        const double dz = gz - s.z;
        const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, soft2)));
        double w;
        if (MODE == FM_SPLIT) {
            // r^-1 from the FP32 reciprocal square root; its cube and the
            // mass factor in FP64, so only r^2 itself must lie in FP32's
            // normal range (about 1e-19 < r < 1.8e19 in simulation units)
            const double yv = (double)__builtin_amdgcn_rsqf((float)r2);
            w = yv * yv * yv * s.w;
        } else {
            w = s.w * rinv3_fp64(r2, c15, c1875);
        }
        if (CHECK) {
            const int j = jbase + k;
            if (skip_pair(i, j, ignore)) w = 0.;
        }
        if (MODE == FM_COMP) {
            kahan_fma(w, dx, sx, cx);
            kahan_fma(w, dy, sy, cy);
            kahan_fma(w, dz, sz, cz);
        } else {
            sx = fma(w, dx, sx);
            sy = fma(w, dy, sy);
            sz = fma(w, dz, sz);
        }
    }
}

// One workgroup of the pair kernel: targets bx*kFast.. of n_recv, sources of
// chunk `by` of [j_begin, j_end).  Writes the chunk's sums and carries to
// `partial` (pstride doubles per component).
template <int MODE, class GBS>
__device__ __forceinline__ void direct_fast_block(const double* __restrict__ x, const double* __restrict__ y,
                                                  const double* __restrict__ z, const double* __restrict__ m,
                                                  int n_recv, int j_begin, int j_end, int chunk, int ignore,
                                                  double soft2, const GBS& gbs, double* __restrict__ partial,
                                                  int pstride, int bx, int by, double4* tile) {
    const int i = bx * kFast + threadIdx.x;
    const bool live = i < n_recv;
    const double xi = live ? x[i] : 0., yi = live ? y[i] : 0., zi = live ? z[i] : 0.;
    const int j0 = j_begin + by * chunk;
    const int j1 = min(j_end, j0 + chunk);
    const int blk_lo = bx * kFast;
    const int blk_hi = blk_lo + kFast;
    double sx = 0., sy = 0., sz = 0.;      // running sums
    double cx = 0., cy = 0., cz = 0.;      // Kahan carries (COMP per pair, FP64/SPLIT per tile)
    const double c15 = vreg_const(1.5);
    const double c1875 = vreg_const(1.875);
    // the next tile's source of this thread, fetched a tile ahead (the first with
    // the targets, not after a barrier that waits for them)
    auto source = [&](int t) {
        const int jj = t + (int)threadIdx.x;
        return jj < j1 ? make_double4(x[jj], y[jj], z[jj], m[jj]) : make_double4(0., 0., 0., 0.);
    };
    double4 ahead = source(j0);
    for (int g = 0; g < gbs.n(); g++) {
        const GB3 gb = gbs.get(g);
        const double gx = gb.x + xi, gy = gb.y + yi, gz = gb.z + zi;
        for (int t = j0; t < j1; t += kFast) {
            __syncthreads();
            tile[threadIdx.x] = ahead;
            __syncthreads();
            ahead = source(t + kFast < j1 ? t + kFast : j0);
            const int n = min(kFast, j1 - t);
            // Only tiles holding a target of this block, or sources 0/1 when
            // terms are ignored, need the per-pair skip test (target 0 with
            // ignore == 2 is zeroed by the reduction).
            const bool check = (t < blk_hi && t + n > blk_lo) || (ignore != 0 && t < 2);
            if (MODE != FM_COMP) {
                // plain FP64 sum over the tile, folded into the running sum with Kahan
                double tx = 0., ty = 0., tz = 0., d0 = 0., d1 = 0., d2 = 0.;
                if (check)
                    pair_tile<MODE, true>(tile, n, t, i, ignore, gx, gy, gz, soft2, tx, ty, tz, d0, d1, d2,
                                          c15, c1875);
                else
                    pair_tile<MODE, false>(tile, n, t, i, ignore, gx, gy, gz, soft2, tx, ty, tz, d0, d1, d2,
                                           c15, c1875);
                kahan_add(tx, sx, cx);
                kahan_add(ty, sy, cy);
                kahan_add(tz, sz, cz);
            } else {
                if (check)
                    pair_tile<MODE, true>(tile, n, t, i, ignore, gx, gy, gz, soft2, sx, sy, sz, cx, cy, cz,
                                          c15, c1875);
                else
                    pair_tile<MODE, false>(tile, n, t, i, ignore, gx, gy, gz, soft2, sx, sy, sz, cx, cy, cz,
                                           c15, c1875);
            }
        }
    }
    if (live) {
        double* p = partial + (size_t)by * 6 * pstride;
        p[0 * pstride + i] = sx;
        p[1 * pstride + i] = sy;
        p[2 * pstride + i] = sz;
        p[3 * pstride + i] = cx;
        p[4 * pstride + i] = cy;
        p[5 * pstride + i] = cz;
    }
}

// Four wavefronts per SIMD (128 VGPRs, no spills in the pair loop) measured
// faster than eight on gfx950; at N=65536 the grid is 256 target blocks x 8
// source chunks.
template <int MODE, class GBS>
__global__ __launch_bounds__(kFast) __attribute__((amdgpu_waves_per_eu(RB_FAST_WAVES, RB_FAST_WAVES))) void k_direct_fast(
    const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
    const double* __restrict__ m, int n_recv, int j_begin, int j_end, int chunk, int ignore, double soft2,
    GBS gbs, double* __restrict__ partial, int pstride) {
    __shared__ double4 tile[kFast];
    direct_fast_block<MODE>(x, y, z, m, n_recv, j_begin, j_end, chunk, ignore, soft2, gbs, partial, pstride,
                            (int)blockIdx.x, (int)blockIdx.y, tile);
}

// Sum the chunk partials in chunk order (Kahan), apply -G and write (or add to)
// the acceleration.  ignore==2 zeroes particle 0 (it feels nothing).  With
// kd.on, the leapfrog's kick and closing drift follow in the same pass
// (kick_store), which is safe because every read of the positions has finished.
__device__ __forceinline__ void reduce_one(const double* __restrict__ partial, int pstride, int nchunk, int i,
                                           double negG, int accumulate, int ignore, double* __restrict__ ax,
                                           double* __restrict__ ay, double* __restrict__ az, const KickDrift& kd) {
    // Per component, chunk by chunk: the chunk's sum, then its carry with the
    // sign flipped, Kahan-added in chunk order.  The loads of eight chunks are
    // issued before their additions, so their latencies overlap.
    const KickState ks = kick_load(kd, i);
    double s[3] = {0., 0., 0.}, k[3] = {0., 0., 0.};
    constexpr int B = 8;
    int q = 0;
    for (; q + B <= nchunk; q += B) {
        double v[B][6];
#pragma unroll
        for (int u = 0; u < B; u++) {
            const double* p = partial + (size_t)(q + u) * 6 * pstride + i;
#pragma unroll
            for (int f = 0; f < 6; f++) v[u][f] = p[(size_t)f * pstride];
        }
#pragma unroll
        for (int u = 0; u < B; u++) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                kahan_add(v[u][c], s[c], k[c]);
                kahan_add(-v[u][c + 3], s[c], k[c]);
            }
        }
    }
    for (; q < nchunk; q++) {
        const double* p = partial + (size_t)q * 6 * pstride + i;
        for (int c = 0; c < 3; c++) {
            kahan_add(p[(size_t)c * pstride], s[c], k[c]);
            kahan_add(-p[(size_t)(c + 3) * pstride], s[c], k[c]);
        }
    }
    double out[3];
    for (int c = 0; c < 3; c++) out[c] = negG * s[c];
    if (ignore == 2 && i == 0) out[0] = out[1] = out[2] = 0.;
    if (accumulate) {
        out[0] = ax[i] + out[0];
        out[1] = ay[i] + out[1];
        out[2] = az[i] + out[2];
    }
    ax[i] = out[0];
    ay[i] = out[1];
    az[i] = out[2];
    kick_store(kd, i, ks, out[0], out[1], out[2]);
}

__global__ void k_reduce(const double* __restrict__ partial, int pstride, int nchunk, int n_recv, double negG,
                         int accumulate, int ignore, double* __restrict__ ax, double* __restrict__ ay,
                         double* __restrict__ az, KickDrift kd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_recv) return;
    reduce_one(partial, pstride, nchunk, i, negG, accumulate, ignore, ax, ay, az, kd);
}

// The same kick and drift after a kernel that writes the accelerations itself.
__global__ void k_kick_drift(const double* __restrict__ ax, const double* __restrict__ ay,
                             const double* __restrict__ az, int n, KickDrift kd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    kick_store(kd, i, kick_load(kd, i), ax[i], ay[i], az[i]);
}

// The positions before an opening drift that was taken ahead.
__global__ void k_undo_drift(double* __restrict__ x, double* __restrict__ y, double* __restrict__ z,
                             const double* __restrict__ back, size_t stride, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    x[i] = back[i];
    y[i] = back[stride + i];
    z[i] = back[2 * stride + i];
}

__global__ void k_zero3(double* __restrict__ a, double* __restrict__ b, double* __restrict__ c, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = b[i] = c[i] = 0.;
}

// ---------------------------------------------------------------- many simulations per launch
// One order-2 leapfrog step with direct gravity (no ghost boxes, no test
// particles, nothing ignored) for a batch of independent simulations in three
// launches: drift, pair workgroups of every simulation, then reduction with
// the kick and closing drift.  Each simulation keeps its own chunking
// (pick_chunks of its own N), so its bits are those of stepping it alone.
__global__ __launch_bounds__(256) void k_seg_drift(const SegJob* __restrict__ jobs, const SegRange* __restrict__ rg) {
    const SegRange R = rg[blockIdx.x];
    const SegJob J = jobs[R.job];
    const int i = R.first + (int)threadIdx.x;
    if (i >= J.n) return;
    J.x[i] += J.drift * J.vx[i];
    J.y[i] += J.drift * J.vy[i];
    J.z[i] += J.drift * J.vz[i];
}

__global__ __launch_bounds__(kFast) __attribute__((amdgpu_waves_per_eu(RB_FAST_WAVES, RB_FAST_WAVES))) void k_seg_direct(
    const SegJob* __restrict__ jobs, const SegTile* __restrict__ tiles) {
    __shared__ double4 tile[kFast];
    const SegTile T = tiles[blockIdx.x];
    const SegJob J = jobs[T.job];
    switch (J.mode) {
        case FM_FP64:
            direct_fast_block<FM_FP64>(J.x, J.y, J.z, J.m, J.n, 0, J.n, J.chunk, 0, J.soft2, GBZero{}, J.partial, J.n,
                                       T.bx, T.by, tile);
            break;
        case FM_SPLIT:
            direct_fast_block<FM_SPLIT>(J.x, J.y, J.z, J.m, J.n, 0, J.n, J.chunk, 0, J.soft2, GBZero{}, J.partial,
                                        J.n, T.bx, T.by, tile);
            break;
        default:
            direct_fast_block<FM_COMP>(J.x, J.y, J.z, J.m, J.n, 0, J.n, J.chunk, 0, J.soft2, GBZero{}, J.partial, J.n,
                                       T.bx, T.by, tile);
            break;
    }
}

__global__ __launch_bounds__(256) void k_seg_reduce(const SegJob* __restrict__ jobs, const SegRange* __restrict__ rg) {
    const SegRange R = rg[blockIdx.x];
    const SegJob J = jobs[R.job];
    const int i = R.first + (int)threadIdx.x;
    if (i >= J.n) return;
    const KickDrift kd{J.x, J.y, J.z, J.vx, J.vy, J.vz, J.kick, J.drift, 1, nullptr, 0};
    reduce_one(J.partial, J.n, J.nchunk, i, J.negG, 0, 0, J.ax, J.ay, J.az, kd);
}

// ---------------------------------------------------------------- symmetric pair kernel
// Newton's third law, as the reference's serial build uses it (gravity.c:195-214
// visits each pair once and adds the term to both bodies): each unordered pair
// of bodies in different superblocks is evaluated once.  The bodies are cut
// into superblocks of kSymSB; a workgroup takes one pair of superblocks A < B
// (a task).  Its 4 wavefronts hold the targets of A, SYM_TPL per lane, in
// registers; the sources of B stream through LDS 64 at a time (a J-block),
// and lane k evaluates source (k - s) & 63 at step s, so the 64 lanes see 64
// different sources at once.  The source-side sum travels with its source:
// after each step the three accumulators are rotated one lane over the whole
// wavefront (DPP wave_ror:1), and after 64 steps every lane again holds the
// sum of the source it started with.  Per unordered pair: the FP64 r^-3 of
// the fast mode (or the split-precision one) once, two mass products, three
// fused multiply-adds on each side; per step the rotation adds six moves.
//
// Outputs, all in fixed order (the results are deterministic):
//   ipart[t][p][c][SB]  target-side sums of part p of the launch's task t (targets of A, sources of B)
//   jpart[t][c][SB]  source-side sums of the launch's task t (bodies of B, all targets of A)
//                    with the sign of the term for A's bodies: S_j = -jpart
//   dpart[d][6][N]   the one-sided sums within each superblock, 256 sources each (direct_fast_block)
// and k_sym_reduce adds, per body, the partials of every superblock in
// ascending order with Kahan compensation.
//
// ipart and jpart grow with the square of the body count (98 KB per task in
// COMPENSATED gravity: 1.9 GB at 200000 bodies), so beyond a limit the tasks run in
// several launches, in task order, each followed by a reduction that carries the
// running sums of every body on to the next: the same additions in the same order.
#ifndef RB_SYM_TPL
#define RB_SYM_TPL 4
#endif
static constexpr int kSymTPL = RB_SYM_TPL;           // targets per lane
static constexpr int kSymSB = 4 * 64 * kSymTPL;       // bodies per superblock
static constexpr int kSymJB = 64;                     // sources per J-block
static constexpr int kSymMinN = 8192;                 // below: the one-sided kernel
static constexpr size_t kSymMaxN = (size_t)kSymSB << 14;   // above: the same (task numbers in 32 bits)
// Partial sums in memory at a time.  Several launches come from about 126000 bodies
// (COMPENSATED: 88000), all but the last of at least 21 rounds of the chip.
static constexpr size_t kSymPartials = (size_t)512 << 20;
static constexpr int kSymDiag = kSymSB / kFast;       // source tiles of a superblock (one-sided pairs)

// Lane k receives lane k-1's value, lane 0 lane 63's (DPP wave_ror:1).
__device__ __forceinline__ double dpp_ror1(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x13C, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x13C, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// Tasks row by row: (0,1) (0,2) .. (0,nsb-1) (1,2) ..
__host__ __device__ __forceinline__ int sym_task(int A, int B, int nsb) {
    return A * nsb - A * (A + 1) / 2 + (B - A - 1);
}

// The pair (A, B) of task t: the root of the row starts' quadratic, corrected in
// integers.  Formed by every workgroup (a few hundred cycles of a 14 us part) and
// not read from a list: a list would share its memory with the partial sums of the
// other paths, or have to be kept in step with them.
__host__ __device__ __forceinline__ int2 sym_pair(int t, int nsb) {
    const double q = 2. * nsb - 1.;
    int A = (int)((q - sqrt(q * q - 8. * t)) * 0.5);
    A = A < 0 ? 0 : (A > nsb - 2 ? nsb - 2 : A);
    while (A > 0 && sym_task(A, A + 1, nsb) > t) A--;
    while (A < nsb - 2 && sym_task(A + 1, A + 2, nsb) <= t) A++;
    return make_int2(A, A + 1 + t - sym_task(A, A + 1, nsb));
}

// Sums of three components; COMPENSATED gravity carries their Kahan corrections.
template <int MODE>
struct Sum3 {
    double x = 0., y = 0., z = 0.;
    __device__ __forceinline__ void add(double w, double dx, double dy, double dz) {
        x = fma(w, dx, x);
        y = fma(w, dy, y);
        z = fma(w, dz, z);
    }
    __device__ __forceinline__ void rotate() {
        x = dpp_ror1(x);
        y = dpp_ror1(y);
        z = dpp_ror1(z);
    }
};
template <>
struct Sum3<FM_COMP> {
    double x = 0., y = 0., z = 0., cx = 0., cy = 0., cz = 0.;
    __device__ __forceinline__ void add(double w, double dx, double dy, double dz) {
        kahan_fma(w, dx, x, cx);
        kahan_fma(w, dy, y, cy);
        kahan_fma(w, dz, z, cz);
    }
    __device__ __forceinline__ void rotate() {
        x = dpp_ror1(x);
        y = dpp_ror1(y);
        z = dpp_ror1(z);
        cx = dpp_ror1(cx);
        cy = dpp_ror1(cy);
        cz = dpp_ror1(cz);
    }
};

// One J-block's 64 steps for the lane's targets.  CHECK: the J-block is the
// last, ragged one of the bodies (its first jlim sources exist).
template <int MODE, bool CHECK>
__device__ __forceinline__ void sym_jblock(const double4* __restrict__ src, int k, int jlim, const double* tx,
                                           const double* ty, const double* tz, const double* tm, double soft2,
                                           double c15, double c1875, Sum3<MODE>* b, Sum3<MODE>& j) {
#pragma unroll MODE == FM_COMP ? 1 : 4
    for (int s = 0; s < kSymJB; s++) {
        const int idx = (k - s) & (kSymJB - 1);     // the source's index in the J-block
        const double4 sj = src[k + kSymJB - s];
#pragma unroll
        for (int q = 0; q < kSymTPL; q++) {
            const double dx = tx[q] - sj.x;
            const double dy = ty[q] - sj.y;
            const double dz = tz[q] - sj.z;
            const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, soft2)));
            double wr;
            if (MODE == FM_SPLIT) {
                const double yv = (double)__builtin_amdgcn_rsqf((float)r2);
                wr = yv * yv * yv;
            } else {
                wr = rinv3_fp64(r2, c15, c1875);
            }
            if (CHECK && idx >= jlim) wr = 0.;
            b[q].add(wr * sj.w, dx, dy, dz);
            j.add(wr * tm[q], dx, dy, dz);
        }
        j.rotate();
    }
}

// Workgroups [0, ntasks * split): part p of task t0 + t, (A, B), takes 1/split of B's
// J-blocks.  One workgroup per task leaves most of the chip idle below ~40000
// bodies (8192 bodies are 28 tasks for 256 CUs), so sym_split cuts the tasks.
// The remaining workgroups (of the first launch) evaluate the pairs inside the superblocks
// (one-sided, 256 targets x 256 sources each); they are short and fill the
// launch's tail.  One launch for full and ragged tasks alike (10007 bodies took
// 237 + 221 us in two).
template <int MODE>
__global__ __launch_bounds__(256) void k_direct_sym(const double* __restrict__ x, const double* __restrict__ y,
                                                    const double* __restrict__ z, const double* __restrict__ m,
                                                    int N, int nsb, int t0, int ntasks, int split, double soft2,
                                                    double* __restrict__ ipart, double* __restrict__ jpart,
                                                    double* __restrict__ dpart) {
    // J-block sources (x, y, z, m), double-buffered, each stored twice in a
    // row so that lane k reads entry k + 64 - s at step s without wrapping
    __shared__ double4 jt[2][2 * kSymJB];
    constexpr bool COMP = MODE == FM_COMP;
    constexpr int NC = COMP ? 6 : 3;               // values per body in the partials
    __shared__ double jred[2][4][NC][kSymJB];      // per-wave source sums of a J-block
    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= ntasks * split) {
        static_assert(sizeof(jt) >= sizeof(double4) * kFast, "the one-sided tile fits the J-block buffers");
        const int u = (int)blockIdx.x - ntasks * split;
        const int bx = u / kSymDiag;
        const int j0 = bx * kFast / kSymSB * kSymSB;
        direct_fast_block<MODE>(x, y, z, m, N, j0, min(N, j0 + kSymSB), kFast, 0, soft2, GBZero{}, dpart, N, bx,
                                u % kSymDiag, &jt[0][0]);
        return;
    }
    const int t = (int)blockIdx.x % ntasks;
    const int part = (int)blockIdx.x / ntasks;
    const int2 tk = sym_pair(t0 + t, nsb);
    const int A = __builtin_amdgcn_readfirstlane(tk.x), B = __builtin_amdgcn_readfirstlane(tk.y);
    const int w = tid >> 6, k = tid & 63;
    // targets of this lane (A < B: never the ragged superblock)
    double tx[kSymTPL], ty[kSymTPL], tz[kSymTPL], tm[kSymTPL];
    Sum3<MODE> sum[kSymTPL];
#pragma unroll
    for (int q = 0; q < kSymTPL; q++) {
        const int i = A * kSymSB + w * 64 * kSymTPL + q * 64 + k;
        tx[q] = x[i];
        ty[q] = y[i];
        tz[q] = z[i];
        tm[q] = m[i];
    }
    const int jbase = B * kSymSB;
    constexpr int NJB = kSymSB / kSymJB;
    const int jb0 = part * NJB / split;
    const int jb1 = min((part + 1) * NJB / split, (N - jbase + kSymJB - 1) / kSymJB);
    auto source = [&](int jb) {
        const int j = jbase + jb * kSymJB + tid;
        return jb < jb1 && j < N ? make_double4(x[j], y[j], z[j], m[j]) : make_double4(0., 0., 0., 0.);
    };
    // prologue: the first J-block into LDS, the second into registers
    double4 nxt = make_double4(0., 0., 0., 0.);
    if (tid < kSymJB) {
        const double4 v0 = source(jb0);
        jt[jb0 & 1][tid] = v0;
        jt[jb0 & 1][tid + kSymJB] = v0;
        nxt = source(jb0 + 1);
    }
    // source sums of a finished J-block: the four waves' in order
    auto flush = [&](int jb) {
        if (w >= 3) return;
        const double* r = &jred[jb & 1][0][w][k];
        constexpr int W = NC * kSymJB;             // from wave to wave
        double* out = jpart + ((size_t)t * NC + w) * kSymSB + jb * kSymJB + k;
        if constexpr (COMP) {
            double v = r[0], c = r[3 * kSymJB];
#pragma unroll
            for (int q = 1; q < 4; q++) {
                kahan_add(r[q * W], v, c);
                kahan_add(-r[q * W + 3 * kSymJB], v, c);
            }
            out[0] = v;
            out[3 * kSymSB] = c;
        } else {
            out[0] = ((r[0] + r[W]) + r[2 * W]) + r[3 * W];
        }
    };
    const double c15 = vreg_const(1.5);
    const double c1875 = vreg_const(1.875);
    for (int jb = jb0; jb < jb1; jb++) {
        __syncthreads();
        if (jb > jb0) flush(jb - 1);
        if (tid < kSymJB) {
            jt[(jb + 1) & 1][tid] = nxt;
            jt[(jb + 1) & 1][tid + kSymJB] = nxt;
            nxt = source(jb + 2);
        }
        // FP64 and split: the J-block's sums apart, then added to the running ones
        Sum3<MODE> part3[kSymTPL], src3;
        Sum3<MODE>* b = COMP ? sum : part3;
        const int jlim = N - (jbase + jb * kSymJB);
        if (jlim >= kSymJB)
            sym_jblock<MODE, false>(jt[jb & 1], k, jlim, tx, ty, tz, tm, soft2, c15, c1875, b, src3);
        else
            sym_jblock<MODE, true>(jt[jb & 1], k, jlim, tx, ty, tz, tm, soft2, c15, c1875, b, src3);
        if constexpr (!COMP) {
#pragma unroll
            for (int q = 0; q < kSymTPL; q++) {
                sum[q].x += part3[q].x;
                sum[q].y += part3[q].y;
                sum[q].z += part3[q].z;
            }
        }
        double* jr = &jred[jb & 1][w][0][k];
        jr[0] = src3.x;
        jr[kSymJB] = src3.y;
        jr[2 * kSymJB] = src3.z;
        if constexpr (COMP) {
            jr[3 * kSymJB] = src3.cx;
            jr[4 * kSymJB] = src3.cy;
            jr[5 * kSymJB] = src3.cz;
        }
    }
    __syncthreads();
    if (jb1 > jb0) flush(jb1 - 1);
#pragma unroll
    for (int q = 0; q < kSymTPL; q++) {
        const int li = w * 64 * kSymTPL + q * 64 + k;
        double* p = ipart + ((size_t)t * split + part) * NC * kSymSB + li;
        p[0] = sum[q].x;
        p[kSymSB] = sum[q].y;
        p[2 * kSymSB] = sum[q].z;
        if constexpr (COMP) {
            p[3 * kSymSB] = sum[q].cx;
            p[4 * kSymSB] = sum[q].cy;
            p[5 * kSymSB] = sum[q].cz;
        }
    }
}

// Adds the two-term number (hi, lo) to (s, c); exact in s whichever is larger,
// where a Kahan addition rounds when the addend is the larger one.
__device__ __forceinline__ void two_add(double hi, double lo, double& s, double& c) {
    const double t = s + hi;
    const double b = t - s;
    c += ((s - (t - b)) + (hi - b)) + lo;
    s = t;
}

// Per body: the partials of every superblock in ascending order (Kahan), then
// -G and the fused kick and drift as in the one-sided reduction.  A workgroup
// takes 64 bodies of one superblock; its four wavefronts each sum a quarter of
// the partials (the loads of eight in flight), and the first adds the four
// sums with their carries in order, as two-term numbers (any of the four can be the
// largest).  A body of superblock X has X source-side sums, kSymDiag one-sided
// sums with their carries, and `split` target-side sums per later superblock; CARRY: the
// others come with carries too (COMPENSATED).
//
// ROUNDS: after the launch of tasks t0 .. t1 - 1 of ntasks.  Tasks are numbered by rows
// (A, A+1) (A, A+2) .., so a body's partials come in ascending order from launch to
// launch; each wavefront continues its quarter from `state` (6 sums and carries of
// N bodies per quarter), and the last launch's reduction ends as the only one does.
template <bool CARRY, bool ROUNDS>
__global__ __launch_bounds__(256) void k_sym_reduce(const double* __restrict__ ipart,
                                                    const double* __restrict__ jpart,
                                                    const double* __restrict__ dpart, int N, int nsb, int split,
                                                    int t0, int t1, int ntasks, double* __restrict__ state,
                                                    double negG, double* __restrict__ ax, double* __restrict__ ay,
                                                    double* __restrict__ az, KickDrift kd) {
    __shared__ double sums[4][6][64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int first = (int)blockIdx.x * 64;
    const int i = first + lane;
    const int X = first / kSymSB, loc = first % kSymSB;
    const int ii = min(i, N - 1) - first;          // lanes past the end read the last body's
    const bool last = !ROUNDS || t1 == ntasks;
    if (!ROUNDS) t0 = 0;
    const KickState ks = w == 0 && last ? kick_load(kd, min(i, N - 1)) : KickState{};
    double s[3] = {0., 0., 0.}, c[3] = {0., 0., 0.};
    constexpr int PER = CARRY ? 2 : 1;             // entries per partial sum: itself, its carry
    const int total = PER * X + 2 * kSymDiag + PER * (nsb - 1 - X) * split;
    int e0 = total * w / 4, e1 = total * (w + 1) / 4;
    if (ROUNDS) {
        // entries of superblock X that the tasks before t complete (the one-sided
        // ones count with the last source-side entry)
        auto before = [&](int t) {
            if (t == 0) return 0;
            if (t == ntasks) return total;
            const int2 next = sym_pair(t, nsb);
            if (next.x < X) return PER * (next.x + (X < next.y ? 1 : 0));
            return next.x > X ? total : PER * X + 2 * kSymDiag + PER * (next.y - X - 1) * split;
        };
        const int b0 = before(t0), b1 = before(t1);
        if (b0 > e0 && i < N) {
#pragma unroll
            for (int f = 0; f < 3; f++) {
                s[f] = state[(size_t)(6 * w + f) * N + i];
                c[f] = state[(size_t)(6 * w + 3 + f) * N + i];
            }
        }
        e0 = max(e0, b0);
        e1 = min(e1, b1);
    }
    // entry e: base pointer of its first component, component stride, sign
    auto load = [&](int e, double* v) {
        const double* p;
        size_t stride = kSymSB;
        double sign = 1.;
        if (e < PER * X) {
            const int carry = e % PER;
            p = jpart + ((size_t)(sym_task(e / PER, X, nsb) - t0) * 3 * PER + 3 * carry) * kSymSB + loc;
            sign = carry ? 1. : -1.;
        } else if (e < PER * X + 2 * kSymDiag) {
            const int q = e - PER * X;
            p = dpart + ((size_t)(q >> 1) * 6 + (q & 1 ? 3 : 0)) * N + first;
            stride = N;
            sign = q & 1 ? -1. : 1.;
        } else {
            const int q = (e - PER * X - 2 * kSymDiag) / PER, carry = (e - PER * X - 2 * kSymDiag) % PER;
            const size_t part = (size_t)(sym_task(X, X + 1 + q / split, nsb) - t0) * split + q % split;
            p = ipart + (part * 3 * PER + 3 * carry) * kSymSB + loc;
            sign = carry ? -1. : 1.;
        }
#pragma unroll
        for (int f = 0; f < 3; f++) v[f] = sign * p[f * stride + ii];
    };
    constexpr int BATCH = 8;
    int e = e0;
    for (; e + BATCH <= e1; e += BATCH) {
        double v[BATCH][3];
#pragma unroll
        for (int u = 0; u < BATCH; u++) load(e + u, v[u]);
#pragma unroll
        for (int u = 0; u < BATCH; u++)
#pragma unroll
            for (int f = 0; f < 3; f++) kahan_add(v[u][f], s[f], c[f]);
    }
    for (; e < e1; e++) {
        double v[3];
        load(e, v);
#pragma unroll
        for (int f = 0; f < 3; f++) kahan_add(v[f], s[f], c[f]);
    }
    if (!last) {
        if (e0 >= e1 || i >= N) return;
#pragma unroll
        for (int f = 0; f < 3; f++) {
            state[(size_t)(6 * w + f) * N + i] = s[f];
            state[(size_t)(6 * w + 3 + f) * N + i] = c[f];
        }
        return;
    }
#pragma unroll
    for (int f = 0; f < 3; f++) {
        sums[w][f][lane] = s[f];
        sums[w][f + 3][lane] = c[f];
    }
    __syncthreads();
    if (w != 0 || i >= N) return;
#pragma unroll
    for (int f = 0; f < 3; f++) {
        c[f] = -c[f];
#pragma unroll
        for (int g = 1; g < 4; g++) two_add(sums[g][f][lane], -sums[g][f + 3][lane], s[f], c[f]);
        s[f] += c[f];
    }
    const double o0 = negG * s[0], o1 = negG * s[1], o2 = negG * s[2];
    ax[i] = o0;
    ay[i] = o1;
    az[i] = o2;
    kick_store(kd, i, ks, o0, o1, o2);
}

// Superblock layout of the symmetric path for N bodies.
struct SymPlan {
    int nsb = 0;          // superblocks
    int ntasks = 0;       // superblock pairs A < B
    int split = 1;        // workgroups per task
    int round = 0;        // tasks per launch
    size_t ipart_off = 0, jpart_off = 0, dpart_off = 0, state_off = 0, bytes = 0;   // workspace layout (bytes)
};

// Workgroups per task: the pair loop of a task takes about 223 us on a CU (its
// SIMDs are issue-bound from one wavefront on, so two workgroups on a CU take twice
// that), and every part writes and the reduction reads 24 KB of target-side
// sums, about 12 ns of the chip's bandwidth.  The split with the least
// modelled time; measured (leapfrog steps, FP64): 8192 bodies 59 us (286
// unsplit), 10007 75 (526), 20000 210 (566), 24576 301 (513), 49152 965 (1200).
static constexpr int kCUs = 256;
static int sym_split(int ntasks) {
    constexpr double kTask = 223., kPart = 0.012;   // us
    int best = 1;
    double least = 1e300;
    for (int s = 1; s <= kSymSB / kSymJB; s *= 2) {
        const long parts = (long)ntasks * s;
        const double t = (parts + kCUs - 1) / kCUs * kTask / s + parts * kPart;
        if (t < least) {
            least = t;
            best = s;
        }
    }
    return best;
}

// The plan whose workspace stays within `limit` bytes, or the least one if none
// does: launches of a whole number of rounds of the chip, at least one (with fewer
// workgroups the one-sided kernels are faster).
static SymPlan sym_plan(int N, bool compensated, size_t limit) {
    SymPlan p;
    p.nsb = (N + kSymSB - 1) / kSymSB;
    p.ntasks = p.nsb * (p.nsb - 1) / 2;
    p.split = sym_split(p.ntasks);
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t part = sizeof(double) * (compensated ? 6 : 3) * (size_t)kSymSB;
    const size_t task = part * (p.split + 1);
    const size_t dpart = up(sizeof(double) * 6 * kSymDiag * (size_t)N);
    const size_t state = up(sizeof(double) * 24 * (size_t)N);
    p.round = p.ntasks;
    if (task * p.ntasks > kSymPartials || task * p.ntasks + dpart > limit) {
        const size_t unit = kCUs / p.split;
        const size_t room = limit > dpart + state ? std::min(limit - dpart - state, kSymPartials) : 0;
        const size_t fit = std::max(room / task / unit, (size_t)1) * unit;
        if (fit < (size_t)p.ntasks) p.round = (int)fit;
    }
    p.jpart_off = part * p.split * p.round;                    // multiples of 24 KB
    p.dpart_off = p.jpart_off + part * p.round;
    p.state_off = p.dpart_off + dpart;
    p.bytes = p.state_off + (p.round < p.ntasks ? state : 0);
    return p;
}

// Number of source chunks for the fast modes: chunks no shorter than kMinChunk
// sources (short chunks keep the time of one step small for N of a few
// thousand, where a single workgroup's chunk sets the kernel's duration), and
// at most max_chunks of them, which the workspaces are sized for.
static constexpr int kMinChunk = 32;
static_assert(kFast % kMinChunk == 0, "chunks tile the LDS tile");
static int round_chunk(int c) { return ((c + kMinChunk - 1) / kMinChunk) * kMinChunk; }
static int max_chunks(int n_recv, int n_src, int ngb) {
    const int blocks_x = (n_recv + kFast - 1) / kFast;
    const int target_blocks = 2048 * 256 / kFast;
    int s = (target_blocks + blocks_x - 1) / blocks_x;
    int max_s = (n_src * ngb) / kMinChunk;
    if (max_s < 1) max_s = 1;
    if (s > max_s) s = max_s;
    if (s > 64) s = 64;
    if (s < 1) s = 1;
    return s;
}
// max_chunks rounds up, so that at many sizes a few workgroups more than the 2048
// of two full rounds (four wavefronts on every SIMD) start a third: the last chunk's.
// One chunk fewer then, if that chunk is nearly a full one (a short one costs
// little) and the others do not grow by more than the third round takes, about an
// eighth.  Measured, us with and without the chunk, targets / sources, FP64: last
// chunk 0.71 to 1 of the others, which grow by 4 to 10 %: 27548 / 27548 520 and 499,
// 30011 / 20011 489 and 469, 34972 844 and 796, 40348 1108 and 1060, 47772 1512 and 1496;
// growth 12 %: 58268 2241 and 2268; last chunk 0.1 to 0.65: 13468 147 and 154, 18332 /
// 9166 133 and 143, 21660 / 10830 177 and 187; chunks below 700 sources, whose lengths
// round up by more: 25105 / 6705 132 and 140, 16628 / 16245 195 and 208.  With half a workgroup per CU or more left
// over the third round is worth its chunks (65000 / 20000: 930 with 254 x 9, 942 with
// 254 x 8).
static int pick_chunks(int n_recv, int n_src, int ngb) {
    const int s = max_chunks(n_recv, n_src, ngb);
    const long blocks = (n_recv + kFast - 1) / kFast;
    if (s <= 2 || blocks * s <= 2048 || blocks * s > 2048 + 128) return s;
    const int c = round_chunk((n_src + s - 1) / s), longer = round_chunk((n_src + s - 2) / (s - 1));
    const int last = n_src - (s - 1) * c;              // none left if rounding made the chunks longer
    return c >= 700 && 10L * last >= 7L * c && 100L * longer <= 112L * c ? s - 1 : s;
}

static size_t workspace_bytes(int n, int nchunk) { return sizeof(double) * 6 * (size_t)n * (size_t)nchunk; }

// The chunking a simulation of n bodies uses when stepped alone (launch_fast).
void seg_plan(int n, int* chunk, int* used, size_t* workspace) {
    const int nchunk = pick_chunks(n, n, 1);
    const int c = round_chunk((n + nchunk - 1) / nchunk);
    *chunk = c;
    *used = n > 0 ? (n + c - 1) / c : 1;
    *workspace = workspace_bytes(n, nchunk) + 256;
}

int seg_tiles_of(int n, int used) { return ((n + kFast - 1) / kFast) * used; }

int seg_step_launch(const SegJob* jobs, const SegRange* ranges, int nranges, const SegTile* tiles, int ntiles,
                    hipStream_t st) {
    if (nranges == 0) return 0;
    hipLaunchKernelGGL(k_seg_drift, dim3(nranges), dim3(256), 0, st, jobs, ranges);
    hipLaunchKernelGGL(k_seg_direct, dim3(ntiles), dim3(kFast), 0, st, jobs, tiles);
    hipLaunchKernelGGL(k_seg_reduce, dim3(nranges), dim3(256), 0, st, jobs, ranges);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int seg_fast_mode(int precision, int compensated) {
    return compensated ? FM_COMP : (precision == REB_AMD_PRECISION_SPLIT ? FM_SPLIT : FM_FP64);
}

// Whether a simulation of N bodies, all active, without ghost boxes or
// ignored terms, takes the symmetric path in this precision and gravity, and
// the workspace it then needs.
bool gravity_symmetric_path(size_t N, int precision) {
    return precision != REB_AMD_PRECISION_EXACT && N >= (size_t)kSymMinN && N <= kSymMaxN;
}
size_t gravity_symmetric_bytes(size_t N, bool compensated, size_t limit) {
    return sym_plan((int)N, compensated, limit).bytes;
}

// Ordered pairs inside the superblocks (evaluated one-sided): sum over superblocks of n_A^2, self pairs included.
static double sym_diag_pairs(int N) {
    const int full = N / kSymSB, rest = N % kSymSB;
    return (double)full * kSymSB * kSymSB + (double)rest * rest;
}

// One force evaluation on the symmetric path: all pairs (events around these
// launches), then the per-body reduction with the fused kick and drift.
static int sym_launch(int mode, const double* x, const double* y, const double* z, const double* m, double* ax,
                      double* ay, double* az, int N, double G, double soft2, const SymPlan& plan, char* base,
                      hipStream_t st, hipEvent_t* ev, const KickDrift& kd) {
    double* ipart = reinterpret_cast<double*>(base + plan.ipart_off);
    double* jpart = reinterpret_cast<double*>(base + plan.jpart_off);
    double* dpart = reinterpret_cast<double*>(base + plan.dpart_off);
    double* state = reinterpret_cast<double*>(base + plan.state_off);
    const auto pairs = mode == FM_COMP    ? k_direct_sym<FM_COMP>
                       : mode == FM_SPLIT ? k_direct_sym<FM_SPLIT>
                                          : k_direct_sym<FM_FP64>;
    const bool rounds = plan.round < plan.ntasks;
    const auto reduce = mode == FM_COMP ? (rounds ? k_sym_reduce<true, true> : k_sym_reduce<true, false>)
                                        : (rounds ? k_sym_reduce<false, true> : k_sym_reduce<false, false>);
    if (ev) (void)hipEventRecord(ev[0], st);
    for (int t0 = 0; t0 < plan.ntasks; t0 += plan.round) {
        const int t1 = std::min(t0 + plan.round, plan.ntasks);
        const int inner = t0 == 0 ? (N + kFast - 1) / kFast * kSymDiag : 0;
        hipLaunchKernelGGL(pairs, dim3((t1 - t0) * plan.split + inner), dim3(256), 0, st, x, y, z, m, N, plan.nsb, t0,
                           t1 - t0, plan.split, soft2, ipart, jpart, dpart);
        if (ev && t1 == plan.ntasks) (void)hipEventRecord(ev[1], st);
        hipLaunchKernelGGL(reduce, dim3((N + 63) / 64), dim3(256), 0, st, ipart, jpart, dpart, N, plan.nsb, plan.split,
                           t0, t1, plan.ntasks, state, -G, ax, ay, az, kd);
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// Launch one fast-mode pass: targets [0,n_recv) feel sources [j_begin,j_end).
static int launch_fast(int mode, const double* x, const double* y, const double* z, const double* m, int n_recv,
                       int j_begin, int j_end, int ignore, double G, double soft2, const GBList& gl,
                       double* partial, int nchunk, int accumulate, double* ax, double* ay, double* az,
                       hipStream_t st, hipEvent_t* ev, const KickDrift& kd) {
    const int nsrc = j_end - j_begin;
    const int chunk = round_chunk((nsrc + nchunk - 1) / nchunk);
    const int used = nsrc > 0 ? (nsrc + chunk - 1) / chunk : 1;
    dim3 grid((n_recv + kFast - 1) / kFast, used);
    if (ev) (void)hipEventRecord(ev[0], st);
    auto pairs = [&](auto gbs) {
        using GBS = decltype(gbs);
        const auto k = mode == FM_FP64    ? k_direct_fast<FM_FP64, GBS>
                       : mode == FM_SPLIT ? k_direct_fast<FM_SPLIT, GBS>
                                          : k_direct_fast<FM_COMP, GBS>;
        hipLaunchKernelGGL(k, grid, dim3(kFast), 0, st, x, y, z, m, n_recv, j_begin, j_end, chunk, ignore, soft2, gbs,
                           partial, n_recv);
    };
    if (gl.zero())
        pairs(GBZero{});
    else
        pairs(GBFromList{gl});
    if (ev) (void)hipEventRecord(ev[1], st);
    hipLaunchKernelGGL(k_reduce, dim3((n_recv + 255) / 256), dim3(256), 0, st, partial, n_recv, used, n_recv, -G,
                       accumulate, ignore, ax, ay, az, kd);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// Shared dispatch for the simulation path and the raw entry point.
static int direct_dispatch(const double* x, const double* y, const double* z, const double* m, double* ax,
                           double* ay, double* az, int N, int N_active, int tp_type, int ignore, double G,
                           double soft2, int precision, int compensated, const GBList& gl,
                           double* workspace, hipStream_t st, hipEvent_t* ev = nullptr,
                           const KickDrift& kd = KickDrift{}) {
    if (N == 0) return 0;
    const KickDrift none{};
    if (precision == REB_AMD_PRECISION_EXACT) {
        if (ev) (void)hipEventRecord(ev[0], st);
        if (compensated)
            launch_exact<true>(st, x, y, z, m, ax, ay, az, N, N_active, tp_type, ignore, G, soft2, gl);
        else
            launch_exact<false>(st, x, y, z, m, ax, ay, az, N, N_active, tp_type, ignore, G, soft2, gl);
        if (ev) (void)hipEventRecord(ev[1], st);
        if (kd.on) hipLaunchKernelGGL(k_kick_drift, dim3((N + 255) / 256), dim3(256), 0, st, ax, ay, az, N, kd);
        return hipGetLastError() == hipSuccess ? 0 : 1;
    }
    const int mode = compensated ? FM_COMP : (precision == REB_AMD_PRECISION_SPLIT ? FM_SPLIT : FM_FP64);
    const int nchunk = pick_chunks(N, N_active, gl.n);
    int rc = 0;
    const bool second = tp_type && N_active < N;
    if (N_active > 0) {
        rc |= launch_fast(mode, x, y, z, m, N, 0, N_active, ignore, G, soft2, gl, workspace, nchunk, 0, ax, ay, az,
                          st, ev, second ? none : kd);
    } else {
        hipLaunchKernelGGL(k_zero3, dim3((N + 255) / 256), dim3(256), 0, st, ax, ay, az, N);
    }
    if (second) {
        // Active targets also feel the test particles (gravity.c:259-276).
        const int nchunk2 = pick_chunks(N_active, N - N_active, gl.n);
        rc |= launch_fast(mode, x, y, z, m, N_active, N_active, N, ignore, G, soft2, gl, workspace,
                          nchunk2 < nchunk ? nchunk2 : nchunk, 1, ax, ay, az, st, nullptr, none);
    }
    if (kd.on && (second || N_active == 0))
        hipLaunchKernelGGL(k_kick_drift, dim3((N + 255) / 256), dim3(256), 0, st, ax, ay, az, N, kd);
    return rc;
}

// ---------------------------------------------------------------- JACOBI
// gravity.c:108-163, the gravity of the WHFast modified-kick and lazy kernels:
// Jacobi and direct terms with every pair visited once (j = 0..N-1, i = 0..j)
// and added to both bodies, without softening.  The order of the additions to
// each body is the whole definition, so one thread walks the pairs; the
// systems it serves have a few bodies (the WHFast group kernel evaluates the
// same sums for its own systems).
__global__ void k_gravity_jacobi(const double* __restrict__ x, const double* __restrict__ y,
                                 const double* __restrict__ z, const double* __restrict__ m, double* ax, double* ay,
                                 double* az, int N, double G) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    double Rx = 0., Ry = 0., Rz = 0., Mt = 0.;
    for (int j = 0; j < N; j++) {
        ax[j] = 0.;
        ay[j] = 0.;
        az[j] = 0.;
        const double xj = x[j], yj = y[j], zj = z[j], mj = m[j];
        for (int i = 0; i <= j; i++) {
            if (j > 1) {
                const double qx = xj - Rx / Mt;
                const double qy = yj - Ry / Mt;
                const double qz = zj - Rz / Mt;
                const double dr = sqrt(qx * qx + qy * qy + qz * qz);
                const double w = i < j ? -mj : Mt;
                const double pf = G * w / (dr * dr * dr);
                ax[i] += pf * qx;
                ay[i] += pf * qy;
                az[i] += pf * qz;
            }
            if (i != j && (i != 0 || j != 1)) {
                const double dx = x[i] - xj;
                const double dy = y[i] - yj;
                const double dz = z[i] - zj;
                const double dr = sqrt(dx * dx + dy * dy + dz * dz);
                const double pf = G / (dr * dr * dr);
                const double pfi = pf * m[i];
                const double pfj = pf * mj;
                ax[i] -= pfj * dx;
                ay[i] -= pfj * dy;
                az[i] -= pfj * dz;
                ax[j] += pfi * dx;
                ay[j] += pfi * dy;
                az[j] += pfi * dz;
            }
        }
        Rx += mj * xj;
        Ry += mj * yj;
        Rz += mj * zj;
        Mt += mj;
    }
}

// ---------------------------------------------------------------- simulation path
bool gravity_jacobi(struct reb_simulation* r) {
    DeviceState* d = dev_of(r);
    const int N = (int)r->N;
    if (N == 0) return true;
    hipLaunchKernelGGL(k_gravity_jacobi, dim3(1), dim3(64), 0, d->stream, d->field(FX), d->field(FY), d->field(FZ),
                       d->field(FM), d->field(FAX), d->field(FAY), d->field(FAZ), N, r->G);
    return RB_HIP(r, hipGetLastError());
}

bool gravity_zero(struct reb_simulation* r) {
    DeviceState* d = dev_of(r);
    const int N = (int)r->N;
    if (N == 0) return true;
    hipLaunchKernelGGL(k_zero3, dim3((N + 255) / 256), dim3(256), 0, d->stream, d->field(FAX), d->field(FAY),
                       d->field(FAZ), N);
    return RB_HIP(r, hipGetLastError());
}

// Room for the positions that gravity_direct(.., ahead) keeps.  Without it, or
// with limited memory, the step is taken as a single one.
bool gravity_drift_room(struct reb_simulation* r) {
    DeviceState* d = dev_of(r);
    if (d->sym_limit != SIZE_MAX) return false;
    if (d->drift_back.ensure(sizeof(double) * 3 * d->cap)) return true;
    (void)hipGetLastError();
    return false;
}

// Back to the positions before the opening drift that the last step took ahead.
bool gravity_undo_drift(struct reb_simulation* r) {
    DeviceState* d = dev_of(r);
    const int N = (int)r->N;
    hipLaunchKernelGGL(k_undo_drift, dim3((N + 255) / 256), dim3(256), 0, d->stream, d->field(FX), d->field(FY),
                       d->field(FZ), d->drift_back.as<double>(), d->cap, N);
    mark_device_newer(r);
    return RB_HIP(r, hipGetLastError());
}

// kick_drift (optional): {kick dt, drift dt} of a leapfrog step, applied in the
// pass that finishes the accelerations; ahead: and the same drift once more, the
// next step's opening one.
bool gravity_direct(struct reb_simulation* r, bool compensated, const double* kick_drift, bool ahead) {
    DeviceState* d = dev_of(r);
    const int N = (int)r->N;
    if (N == 0) return true;
    const int N_active = (r->N_active == SIZE_MAX) ? N : (int)r->N_active;
    const double soft2 = r->softening * r->softening;
    // Ghost boxes (BASIC only; gravity.c:184-186).  COMPENSATED has none.
    std::vector<struct reb_vec6d> gbv;
    if (compensated)
        gbv.push_back(reb_vec6d{0, 0, 0, 0, 0, 0});
    else
        gbv = ghostboxes(r, r->N_ghost_x, r->N_ghost_y, r->N_ghost_z);
    const int ngb = (int)gbv.size();
    if (ngb > kMaxGB) {
        reb_simulation_error(r, "Too many ghost boxes for direct gravity (at most 125).");
        return false;
    }
    GBList gl;
    gl.n = ngb;
    for (int g = 0; g < ngb; g++) gl.g[g] = GB3{gbv[g].x, gbv[g].y, gbv[g].z};
    hipEvent_t* ev = nullptr;
    if (d->profiling) {
        if (d->kev_used + 2 > d->kev.size()) {
            for (int k = 0; k < 64; k++) {
                hipEvent_t e;
                if (!RB_HIP(r, hipEventCreate(&e))) return false;
                d->kev.push_back(e);
            }
        }
        ev = &d->kev[d->kev_used];
        d->kev_used += 2;
    }
    KickDrift kd{};
    if (kick_drift) {
        kd = KickDrift{d->field(FX), d->field(FY), d->field(FZ), d->field(FVX), d->field(FVY), d->field(FVZ),
                       kick_drift[0], kick_drift[1], ahead ? 2 : 1, d->drift_back.as<double>(), d->cap};
    }
    // Every body active, no ghost boxes, nothing ignored: each pair once
    // (Newton's third law); otherwise the one-sided kernels.
    if (ngb == 1 && N_active == N && r->gravity_ignore_terms == 0 &&
        gravity_symmetric_path((size_t)N, d->precision)) {
        // The tasks go in as many launches as the memory asks for (the same bits);
        // a simulation without room for even the shortest takes the one-sided
        // kernels below.
        for (;;) {
            const SymPlan plan = sym_plan(N, compensated, d->sym_limit);
            if (plan.bytes > d->sym_limit) break;
            if (!d->partial.ensure(plan.bytes)) {
                (void)hipGetLastError();
                d->sym_limit = plan.bytes / 2;
                continue;
            }
            if (d->profiling) d->kpairs += (double)N * (double)N - sym_diag_pairs(N);
            const int rc = sym_launch(seg_fast_mode(d->precision, compensated), d->field(FX), d->field(FY),
                                      d->field(FZ), d->field(FM), d->field(FAX), d->field(FAY), d->field(FAZ), N, r->G,
                                      soft2, plan, static_cast<char*>(d->partial.p), d->stream, ev, kd);
            if (rc) return RB_HIP(r, hipGetLastError());
            return true;
        }
    }
    const int nchunk = pick_chunks(N, N_active, ngb);
    if (!d->partial.ensure(workspace_bytes(N, nchunk) + 256)) {
        reb_simulation_error(r, "Out of device memory for the gravity workspace.");
        return false;
    }
    if (d->profiling) d->kpairs += (double)N * (double)(N - 1);
    int rc = direct_dispatch(d->field(FX), d->field(FY), d->field(FZ), d->field(FM), d->field(FAX), d->field(FAY),
                             d->field(FAZ), N, N_active, r->testparticle_type, (int)r->gravity_ignore_terms, r->G,
                             soft2, d->precision, compensated ? 1 : 0, gl, d->partial.as<double>(), d->stream, ev, kd);
    if (rc) return RB_HIP(r, hipGetLastError());
    return true;
}

// ---------------------------------------------------------------- energy
// tools.c:108-162.  EXACT: the kinetic and potential sums are accumulated in
// the reference's sequential order, so the value is bit-identical: the
// kinetic terms by one wavefront (lanes evaluate 64 terms, lane 0 folds them
// in order); the pair terms of a batch of rows are written in the
// reference's (i, j > i) order by a grid, then one lane folds them in order
// while its wavefront streams the next chunk in.  Otherwise k_energy_tiles.
__global__ __launch_bounds__(64) void k_energy_kin(const double* __restrict__ vx, const double* __restrict__ vy,
                                                   const double* __restrict__ vz, const double* __restrict__ m,
                                                   int N_interact, double* __restrict__ out) {
    __shared__ double terms[64];
    const int lane = threadIdx.x;
    double e_kin = 0.;
    for (int b = 0; b < N_interact; b += 64) {
        const int i = b + lane;
        if (i < N_interact) {
            const double vv = vx[i] * vx[i] + vy[i] * vy[i] + vz[i] * vz[i];
            terms[lane] = 0.5 * m[i] * vv;
        }
        __syncthreads();
        if (lane == 0) {
            const int n = min(64, N_interact - b);
            for (int k = 0; k < n; k++) e_kin += terms[k];
        }
        __syncthreads();
    }
    if (lane == 0) {
        out[0] = e_kin;
        out[1] = 0.;
    }
}

// Pair terms G m_j m_i / r_ij of rows i0 .. i0 + gridDim.x - 1, j = i+1 ..
// N_interact-1, row after row (the reference's loop order).
__device__ __forceinline__ long energy_row_start(long i, long NI) { return i * (NI - 1) - i * (i - 1) / 2; }

__global__ __launch_bounds__(256) void k_energy_pair_terms(const double* __restrict__ x, const double* __restrict__ y,
                                                           const double* __restrict__ z, const double* __restrict__ m,
                                                           int i0, int N_interact, double G,
                                                           double* __restrict__ buf) {
    const int i = i0 + blockIdx.x;
    const long off = energy_row_start(i, N_interact) - energy_row_start(i0, N_interact) - (i + 1);
    const double xi = x[i], yi = y[i], zi = z[i], mi = m[i];
    for (int j = i + 1 + (int)threadIdx.x; j < N_interact; j += blockDim.x) {
        const double dx = xi - x[j];
        const double dy = yi - y[j];
        const double dz = zi - z[j];
        buf[off + j] = G * m[j] * mi / sqrt(dx * dx + dy * dy + dz * dz);
    }
}

// e_pot -= buf[0 .. n-1] in order, continuing out[1].
__global__ __launch_bounds__(64) void k_energy_fold_terms(const double* __restrict__ buf, long n,
                                                          double* __restrict__ out) {
    constexpr int PER = 16;
    constexpr int CH = 64 * PER;
    __shared__ __align__(16) double stage[2][CH];
    const int lane = threadIdx.x;
    double e = out[1];
    const long nch = (n + CH - 1) / CH;
    double r[PER];
    auto load = [&](long c) {
        const long base = c * CH + (long)lane * PER;
#pragma unroll
        for (int q = 0; q < PER; q++) r[q] = base + q < n ? buf[base + q] : 0.;
    };
    auto store = [&](int b) {
#pragma unroll
        for (int q = 0; q < PER; q++) stage[b][lane * PER + q] = r[q];
    };
    if (nch > 0) {
        load(0);
        store(0);
    }
    __syncthreads();
    for (long c = 0; c < nch; c++) {
        const int b = (int)(c & 1);
        if (c + 1 < nch) load(c + 1);   // in flight while lane 0 folds chunk c
        if (lane == 0) {
            const long cnt = n - c * CH;
            if (cnt >= CH) {
#pragma unroll 16
                for (int k = 0; k < CH; k++) e -= stage[b][k];
            } else {
                for (int k = 0; k < (int)cnt; k++) e -= stage[b][k];
            }
        }
        // stage[b ^ 1] was last read in the previous iteration, before its barrier
        if (c + 1 < nch) store(b ^ 1);
        __syncthreads();
    }
    if (lane == 0) out[1] = e;
}

// The parallel energy.  Workgroup (I, c): 256 targets against the source tiles
// I + c, I + c + C, ... of 256, pairs j > i.  A term G m_j m_i / r takes the
// reciprocal square root refined to full FP64 accuracy (as the FP64 forces),
// not the IEEE square root and division, and every term is Kahan-added; the
// lanes' sums are added with their rounding errors kept (two_add).  Tiles are
// spread over blockIdx.y: with one workgroup per 256 targets walking its whole
// triangle row the first one set the time (65536 bodies 12.5 ms, 10007 1.94, 1024 0.216;
// now 1.80, 0.084 and 0.047, the call's copy and wait included).  A lane whose sum is not
// finite (coincident, non-finite or overflowing distances, or squares of distances below
// the normal range, whose reciprocal overflows in the refinement) repeats its tile with
// IEEE arithmetic.

// Sum of (s, c) over the workgroup's threads into out[0] (sum) and out[1] (its
// rounding error), in a fixed order.
template <int THREADS>
__device__ __forceinline__ void block_two_sum(double s, double c, double (*red)[THREADS], double* out) {
    const int tid = threadIdx.x;
    __syncthreads();
    red[0][tid] = s;
    red[1][tid] = c;
    __syncthreads();
    for (int w = THREADS / 2; w > 0; w >>= 1) {
        if (tid < w) {
            double a = red[0][tid], e = red[1][tid];
            two_add(red[0][tid + w], red[1][tid + w], a, e);
            red[0][tid] = a;
            red[1][tid] = e;
        }
        __syncthreads();
    }
    if (tid == 0) {
        out[0] = red[0][0];
        out[1] = red[1][0];
    }
}

__global__ __launch_bounds__(256) void k_energy_tiles(const double* __restrict__ x, const double* __restrict__ y,
                                                      const double* __restrict__ z, const double* __restrict__ vx,
                                                      const double* __restrict__ vy, const double* __restrict__ vz,
                                                      const double* __restrict__ m, int N_active, int N_interact,
                                                      double G, double* __restrict__ pot, double* __restrict__ kin) {
    __shared__ double4 tile[256];
    __shared__ double red[2][256];
    const int tid = threadIdx.x;
    const int I = blockIdx.x, c0 = blockIdx.y, C = gridDim.y, T = gridDim.x;
    const int i = I * 256 + tid;
    const bool live = i < N_interact;
    const double xi = live ? x[i] : 0., yi = live ? y[i] : 0., zi = live ? z[i] : 0., mi = live ? m[i] : 0.;
    const bool target = live && i < N_active;
    double s = 0., c = 0.;
    for (int J = I + c0; J < T; J += C) {
        const int t = J * 256;
        __syncthreads();
        if (t + tid < N_interact) tile[tid] = make_double4(x[t + tid], y[t + tid], z[t + tid], m[t + tid]);
        __syncthreads();
        const int n = min(256, N_interact - t);
        if (!target) continue;
        const double s0 = s, c0s = c;
        const int first = J == I ? tid + 1 : 0;       // pairs j > i
#pragma unroll 4
        for (int k = 0; k < n; k++) {
            const double4 q = tile[k];
            const double dx = xi - q.x, dy = yi - q.y, dz = zi - q.z;
            const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
            const double r = __builtin_amdgcn_rsq(r2);
            const double e = fma(-r2, r * r, 1.0);
            const double ri = fma(r * e, fma(e, 0.375, 0.5), r);
            // s += m_j / r, Kahan; the skipped pairs of the diagonal tile add nothing
            const double mj = k >= first ? q.w : 0.;
            const double yv = fma(mj, k >= first ? ri : 0., -c);
            const double tv = s + yv;
            c = (tv - s) - yv;
            s = tv;
        }
        if (!(fabs(s) < __builtin_inf())) {
            s = s0;
            c = c0s;
            for (int k = first; k < n; k++) {
                const double4 q = tile[k];
                const double dx = xi - q.x, dy = yi - q.y, dz = zi - q.z;
                kahan_add(q.w / sqrt(dx * dx + dy * dy + dz * dz), s, c);
            }
        }
    }
    // -G m_i (s - c) with its rounding error
    const double w = target ? -G * mi : 0.;
    const double hi = target ? w * s : 0.;
    const double lo = target ? fma(w, s, -hi) - w * c : 0.;
    block_two_sum<256>(hi, lo, red, pot + 2 * ((size_t)I * C + c0));
    if (c0 == 0) {
        double ek = 0.;
        if (live) {
            const double vxi = vx[i], vyi = vy[i], vzi = vz[i];
            ek = 0.5 * mi * (vxi * vxi + vyi * vyi + vzi * vzi);
        }
        block_two_sum<256>(ek, 0., red, kin + 2 * I);
    }
}

__global__ __launch_bounds__(1024) void k_energy_total(const double* __restrict__ pot, int npot,
                                                       const double* __restrict__ kin, int nkin,
                                                       double* __restrict__ out) {
    __shared__ double red[2][1024];
    __shared__ double sum[2];
    for (int which = 0; which < 2; which++) {
        const double* p = which ? kin : pot;
        const int n = which ? nkin : npot;
        double s = 0., c = 0.;
        for (int k = threadIdx.x; k < n; k += 1024) two_add(p[2 * k], p[2 * k + 1], s, c);
        block_two_sum<1024>(s, c, red, sum);
        if (threadIdx.x == 0) out[which ? 0 : 1] = sum[0] + sum[1];
    }
}

// Source tiles of a target tile spread over this many workgroups: one tile each
// up to 127 tiles, and the partial sums (two doubles each, and two per target
// tile, after the first 16) fit the caller's scratch.
static constexpr int energy_split(int tiles) { return tiles < 128 ? tiles : 128 - 1; }
static constexpr bool energy_fits(int tiles) {      // the fewest bodies of so many tiles
    return 16 + 2 * (size_t)tiles * (energy_split(tiles) + 1) <= energy_scratch(256 * (size_t)(tiles - 1) + 1);
}
static constexpr bool energy_fits_upto(int tiles) { return tiles < 1 || (energy_fits(tiles) && energy_fits_upto(tiles - 1)); }
static_assert(energy_fits_upto(400) && energy_fits(4096) && energy_fits(1 << 20), "energy scratch");

int energy_launch(const double* x, const double* y, const double* z, const double* vx, const double* vy,
                  const double* vz, const double* m, int n, int n_active, int n_interact, double G, bool exact,
                  double* out, hipStream_t st, double* terms, size_t terms_cap) {
    if (exact && !(terms && terms_cap > 0)) return 1;
    if (exact) {
        hipLaunchKernelGGL(k_energy_kin, dim3(1), dim3(64), 0, st, vx, vy, vz, m, n_interact, out);
        // rows in batches whose terms fit the buffer (a row has at most n_interact - 1)
        const long NI = n_interact;
        for (int i0 = 0; i0 < n_active;) {
            int i1 = i0;
            long cnt = 0;
            while (i1 < n_active && cnt + (NI - 1 - i1) <= (long)terms_cap) {
                cnt += NI - 1 - i1;
                i1++;
            }
            if (i1 == i0) return 1;   // a single row larger than the buffer
            if (cnt > 0) {
                hipLaunchKernelGGL(k_energy_pair_terms, dim3(i1 - i0), dim3(256), 0, st, x, y, z, m, i0, n_interact, G,
                                   terms);
                hipLaunchKernelGGL(k_energy_fold_terms, dim3(1), dim3(64), 0, st, terms, cnt, out);
            }
            i0 = i1;
        }
    } else {
        const int T = (n_interact + 255) / 256, C = energy_split(T);
        double* pot = out + 16;
        double* kin = pot + 2 * (size_t)T * C;
        if (T > 0)
            hipLaunchKernelGGL(k_energy_tiles, dim3(T, C), dim3(256), 0, st, x, y, z, vx, vy, vz, m, n_active,
                               n_interact, G, pot, kin);
        hipLaunchKernelGGL(k_energy_total, dim3(1), dim3(1024), 0, st, pot, T * C, kin, T, out);
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

static constexpr size_t kEnergyExactMax = 16384;             // bodies
static constexpr size_t kEnergyTermsMax = size_t(4) << 20;    // pair terms per batch (32 MB)

double energy_device(struct reb_simulation* r) {
    DeviceState* d = dev_of(r);
    const size_t N = r->N;
    const size_t N_active = (r->N_active == SIZE_MAX) ? N : r->N_active;
    const size_t N_interact = (r->testparticle_type == 0) ? N_active : N;
    if (N == 0) return r->energy_offset;
    // EXACT: the reference's sequential sum, bit-identical, up to kEnergyExactMax
    // bodies (a serial chain of N^2/2 additions); above, the compensated sum.
    const bool exact = d->precision == REB_AMD_PRECISION_EXACT && N_interact <= kEnergyExactMax;
    if (d->precision == REB_AMD_PRECISION_EXACT && !exact && !d->warned_energy_exact) {
        d->warned_energy_exact = true;
        reb_simulation_warning(r,
                               "EXACT precision: above 16384 interacting bodies the energy is summed with Kahan "
                               "compensation in parallel, not in the reference's serial order, so its last bits "
                               "can differ from the reference's.");
    }
    const size_t terms_cap = exact ? std::min<size_t>(kEnergyTermsMax, N_active * N_interact / 2 + N_interact) : 0;
    const size_t head = energy_scratch(N);
    if (!d->scratch.ensure(sizeof(double) * (head + terms_cap))) {
        reb_simulation_error(r, "Out of device memory for the energy reduction.");
        return nan("");
    }
    double* out = d->scratch.as<double>();
    if (energy_launch(d->field(FX), d->field(FY), d->field(FZ), d->field(FVX), d->field(FVY), d->field(FVZ),
                      d->field(FM), (int)N, (int)N_active, (int)N_interact, r->G, exact, out, d->stream,
                      exact ? out + head : nullptr, terms_cap)) {
        (void)RB_HIP(r, hipGetLastError());
        return nan("");
    }
    double h[2] = {0, 0};
    if (!RB_HIP(r, hipMemcpyAsync(h, out, sizeof(h), hipMemcpyDeviceToHost, d->stream))) return nan("");
    if (!stream_sync(r)) return nan("");
    return h[0] + h[1] + r->energy_offset;
}

}  // namespace rbamd

using namespace rbamd;

extern "C" {

REB_API size_t reb_amd_gravity_workspace_bytes(size_t N, int precision) {
    if (precision == REB_AMD_PRECISION_EXACT) return 256;
    return workspace_bytes((int)N, max_chunks((int)N, (int)N, 1)) + 256;
}

REB_API int reb_amd_gravity_direct(const double* x, const double* y, const double* z, const double* m, double* ax,
                                   double* ay, double* az, size_t N, size_t N_active, int testparticle_type,
                                   int ignore_terms, double G, double softening, int precision, int compensated,
                                   void* workspace, void* stream) {
    if (N > (size_t)INT32_MAX / 8) {
        set_last_error("reb_amd_gravity_direct: N too large");
        return 2;
    }
    if (N_active == SIZE_MAX || N_active > N) N_active = N;
    if (precision != REB_AMD_PRECISION_EXACT && workspace == nullptr) {
        set_last_error("reb_amd_gravity_direct: workspace required for this precision");
        return 3;
    }
    hipStream_t st = (hipStream_t)stream;
    GBList gl;
    gl.n = 1;
    gl.g[0] = GB3{0., 0., 0.};
    return direct_dispatch(x, y, z, m, ax, ay, az, (int)N, (int)N_active, testparticle_type, ignore_terms, G,
                           softening * softening, precision, compensated, gl, static_cast<double*>(workspace), st);
}

}  // extern "C"

// ---------------------------------------------------------------- no-allocation variant
// The chunk partial sums of the fast modes live in a fixed device array
// instead of a caller workspace.  The name `scratch` is a host-side stand-in
// in host code; its device address is looked up once per device
// (hipGetSymbolAddress with that device current) and only that address is
// passed to kernels.  Every partial-sum entry the reduction reads is written
// by the pair kernel of the same call first, so nothing needs clearing.
// Calls that overlap on one device share the array and race.
namespace rbamd {

static constexpr size_t kScratchBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices];

static void* scratch_on_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_last_error("reb_amd_gravity_direct_noalloc: no current HIP device");
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            set_last_error(std::string("reb_amd_gravity_direct_noalloc: hipGetSymbolAddress failed: ") +
                           hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

}  // namespace rbamd

extern "C" {

REB_API size_t reb_amd_gravity_noalloc_max_bytes(void) { return kScratchBytes; }

REB_API int reb_amd_gravity_direct_noalloc(const double* x, const double* y, const double* z, const double* m,
                                           double* ax, double* ay, double* az, size_t N, size_t N_active,
                                           int testparticle_type, int ignore_terms, double G, double softening,
                                           int precision, int compensated, void* stream) {
    if (N > (size_t)INT32_MAX / 8) {
        set_last_error("reb_amd_gravity_direct_noalloc: N too large");
        return 2;
    }
    if (N_active == SIZE_MAX || N_active > N) N_active = N;
    const size_t need = reb_amd_gravity_workspace_bytes(N, precision);
    if (need > kScratchBytes) {
        set_last_error("reb_amd_gravity_direct_noalloc: N=" + std::to_string(N) + " needs " + std::to_string(need) +
                       " bytes of partial sums, above the fixed " + std::to_string(kScratchBytes) +
                       "-byte device array; use reb_amd_gravity_direct with a workspace");
        return 4;
    }
    void* ws = scratch_on_current_device();
    if (ws == nullptr) return 5;
    hipStream_t st = (hipStream_t)stream;
    GBList gl;
    gl.n = 1;
    gl.g[0] = GB3{0., 0., 0.};
    return direct_dispatch(x, y, z, m, ax, ay, az, (int)N, (int)N_active, testparticle_type, ignore_terms, G,
                           softening * softening, precision, compensated, gl, static_cast<double*>(ws), st);
}

}  // extern "C"
