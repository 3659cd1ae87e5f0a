// Device functions shared by the WHFast kernels (whfast.hip, whfast_lane.hip):
// the universal-variable Kepler solver with its Stumpff series
// (integrator_whfast.c:161-427), the variational drift and the symplectic
// corrector coefficients.  Internal linkage: every translation unit has its
// own copy of the constants.
#pragma once

#include <hip/hip_runtime.h>
#include <cmath>

namespace rbamd {

// 1/k! as the reference spells them (integrator_whfast.c:158); 0..13 are used
// by the solver, 0..15 by the variational drift.
static __constant__ double kInvFact[16] = {1.,
                                    1.,
                                    1. / 2.,
                                    1. / 6.,
                                    1. / 24.,
                                    1. / 120.,
                                    1. / 720.,
                                    1. / 5040.,
                                    1. / 40320.,
                                    1. / 362880.,
                                    1. / 3628800.,
                                    1. / 39916800.,
                                    1. / 479001600.,
                                    1. / 6227020800.,
                                    1. / 87178291200.,
                                    1. / 1307674368000.};

// The warning bits (0 .. 3) of lanes first .. first + G - 1, a group; groups of any
// size lie side by side, so exchanges over powers of two would mix neighbours.
__device__ __forceinline__ int group_or(int warn, int first, int G) {
    const unsigned long long group = (G < 64 ? (1ull << G) - 1ull : ~0ull) << first;
    int any = 0;
    for (int b = 0; b < 4; b++)
        if (__ballot(warn & (1 << b)) & group) any |= 1 << b;
    return any;
}

__device__ __forceinline__ double fastabs(double x) { return (x > 0.) ? x : -x; }

// The number of times z is divided by 4 until |z| <= 0.1
// (integrator_whfast.c:190-194), and that quotient in z.  Powers of 4 are
// exact, so it follows from z's exponent E: 0.1 = 1.6 * 2^-4, so ceil((E+4)/2)
// divisions leave |z| < 2^-4 * 2, and one more is needed when that exceeds
// 0.1.  No loop, so a wavefront whose lanes need different counts branches
// once.  An infinite z never comes below 0.1 (the reference's loop would not
// end): it becomes NaN, and with it every function of it.
__device__ __forceinline__ int quarterings(double& z) {
    int n = 0;
    if (fabs(z) > 0.1) {
        n = (__builtin_amdgcn_frexp_exp(z) + 4) >> 1;
        double q = __builtin_amdgcn_ldexp(z, -2 * n);
        if (fabs(q) > 0.1) {
            q *= 0.25;
            n++;
        }
        if (isinf(z)) {
            q = __builtin_nan("");
            n = 0;
        }
        z = q;
    }
    return n;
}

// c_0..c_3 Stumpff functions of z by series + quartering (integrator_whfast.c:189-213).
__device__ __forceinline__ void stumpff_cs3(double* cs, double z) {
    int n = quarterings(z);
    double c_odd = kInvFact[13];
    double c_even = kInvFact[12];
#pragma unroll
    for (int np = 11; np >= 3; np -= 2) {
        c_odd = kInvFact[np] - z * c_odd;
        c_even = kInvFact[np - 1] - z * c_even;
    }
    cs[3] = c_odd;
    cs[2] = c_even;
    cs[1] = kInvFact[1] - z * c_odd;
    cs[0] = kInvFact[0] - z * c_even;
    for (; n > 0; n--) {
        cs[3] = (cs[2] + cs[0] * cs[3]) * 0.25;
        cs[2] = cs[1] * cs[1] * 0.5;
        cs[1] = cs[0] * cs[1];
        cs[0] = 2. * cs[0] * cs[0] - 1.;
    }
}

__device__ __forceinline__ void stiefel_Gs3(double* Gs, double beta, double X) {
    const double X2 = X * X;
    stumpff_cs3(Gs, beta * X2);
    Gs[1] *= X;
    Gs[2] *= X2;
    Gs[3] *= X2 * X;
}

// c_0..c_5 (integrator_whfast.c:161-187), for the variational drift.
__device__ __forceinline__ void stumpff_cs(double* cs, double z) {
    int n = quarterings(z);
    double c_odd = kInvFact[15];
    double c_even = kInvFact[14];
#pragma unroll
    for (int np = 13; np >= 5; np -= 2) {
        c_odd = kInvFact[np] - z * c_odd;
        c_even = kInvFact[np - 1] - z * c_even;
    }
    cs[5] = c_odd;
    cs[4] = c_even;
    cs[3] = kInvFact[3] - z * cs[5];
    cs[2] = kInvFact[2] - z * cs[4];
    cs[1] = kInvFact[1] - z * cs[3];
    for (; n > 0; n--) {
        z = z * 4.;
        cs[5] = (cs[5] + cs[4] + cs[3] * cs[2]) * 0.0625;
        cs[4] = (1. + cs[1]) * cs[3] * 0.125;
        cs[3] = 1. / 6. - z * cs[5];
        cs[2] = 0.5 - z * cs[4];
        cs[1] = 1. - z * cs[3];
    }
    cs[0] = kInvFact[0] - z * cs[2];
}

__device__ __forceinline__ void stiefel_Gs(double* Gs, double beta, double X) {
    const double X2 = X * X;
    stumpff_cs(Gs, beta * X2);
    Gs[1] *= X;
    Gs[2] *= X2;
    double pw = X2 * X;
    Gs[3] *= pw;
    pw *= X;
    Gs[4] *= pw;
    pw *= X;
    Gs[5] *= pw;
}

// What the variational drift of a body needs from its Kepler solve: the
// state before the drift, the solver's scalars and the drift coefficients.
struct KepOut {
    double x0, y0, z0, vx0, vy0, vz0;
    double r0, r0i, ri, beta, eta0, zeta0, X, mu;
    double f, g, fd, gd;
};

// One quartic (Laguerre-Conway) update of X (integrator_whfast.c:292-300).
// Gs receives the Stiefel functions of the X the update started from.
__device__ __forceinline__ double quartic_next(double X, double beta, double r0, double eta0, double zeta0,
                                               double dt, double* Gs) {
    stiefel_Gs3(Gs, beta, X);
    const double f = r0 * X + eta0 * Gs[2] + zeta0 * Gs[3] - dt;
    const double fp = r0 + eta0 * Gs[1] + zeta0 * Gs[2];
    const double fpp = eta0 * Gs[0] + zeta0 * Gs[1];
    const double denom = fp + sqrt(fabs(16. * fp * fp - 20. * f * fpp));
    return (X * denom - 5. * f) / denom;
}

// Universal-variable Kepler drift of one body (integrator_whfast.c:241-390),
// in place.  Returns a bit mask: 1 = the step exceeded one orbital period
// (the reference warns once), 4 = the quartic iteration ran, 8 = the
// bisection fallback ran.
__device__ __forceinline__ int kepler_solver(double& px, double& py, double& pz, double& pvx, double& pvy, double& pvz, double mu,
                             double dt, KepOut* out = nullptr) {
    const double x0 = px, y0 = py, z0 = pz, vx0 = pvx, vy0 = pvy, vz0 = pvz;
    int flags = 0;
    const double r0 = sqrt(x0 * x0 + y0 * y0 + z0 * z0);
    const double r0i = 1. / r0;
    const double v2 = vx0 * vx0 + vy0 * vy0 + vz0 * vz0;
    const double beta = 2. * mu * r0i - v2;
    const double eta0 = x0 * vx0 + y0 * vy0 + z0 * vz0;
    const double zeta0 = mu - beta * r0;
    double X;
    double Gs[4];
    double sqrt_beta = 0.;
    if (beta > 0.) {
        sqrt_beta = sqrt(beta);
        // |dt| / period > 1 (:262-273): the product decides it without the
        // division unless it is near the limit (or mu is not an ordinary
        // positive number)
        const double num = sqrt_beta * beta, den = 2. * M_PI * mu;
        if (!(den > 1e-250 && fabs(dt) * num < 0.99 * den) && fabs(dt) * (num / den) > 1.) flags |= 1;
        const double dtr0i = dt * r0i;
        X = dtr0i * (1. - dtr0i * eta0 * 0.5 * r0i);
    } else {
        X = 0.;
    }
    unsigned int converged = 0;
    double oldX = X;
    stiefel_Gs3(Gs, beta, X);
    const double e0 = eta0 * Gs[1] + zeta0 * Gs[2];
    double ri = 1. / (r0 + e0);
    X = ri * (X * e0 - eta0 * Gs[2] - zeta0 * Gs[3] + dt);

    // |X - oldX| > 0.01 X_per_period with X_per_period = 2 pi / sqrt(beta) (NaN
    // unless beta > 0), again without the division unless it is near the limit
    // (2 pi / 100 = 0.0628)
    bool quartic = false;
    if (beta > 0.) {
        const double d = fastabs(X - oldX), dq = d * sqrt_beta;
        quartic = dq > 0.066;
        if (!(dq < 0.06) && !quartic) quartic = d > 0.01 * (2. * M_PI / sqrt_beta);
    }
    if (quartic) {
        // Quartic (Laguerre-Conway) iteration with cycle detection (:289-312):
        // converged at the first iterate equal to any earlier one.  The last
        // eight iterates are compared in registers (NaN: empty, equal to
        // nothing); an iterate leaving that window is stored in `older`,
        // which is read only when the loop runs past nine iterations.  Short
        // loops (most of them) touch no memory.
        flags |= 4;
        X = beta * dt / mu;
        double older[56];      // older[k] = X_k once it has left the window
        double w0 = __builtin_nan(""), w1 = w0, w2 = w0, w3 = w0, w4 = w0, w5 = w0, w6 = w0, w7 = w0;
        for (int n_lag = 1; n_lag < 64; n_lag++) {
            // X_{n_lag} from X_{n_lag-1}; w0..w7 hold X_{n_lag-1}..X_{n_lag-8}
            X = quartic_next(X, beta, r0, eta0, zeta0, dt, Gs);
            if (X == w0 || X == w1 || X == w2 || X == w3 || X == w4 || X == w5 || X == w6 || X == w7) {
                converged = 1;
                break;
            }
            for (int k = 1; k < n_lag - 8; k++) {
                if (X == older[k]) {
                    converged = 1;
                    break;
                }
            }
            if (converged) break;
            if (n_lag > 8) older[n_lag - 8] = w7;
            w7 = w6; w6 = w5; w5 = w4; w4 = w3; w3 = w2; w2 = w1; w1 = w0; w0 = X;
        }
        const double e1 = eta0 * Gs[1] + zeta0 * Gs[2];
        ri = 1. / (r0 + e1);
    } else {
        // Newton's method (:313-330).
        double oldX2 = __builtin_nan("");
        for (int n_hg = 1; n_hg < 32; n_hg++) {
            oldX2 = oldX;
            oldX = X;
            stiefel_Gs3(Gs, beta, X);
            const double e1 = eta0 * Gs[1] + zeta0 * Gs[2];
            ri = 1. / (r0 + e1);
            X = ri * (X * e1 - eta0 * Gs[2] - zeta0 * Gs[3] + dt);
            if (X == oldX || X == oldX2) {
                converged = 1;
                break;
            }
        }
    }
    if (converged == 0) {
        // Bisection fallback (:333-369).
        flags |= 8;
        double X_min, X_max;
        if (beta > 0.) {
            const double invperiod = sqrt_beta * beta / (2. * M_PI * mu);
            const double X_per_period = 2. * M_PI / sqrt_beta;
            X_min = X_per_period * floor(dt * invperiod);
            X_max = X_min + X_per_period;
        } else {
            const double h2 = r0 * r0 * v2 - eta0 * eta0;
            const double q = h2 / mu / (1. + sqrt(1. - h2 * beta / (mu * mu)));
            const double vq = copysign(sqrt(h2) / q, dt);
            X_min = dt / (fastabs(vq * dt) + r0);
            X_max = dt / q;
            if (dt < 0.) {
                const double temp = X_min;
                X_min = X_max;
                X_max = temp;
            }
        }
        X = (X_max + X_min) / 2.;
        // halving exhausts the doubles of any finite interval in < 2200 steps
        int guard = 0;
        do {
            stiefel_Gs3(Gs, beta, X);
            const double s = r0 * X + eta0 * Gs[2] + zeta0 * Gs[3] - dt;
            if (s >= 0.) {
                X_max = X;
            } else {
                X_min = X;
            }
            X = (X_max + X_min) / 2.;
        } while (fastabs((X_max - X_min)) > fastabs((X_max + X_min) * 1e-15) && ++guard < 4096);
        const double e1 = eta0 * Gs[1] + zeta0 * Gs[2];
        ri = 1. / (r0 + e1);
    }
    if (isnan(ri)) {
        ri = 0.;
        Gs[1] = 0.;
        Gs[2] = 0.;
        Gs[3] = 0.;
    }
    const double f = -mu * Gs[2] * r0i;
    const double g = dt - mu * Gs[3];
    const double fd = -mu * Gs[1] * r0i * ri;
    const double gd = -mu * Gs[2] * ri;
    px += f * x0 + g * vx0;
    py += f * y0 + g * vy0;
    pz += f * z0 + g * vz0;
    pvx += fd * x0 + gd * vx0;
    pvy += fd * y0 + gd * vy0;
    pvz += fd * z0 + gd * vz0;
    if (out) {
        *out = KepOut{x0, y0, z0, vx0, vy0, vz0, r0, r0i, ri, beta, eta0, zeta0, X, mu, f, g, fd, gd};
    }
    return flags;
}

// The drift of one body's variational particle d along its Kepler solve k
// (integrator_whfast.c:392-426): the Stiefel functions at the final X, then
// the derivatives of X, r and the drift coefficients.
__device__ __forceinline__ void kepler_var(const KepOut& k, double& dx, double& dy, double& dz, double& dvx,
                                           double& dvy, double& dvz) {
    const double d_x = dx, d_y = dy, d_z = dz, d_vx = dvx, d_vy = dvy, d_vz = dvz;
    double Gs[6];
    stiefel_Gs(Gs, k.beta, k.X);
    const double mu = k.mu, r0 = k.r0, r0i = k.r0i, ri = k.ri, X = k.X, beta = k.beta;
    const double dr0 = (d_x * k.x0 + d_y * k.y0 + d_z * k.z0) * r0i;
    const double dbeta = -2. * mu * dr0 * r0i * r0i - 2. * (d_vx * k.vx0 + d_vy * k.vy0 + d_vz * k.vz0);
    const double deta0 = d_x * k.vx0 + d_y * k.vy0 + d_z * k.vz0 + k.x0 * d_vx + k.y0 * d_vy + k.z0 * d_vz;
    const double dzeta0 = -beta * dr0 - r0 * dbeta;
    const double G3beta = 0.5 * (3. * Gs[5] - X * Gs[4]);
    const double G2beta = 0.5 * (2. * Gs[4] - X * Gs[3]);
    const double G1beta = 0.5 * (Gs[3] - X * Gs[2]);
    const double tbeta = k.eta0 * G2beta + k.zeta0 * G3beta;
    const double dX = -1. * ri * (X * dr0 + Gs[2] * deta0 + Gs[3] * dzeta0 + tbeta * dbeta);
    const double dG1 = Gs[0] * dX + G1beta * dbeta;
    const double dG2 = Gs[1] * dX + G2beta * dbeta;
    const double dG3 = Gs[2] * dX + G3beta * dbeta;
    const double dr = dr0 + Gs[1] * deta0 + Gs[2] * dzeta0 + k.eta0 * dG1 + k.zeta0 * dG2;
    const double df = mu * Gs[2] * dr0 * r0i * r0i - mu * dG2 * r0i;
    const double dg = -mu * dG3;
    const double dfd = -mu * dG1 * r0i * ri + mu * Gs[1] * (dr0 * r0i + dr * ri) * r0i * ri;
    const double dgd = -mu * dG2 * ri + mu * Gs[2] * dr * ri * ri;
    dx += k.f * d_x + k.g * d_vx + df * k.x0 + dg * k.vx0;
    dy += k.f * d_y + k.g * d_vy + df * k.y0 + dg * k.vy0;
    dz += k.f * d_z + k.g * d_vz + df * k.z0 + dg * k.vz0;
    dvx += k.fd * d_x + k.gd * d_vx + dfd * k.x0 + dgd * k.vx0;
    dvy += k.fd * d_y + k.gd * d_vy + dfd * k.y0 + dgd * k.vy0;
    dvz += k.fd * d_z + k.gd * d_vz + dfd * k.z0 + dgd * k.vz0;
}

// Symplectic corrector coefficients of Wisdom, Holman & Touma (1996), the
// values integrator_whfast.c:125-152 spells: a_k = k * sqrt(7/40) and the
// b coefficients of the 3rd to 17th order correctors; kCorr2B is the second
// corrector's coefficient (Wisdom 2006).
static __constant__ double kCorrA[9] = {0.,
                                 0.41833001326703777398908601289259374469640768464934,
                                 0.83666002653407554797817202578518748939281536929867,
                                 1.2549900398011133219672580386777812340892230539480,
                                 1.6733200530681510959563440515703749787856307385973,
                                 2.0916500663351888699454300644629687234820384232467,
                                 2.5099800796022266439345160773555624681784461078960,
                                 2.9283100928692644179236020902481562128748537925454,
                                 3.3466401061363021919126881031407499575712614771947};
static constexpr double kCorr2B = 0.03486083443891981449909050107438281205803;
// One corrector of order n is a chain of Z(a, b) operators.  An entry holds
// the signed index of a (a = sign * a_|k| * dt) and the b coefficient for
// inv = +1 (b = inv * coef * dt); the chains of integrator_whfast.c:696-751.
struct CorrZ {
    signed char ka;
    double kb;
};
static __constant__ CorrZ kCorr3[2] = {{1, 0.024900596027799867499350357910273437184309981229127},
                                {-1, -0.024900596027799867499350357910273437184309981229127}};
static __constant__ CorrZ kCorr5[4] = {{-2, 0.0083001986759332891664501193034244790614366604097090},
                                {-1, -0.041500993379666445832250596517122395307183302048545},
                                {1, 0.041500993379666445832250596517122395307183302048545},
                                {2, -0.0083001986759332891664501193034244790614366604097090}};
static __constant__ CorrZ kCorr7[6] = {{-3, -0.0024926811426922105779030593952776964450539008582219},
                                {-2, 0.018270923246702131478062356884535264841652263842597},
                                {-1, -0.053964399093127498721765893493510877532452806339655},
                                {1, 0.053964399093127498721765893493510877532452806339655},
                                {2, -0.018270923246702131478062356884535264841652263842597},
                                {3, 0.0024926811426922105779030593952776964450539008582219}};
static __constant__ CorrZ kCorr11[10] = {{-5, -0.00020361579647854651301632818774633716473696537436847},
                                  {-4, 0.0023487215292295354188307328851055489876255097419754},
                                  {-3, -0.012309078592019946317544564763237909911330686448336},
                                  {-2, 0.038121613681288650508647613260247372125243616270670},
                                  {-1, -0.072593394748842738674253180742744961827622366521517},
                                  {1, 0.072593394748842738674253180742744961827622366521517},
                                  {2, -0.038121613681288650508647613260247372125243616270670},
                                  {3, 0.012309078592019946317544564763237909911330686448336},
                                  {4, -0.0023487215292295354188307328851055489876255097419754},
                                  {5, 0.00020361579647854651301632818774633716473696537436847}};
static __constant__ CorrZ kCorr17[16] = {{-8, 0.0000043347415473373580190650223498124944896789841432241},
                                  {-7, -0.000076436355227935738363241846979413475106795392377415},
                                  {-6, 0.00063599983075817658983166881625078545864140848560259},
                                  {-5, -0.0033132577069380655655490196833451994080066801611459},
                                  {-4, 0.012071760822342291062449751726959664253913904872527},
                                  {-3, -0.032422198864713580293681523029577130832258806467604},
                                  {-2, 0.065192863576377893658290760803725762027864651086787},
                                  {-1, -0.093056103771425958591541059067553547100903397724386},
                                  {1, 0.093056103771425958591541059067553547100903397724386},
                                  {2, -0.065192863576377893658290760803725762027864651086787},
                                  {3, 0.032422198864713580293681523029577130832258806467604},
                                  {4, -0.012071760822342291062449751726959664253913904872527},
                                  {5, 0.0033132577069380655655490196833451994080066801611459},
                                  {6, -0.00063599983075817658983166881625078545864140848560259},
                                  {7, 0.000076436355227935738363241846979413475106795392377415},
                                  {8, -0.0000043347415473373580190650223498124944896789841432241}};

__device__ __forceinline__ const CorrZ* corrector_chain(int order, int& n) {
    switch (order) {
        case 3: n = 2; return kCorr3;
        case 5: n = 4; return kCorr5;
        case 7: n = 6; return kCorr7;
        case 11: n = 10; return kCorr11;
        case 17: n = 16; return kCorr17;
        default: n = 0; return nullptr;
    }
}

}  // namespace rbamd
