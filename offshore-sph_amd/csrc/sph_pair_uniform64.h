// sph_pair_uniform64.h — the double pair pass for one smoothing length for
// every particle and one mass for every fluid particle, bit-identical to the
// general double pass (sph_pair_impl.h) and so to the reference's loop
// (src/Tools/SolverTools.py:120-175). Included by sph_pair_fp64.hip only
// (-ffp-contract=off).
//
// Every contribution keeps the reference's operation order; what the uniform
// case changes is everything around it:
//   * h_ij = 0.5 (h + h) = h, the re-averaged h of the viscosity likewise,
//     m_j = m: the kernel normalisation 10 / (7 pi) / (h h) (Wendland's,
//     the Gaussian's (1 / pi) / (h h)), 0.01 h h and c_ij = c0 / 2 are formed
//     once on the host with the same operations, so their bits are the ones
//     the reference forms per pair;
//   * the kernel support (2h; 3h for the Gaussian) lies within the cut-off
//     q_max h and the wall range r0 inside it: the walk lists every particle
//     within max(support, r0) (a double r^2 test, no cut-off test, no square
//     root), and a listed pair outside the support or the wall range adds
//     nothing, as in the reference (a Gaussian pair at q <= 3 is a neighbour
//     whenever q_max >= 3: the same double q decides both);
//   * records: A = (x, y), B = (vx, vy, rho, p / rho^2) with a NaN in place of
//     p / rho^2 for particles that are not fluid;
//   * the walk visits the reference's nine cells in its order (x shift outer,
//     y shift inner, each cell from its highest slot down), UNROLL records
//     loaded before they are tested; a thread-per-target workgroup stages the
//     records of its targets' cells in LDS first (StagedWalk64).
#pragma once
#include "sph_common.h"
#include "sph_pair_group.h"

namespace hipsph {
namespace {

#ifndef HIPSPH_PEC64_EARLY
#define HIPSPH_PEC64_EARLY 0  // 1: the corrector's gathers before the walk (99 VGPRs instead of 85, 4 waves: no faster)
#endif

#ifndef HIPSPH_UNIFORM64_UNROLL
#define HIPSPH_UNIFORM64_UNROLL 4
#endif
#ifndef HIPSPH_UNIFORM64_LIST
#define HIPSPH_UNIFORM64_LIST 30
#endif
// contributor-list entries per thread (4 B each, 2 B in a staged walk): 30, with
// which either walk's LDS leaves five workgroups per CU
constexpr int kUniform64List = HIPSPH_UNIFORM64_LIST;
// the Gaussian's pass keeps no list (uniform64_rates_direct)
template <int KERNEL>
__host__ __device__ constexpr int uniform64_list() {
    return KERNEL == SPH_KERNEL_GAUSSIAN ? 1 : kUniform64List;
}

struct Uniform64Args {
    const double2 *A;  // (x, y)
    const double4 *B;  // (vx, vy, rho, p / rho^2); p / rho^2 is NaN for particles that are not fluid
    const int2 *cxy;
    const int *cellStart;
    double *ax, *ay, *drho;
    int n;
};

struct Uniform64Const {
    double lim2;           // max((2h)^2, r0^2) (1 + 1e-12): the listed pairs
    double hinv, hinv2;    // 1 / h, 2 / h
    double h, m, alpha_k;  // alpha_k: the kernel normalisation 10 / (7 pi) / (h h) (Wendland: 9 / (4 pi) / (h h))
    double c01;            // 0.01 h h, in the reference's order (0.01 h) h
    double cij, alpha, beta;
    double ih2, g2;        // the Gaussian's 1 / h^2 and -2 alpha_k / h^2 (gauss_factor)
    double r0, D, p1, p2, g, qmax;
    int stage;             // stage the candidates' records in LDS
};

constexpr double kPairNone = 1e-280;  // a pair at this r^2 or less adds nothing
__device__ inline bool not_fluid64(double prs) { return prs != prs; }

// Square roots and quotients of the pair terms with the bits of sqrt() and /,
// without what those spend on the ends of the exponent range (scaling before
// and after, 6 of a root's 16 instructions and 3 of a quotient's 11). A root is
// Goldschmidt's coupled iteration for a^1/2 and a^-1/2 / 2 (R. E. Goldschmidt,
// MIT, 1964) from the hardware's estimate, a quotient a Newton step on the
// hardware's reciprocal; each ends with a correction by the exact remainder,
// which rounds a quotient as / does when the reciprocal is itself the rounded
// one (P. Markstein, IBM J. Res. Dev. 34, 1990; no bit differed in 2.1e9
// random operands of each form). That needs an exact remainder and a normal
// result: the walk lists no pair with r^2 <= 1e-280, which adds nothing anywhere
// (r < 1e-12), and uniform_eligible keeps h between 1e-100 and 1e68 (1e57 for
// Wendland), which keeps the roots and the quotients by h and h r of pairs that
// count (r >= 1e-10) inside. The viscosity's operands depend on velocities and
// densities and may lie anywhere, so they are divided by / (without scaling the
// last bits of rates below 1e-300 differed; 30 steps of 500k particles take 3.62
// ms instead of 3.58).
//
// root(a) also leaves half = 0.5 / root(a) to about 2^-50, from which the
// quotient by h root(a) needs no estimate of its own.
__device__ inline double pair_root(double a, double &half) {
    const double y = __builtin_amdgcn_rsq(a);
    double g = a * y;
    half = 0.5 * y;
    const double e = __builtin_fma(-half, g, 0.5);
    g = __builtin_fma(g, e, g);
    half = __builtin_fma(half, e, half);
    g = __builtin_fma(__builtin_fma(-g, g, a), half, g);
    return __builtin_fma(__builtin_fma(-g, g, a), half, g);
}
// a / b from y, the rounded 1 / b
__device__ inline double pair_quotient(double a, double b, double y) {
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
// 1 / b from an estimate y
__device__ inline double pair_recip(double b, double y) {
    return __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
}

// Whether the target at (X, Y) in cell c has a neighbour: one whose own cell
// is in the grid finds itself (q = 0); one outside looks (SolverTools.py:
// 166-169).
__device__ inline bool uniform64_has_neighbour(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy,
                                               long long base, double X, double Y, int2 c) {
    if (c.x >= 0 && c.x < ncx && c.y >= 0 && c.y < ncy) return true;
    const double lim = (K.qmax * K.h) * (K.qmax * K.h);
    for (int da = -1; da <= 1; ++da) {
        const int cx = c.x + da;
        if (!(ncx > cx && cx > -1)) continue;
        for (int db = -1; db <= 1; ++db) {
            const int cy = c.y + db;
            if (!(ncy > cy && cy > -1)) continue;
            const long long cell = base + cx + (long long)ncx * cy;
            for (int k = P.cellStart[cell]; k < P.cellStart[cell + 1]; ++k) {
                const double2 a = at32(P.A, (unsigned)k);
                const double ddx = X - a.x, ddy = Y - a.y;
                const double r2 = ddx * ddx + ddy * ddy;
                if (r2 < lim * (1.0 - 1e-12)) return true;
                if (!(r2 > lim * (1.0 + 1e-12)) && exact_q_test(X, Y, K.h, a.x, a.y, K.h, K.qmax)) return true;
            }
        }
    }
    return false;
}

// The rates of fluid target t (bt: its B record) over a grid of ncx x ncy
// cells starting at bin `base` (0 for a single simulation, the instance's
// first bin in a batch); false when t has no neighbour and keeps its
// previous rates. MODE kContinuity sums drho only, kMomentum ax and ay only
// (the other outputs are then zero); each sum keeps the order of the fused
// pass, so the split passes give its bits.
template <int KERNEL, int MODE = kFused>
__device__ inline bool uniform64_rates_listed(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy,
                                       long long base, int t, const double4 &bt, unsigned *s_list, double &drho,
                                       double &ax, double &ay) {
    const double2 at = P.A[t];
    const double X = at.x, Y = at.y;
    const int2 c = P.cxy[t];
    const unsigned stride = blockDim.x;
    unsigned *const list0 = s_list + threadIdx.x;
    unsigned *lp = list0;
    double arho = 0.0, a0 = 0.0, a1 = 0.0, f0 = 0.0, f1 = 0.0;
    // The reference's expressions (Continuity.py:13-16, Momentum.py:36-56,
    // BoundaryForce.py:31-41, CubicSpline.py:53-70 / Gaussian.py:41-60 /
    // Wendland.py:32-64) for each listed pair, in listing order.
    auto flush = [&]() {
        for (unsigned *q = list0; q != lp; q += stride) {
            const unsigned u = *q;
            const double2 a = at32(P.A, u);
            const double4 b = at32(P.B, u);
            const double dx = X - a.x, dy = Y - a.y;
            const double xij2 = dx * dx + dy * dy;
            double half;
            const double r = pair_root(xij2, half);
            if (!not_fluid64(b.w)) {
                const double qq = pair_quotient(r, K.h, K.hinv);
                double dwx, dwy;
                double grad;
                if (KERNEL == SPH_KERNEL_WENDLAND) {
                    if ((qq >= 2.0) || (r < 1e-10)) continue;
                    const double inner = 1.0 - 0.5 * qq;
                    grad = ipow(inner, 5.0) * (-14.0 / 3.0) * qq * (1 + 2.5 * qq);
                } else {
                    if ((qq > 2.0) || (r < 1e-10)) continue;
                    grad = (qq > 1.0) ? -0.75 * ((2.0 - qq) * (2.0 - qq)) : -3.0 * qq * (1.0 - 0.75 * qq);
                }
                const double hr = K.h * r;
                const double norm = pair_quotient(K.alpha_k * grad, hr, pair_recip(hr, half * K.hinv2));
                dwx = norm * dx;
                dwy = norm * dy;
                const double vx = bt.x - b.x, vy = bt.y - b.y;
                const double dot = vx * dwx + vy * dwy;
                if constexpr ((MODE & kEquations) != kMomentum) arho += K.m * dot;
                if constexpr ((MODE & kEquations) == kContinuity) continue;
                const double dv = vx * dx + vy * dy;
                double PI_ij = 0.0;
                if (dv < 0) {
                    const double rhoij = 0.5 * (bt.z + b.z);
                    const double muij = K.h * dv / (r * r + K.c01);
                    const double ppij = muij * (K.beta * muij - K.alpha * K.cij);
                    PI_ij = ppij / rhoij;
                }
                const double factor = bt.w + b.w + PI_ij;
                a0 += -K.m * factor * dwx;
                a1 += -K.m * factor * dwy;
            } else if ((MODE & kEquations) != kContinuity && !(r > K.r0) && r > 1e-12) {
                const double frac = K.r0 / r;
                const double tmp = wall_pow<MODE>(frac, K.p1) - wall_pow<MODE>(frac, K.p2);
                const double fac = K.D * tmp;
                f0 += fac * dx / (r * r);
                f1 += fac * dy / (r * r);
            }
        }
        lp = list0;
    };
    constexpr int U = HIPSPH_UNIFORM64_UNROLL, LIST = kUniform64List;
    static_assert(U >= 1 && U < LIST, "unroll within the list");
    unsigned *const full = list0 + (LIST - U) * stride;  // past this, U appends could overflow
    auto overflow = [&]() { return lp > full; };
    auto test = [&](double2 a, int k) {
        const double dx = X - a.x, dy = Y - a.y;
        const double r2 = dx * dx + dy * dy;
        // written whether or not it is kept (within the list's bounds either
        // way): no branch per candidate
        *lp = (unsigned)k;
        lp += (r2 <= K.lim2 && r2 > kPairNone) ? stride : 0u;
    };
    // src/Tools/NNLinkedList.py:50-56: x shift outer, y shift inner, cells at
    // the grid's edge dropped; each cell from its highest slot down (:129-141)
    for (int da = -1; da <= 1; ++da) {
        const int cx = c.x + da;
        if (!(ncx > cx && cx > -1)) continue;
        for (int db = -1; db <= 1; ++db) {
            const int cy = c.y + db;
            if (!(ncy > cy && cy > -1)) continue;
            const long long cell = base + cx + (long long)ncx * cy;
            const int s = P.cellStart[cell], e = P.cellStart[cell + 1];
            int k = e - 1;
            for (; k - U + 1 >= s; k -= U) {
                if (overflow()) flush();
                double2 a[U];
#pragma unroll
                for (int j = 0; j < U; ++j) a[j] = at32j(P.A, (unsigned)k, -j);
#pragma unroll
                for (int j = 0; j < U; ++j) test(a[j], k - j);
            }
            if (k >= s) {
                if (overflow()) flush();
                for (; k >= s; --k) test(at32(P.A, (unsigned)k), k);  // fewer than U
            }
        }
    }
    flush();
    if (!uniform64_has_neighbour(P, K, ncx, ncy, base, X, Y, c)) return false;
    drho = arho;
    ax = a0 + f0;
    ay = (MODE & kEquations) == kContinuity ? 0.0 : (a1 - K.g) + f1;  // WCSPH.py:169, then SolverTools.py:170-171
    return true;
}

// The Gaussian's pass: the same walk, each candidate's terms formed as it is
// met, its records and the next one's in flight. About 42 of 61 candidates
// contribute; listing them first left lanes idle in the flushes of lists that
// filled at different candidates, fetched every contributor's records a second
// time from scattered places, and its 40 KB of lists kept the pass at 4
// wavefronts per SIMD (1M particles: continuity 394 -> 178 us, momentum 456 ->
// 330 us; the cubic spline, 21 of 61, keeps the lists).
template <int MODE>
__device__ inline bool uniform64_rates_direct(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy,
                                              long long base, int t, const double4 &bt, double &drho, double &ax,
                                              double &ay) {
    const double2 at = P.A[t];
    const double X = at.x, Y = at.y;
    const int2 c = P.cxy[t];
    double arho = 0.0, a0 = 0.0, a1 = 0.0, f0 = 0.0, f1 = 0.0;
    for (int da = -1; da <= 1; ++da) {
        const int cx = c.x + da;
        if (!(ncx > cx && cx > -1)) continue;
        for (int db = -1; db <= 1; ++db) {
            const int cy = c.y + db;
            if (!(ncy > cy && cy > -1)) continue;
            const long long cell = base + cx + (long long)ncx * cy;
            const int s = P.cellStart[cell], e = P.cellStart[cell + 1];
            double2 an{};
            double4 bn{};
            if (s < e) {
                an = at32(P.A, (unsigned)(e - 1));
                bn = at32(P.B, (unsigned)(e - 1));
            }
            for (int k = e - 1; k >= s; --k) {
                const double2 a = an;
                const double4 b = bn;
                if (k > s) {
                    an = at32(P.A, (unsigned)(k - 1));
                    bn = at32(P.B, (unsigned)(k - 1));
                }
                const double dx = X - a.x, dy = Y - a.y;
                const double xij2 = dx * dx + dy * dy;
                if (!(xij2 <= K.lim2 && xij2 > kPairNone)) continue;
                if (!not_fluid64(b.w)) {
                    double f;
                    if (!gauss_factor(xij2, K.h, K.ih2, K.g2, f)) continue;
                    const double dwx = f * dx, dwy = f * dy;
                    const double vx = bt.x - b.x, vy = bt.y - b.y;
                    const double dot = vx * dwx + vy * dwy;
                    if constexpr ((MODE & kEquations) != kMomentum) arho += K.m * dot;
                    if constexpr ((MODE & kEquations) == kContinuity) continue;
                    const double dv = vx * dx + vy * dy;
                    double PI_ij = 0.0;
                    if (dv < 0) {
                        const double rhoij = 0.5 * (bt.z + b.z);
                        const double muij = K.h * dv / (xij2 + K.c01);
                        const double ppij = muij * (K.beta * muij - K.alpha * K.cij);
                        PI_ij = ppij / rhoij;
                    }
                    const double factor = bt.w + b.w + PI_ij;
                    a0 += -K.m * factor * dwx;
                    a1 += -K.m * factor * dwy;
                } else if ((MODE & kEquations) != kContinuity) {
                    const double r = sqrt(xij2);
                    if (!(r > K.r0) && r > 1e-12) {
                        const double frac = K.r0 / r;
                        const double tmp = wall_pow<MODE>(frac, K.p1) - wall_pow<MODE>(frac, K.p2);
                        const double fac = K.D * tmp;
                        f0 += fac * dx / (r * r);
                        f1 += fac * dy / (r * r);
                    }
                }
            }
        }
    }
    if (!uniform64_has_neighbour(P, K, ncx, ncy, base, X, Y, c)) return false;
    drho = arho;
    ax = a0 + f0;
    ay = (MODE & kEquations) == kContinuity ? 0.0 : (a1 - K.g) + f1;  // WCSPH.py:169, then SolverTools.py:170-171
    return true;
}

template <int KERNEL, int MODE = kFused>
__device__ inline bool uniform64_rates(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy,
                                       long long base, int t, const double4 &bt, unsigned *s_list, double &drho,
                                       double &ax, double &ay) {
    if constexpr (KERNEL == SPH_KERNEL_GAUSSIAN)
        return uniform64_rates_direct<MODE>(P, K, ncx, ncy, base, t, bt, drho, ax, ay);
    else
        return uniform64_rates_listed<KERNEL, MODE>(P, K, ncx, ncy, base, t, bt, s_list, drho, ax, ay);
}

// The same walk over A records staged in LDS (stage_plan: the three row ranges
// of the workgroup's targets), with a 16-bit list. Walking them in
// global memory kept the vector memory path 66 % busy (500k particles; VALU 53 %),
// as 61 candidates and 21 contributors are 16-byte gathers each: 89 us, 83 staged
// (30 steps 3.74 -> 3.62 ms; 3 instead of 4 records per round 3.66).
template <int KERNEL, int MODE = kFused>
__device__ inline bool uniform64_rates_staged(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy, int t,
                                              const double4 &bt, const Stage &S, const double2 *sA,
                                              unsigned short *s_list, double &drho, double &ax, double &ay) {
    const double2 at = P.A[t];
    const double X = at.x, Y = at.y;
    const int2 c = P.cxy[t];
    const unsigned stride = blockDim.x;
    unsigned short *const list0 = s_list + threadIdx.x;
    unsigned short *lp = list0;
    // LDS record i holds slot i - sh of the row it lies in
    const int off1 = S.off[1], off2 = S.off[2];
    const int sh0 = S.off[0] - S.smin[0], sh1 = off1 - S.smin[1], sh2 = off2 - S.smin[2];
    double arho = 0.0, a0 = 0.0, a1 = 0.0, f0 = 0.0, f1 = 0.0;
    // The reference's expressions (Continuity.py:13-16, Momentum.py:36-56,
    // BoundaryForce.py:31-41, CubicSpline.py:53-70 / Gaussian.py:41-60 /
    // Wendland.py:32-64) for each listed pair, in listing order.
    auto flush = [&]() {
        for (unsigned short *q = list0; q != lp; q += stride) {
            const int i = *q;
            const double2 a = sA[i];
            const double4 b = at32(P.B, (unsigned)(i - (i >= off2 ? sh2 : (i >= off1 ? sh1 : sh0))));
            const double dx = X - a.x, dy = Y - a.y;
            const double xij2 = dx * dx + dy * dy;
            double half;
            const double r = pair_root(xij2, half);
            if (!not_fluid64(b.w)) {
                const double qq = pair_quotient(r, K.h, K.hinv);
                double dwx, dwy;
                double grad;
                if (KERNEL == SPH_KERNEL_WENDLAND) {
                    if ((qq >= 2.0) || (r < 1e-10)) continue;
                    const double inner = 1.0 - 0.5 * qq;
                    grad = ipow(inner, 5.0) * (-14.0 / 3.0) * qq * (1 + 2.5 * qq);
                } else {
                    if ((qq > 2.0) || (r < 1e-10)) continue;
                    grad = (qq > 1.0) ? -0.75 * ((2.0 - qq) * (2.0 - qq)) : -3.0 * qq * (1.0 - 0.75 * qq);
                }
                const double hr = K.h * r;
                const double norm = pair_quotient(K.alpha_k * grad, hr, pair_recip(hr, half * K.hinv2));
                dwx = norm * dx;
                dwy = norm * dy;
                const double vx = bt.x - b.x, vy = bt.y - b.y;
                const double dot = vx * dwx + vy * dwy;
                if constexpr ((MODE & kEquations) != kMomentum) arho += K.m * dot;
                if constexpr ((MODE & kEquations) == kContinuity) continue;
                const double dv = vx * dx + vy * dy;
                double PI_ij = 0.0;
                if (dv < 0) {
                    const double rhoij = 0.5 * (bt.z + b.z);
                    const double muij = K.h * dv / (r * r + K.c01);
                    const double ppij = muij * (K.beta * muij - K.alpha * K.cij);
                    PI_ij = ppij / rhoij;
                }
                const double factor = bt.w + b.w + PI_ij;
                a0 += -K.m * factor * dwx;
                a1 += -K.m * factor * dwy;
            } else if ((MODE & kEquations) != kContinuity && !(r > K.r0) && r > 1e-12) {
                const double frac = K.r0 / r;
                const double tmp = wall_pow<MODE>(frac, K.p1) - wall_pow<MODE>(frac, K.p2);
                const double fac = K.D * tmp;
                f0 += fac * dx / (r * r);
                f1 += fac * dy / (r * r);
            }
        }
        lp = list0;
    };
    constexpr int U = HIPSPH_UNIFORM64_UNROLL, LIST = kUniform64List;
    static_assert(U >= 1 && U < LIST, "unroll within the list");
    unsigned short *const full = list0 + (LIST - U) * stride;  // past this, U appends could overflow
    auto overflow = [&]() { return lp > full; };
    auto test = [&](double2 a, int k) {
        const double dx = X - a.x, dy = Y - a.y;
        const double r2 = dx * dx + dy * dy;
        // written whether or not it is kept (within the list's bounds either
        // way): no branch per candidate
        *lp = (unsigned short)k;
        lp += (r2 <= K.lim2 && r2 > kPairNone) ? stride : 0u;
    };
    // the cells in uniform64_rates_listed's order
    for (int da = -1; da <= 1; ++da) {
        const int cx = c.x + da;
        if (!(ncx > cx && cx > -1)) continue;
        for (int db = -1; db <= 1; ++db) {
            const int cy = c.y + db;
            if (!(ncy > cy && cy > -1)) continue;
            const long long cell = cx + (long long)ncx * cy;
            const int sh = db < 0 ? sh0 : (db == 0 ? sh1 : sh2);
            const int s = P.cellStart[cell] + sh, e = P.cellStart[cell + 1] + sh;
            int k = e - 1;
            for (; k - U + 1 >= s; k -= U) {
                if (overflow()) flush();
                double2 a[U];
#pragma unroll
                for (int j = 0; j < U; ++j) a[j] = sA[k - j];
#pragma unroll
                for (int j = 0; j < U; ++j) test(a[j], k - j);
            }
            if (k >= s) {
                if (overflow()) flush();
                for (; k >= s; --k) test(sA[k], k);  // fewer than U
            }
        }
    }
    flush();
    if (!uniform64_has_neighbour(P, K, ncx, ncy, 0, X, Y, c)) return false;
    drho = arho;
    ax = a0 + f0;
    ay = (MODE & kEquations) == kContinuity ? 0.0 : (a1 - K.g) + f1;  // WCSPH.py:169, then SolverTools.py:170-171
    return true;
}

// LDS of a pass that stages: the records and a 16-bit list, or (a workgroup
// whose ranges exceed the stage) a 32-bit list.
template <int KERNEL>
__host__ __device__ constexpr int stage_bytes64() {
    constexpr int global = uniform64_list<KERNEL>() * 256 * 4;
    constexpr int staged = kStageCap * 16 + uniform64_list<KERNEL>() * 256 * 2;
    return KERNEL == SPH_KERNEL_GAUSSIAN || global > staged ? global : staged;
}
template <int KERNEL>
struct StagedWalk64 {
    unsigned char *mem;
    Stage S{};
    bool staged = false;
    __device__ StagedWalk64(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy, int t, bool walks,
                            unsigned char *s_mem, int *s_red)
        : mem(s_mem) {
        if (KERNEL == SPH_KERNEL_GAUSSIAN || !K.stage) return;  // uniform over the workgroup
        int rs[3] = {0, 0, 0}, re[3] = {0, 0, 0};
        if (walks) row_runs(P, ncx, ncy, 0, P.cxy[t], 0u, rs, re);
        S = stage_plan(rs, re, s_red);
        staged = S.total <= kStageCap;
        if (staged) stage_copy(P, S, reinterpret_cast<double2 *>(mem));
    }
    template <int MODE>
    __device__ bool rates(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy, int t, const double4 &bt,
                          double &drho, double &ax, double &ay) {
        if constexpr (KERNEL != SPH_KERNEL_GAUSSIAN)
            if (staged)
                return uniform64_rates_staged<KERNEL, MODE>(P, K, ncx, ncy, t, bt, S,
                                                            reinterpret_cast<const double2 *>(mem),
                                                            reinterpret_cast<unsigned short *>(mem + kStageCap * 16),
                                                            drho, ax, ay);
        return uniform64_rates<KERNEL, MODE>(P, K, ncx, ncy, 0, t, bt, reinterpret_cast<unsigned *>(mem), drho, ax, ay);
    }
};

// One target t of the pass: its rates, or nothing for a wall or a target
// that keeps its previous rates; MODE selects the rates written.
template <int KERNEL, int MODE = kFused>
__device__ inline void uniform64_target(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy,
                                        long long base, int t, unsigned *s_list) {
    const double4 bt = P.B[t];
    if (not_fluid64(bt.w)) return;  // walls are not targets
    double drho, ax, ay;
    if (!uniform64_rates<KERNEL, MODE>(P, K, ncx, ncy, base, t, bt, s_list, drho, ax, ay)) return;
    if constexpr ((MODE & kEquations) != kMomentum) P.drho[t] = drho;
    if constexpr ((MODE & kEquations) != kContinuity) {
        P.ax[t] = ax;
        P.ay[t] = ay;
    }
}

template <int KERNEL, int MODE>
__global__ __launch_bounds__(256) void k_pair_uniform64(const Ctrl *ctrl, Uniform64Args P, Uniform64Const K) {
    __shared__ __align__(16) unsigned char s_mem[stage_bytes64<KERNEL>()];
    __shared__ int s_red[6 * 4];
    if (!ctrl->active) return;
    const int t = xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const Grid &g = ctrl->grid;
    const int ncx = (int)g.ncx, ncy = (int)g.ncy;
    double4 bt = make_double4(0.0, 0.0, 0.0, __builtin_nan(""));
    if (t < P.n) bt = P.B[t];
    const bool walks = t < P.n && !not_fluid64(bt.w);  // walls are not targets
    StagedWalk64<KERNEL> W(P, K, ncx, ncy, t, walks, s_mem, s_red);
    double drho, ax, ay;
    if (!walks || !W.template rates<MODE>(P, K, ncx, ncy, t, bt, drho, ax, ay)) return;
    if constexpr ((MODE & kEquations) != kMomentum) P.drho[t] = drho;
    if constexpr ((MODE & kEquations) != kContinuity) {
        P.ax[t] = ax;
        P.ay[t] = ay;
    }
}

// A batch target t: its instance's grid and constants. The lanes of a wave
// may hold targets of two (rarely more) instances; each pass of the loop
// takes the first remaining lane's instance, whose grid and constants are
// then the same for the whole pass (scalar registers, not one copy per
// lane), and runs the lanes of that instance. Every pass retires at least
// the lane it was chosen from.
template <int KERNEL>
__device__ inline void uniform64_target_batch(const BInst *inst, const int *instOf, const Uniform64Args &P, const Uniform64Const *Ks, int t,
                                   unsigned *s_list) {
    const int k = instOf[t];
    for (;;) {
        const int k0 = __builtin_amdgcn_readfirstlane(k);
        if (k == k0) {
            const BInst &I = inst[k0];
            if (I.active) uniform64_target<KERNEL>(P, Ks[k0], (int)I.grid.ncx, (int)I.grid.ncy, I.cellBase, t, s_list);
            break;
        }
    }
}

// The pass with PEC's corrector and the next dt's partials fused in, as the
// float pass's k_pair_uniform_pec (the corrector's arithmetic is the
// engine's, bit for bit).
template <int KERNEL, int MODE>
__global__ __launch_bounds__(256) void k_pair_uniform64_pec(Ctrl *ctrl, Uniform64Args P, Uniform64Const K,
                                                            PecArgs C) {
    __shared__ __align__(16) unsigned char s_mem[stage_bytes64<KERNEL>()];
    __shared__ double lds[kDtQ * 16];
    __shared__ int s_red[6 * 4];
    if (!ctrl->active) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctrl->dt_parts = kDtSlots;
        ctrl->pec_parts = 1;
    }
    const int t = xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const Grid &g = ctrl->grid;
    const int ncx = (int)g.ncx, ncy = (int)g.ncy;
    double4 bt = make_double4(0.0, 0.0, 0.0, __builtin_nan(""));
    if (t < P.n) bt = P.B[t];
    const bool walks = t < P.n && !not_fluid64(bt.w);
    StagedWalk64<KERNEL> W(P, K, ncx, ncy, t, walks, s_mem, s_red);
    DtVars v;
    if (walks) {
        const double dt = ctrl->dt, damping = ctrl->damping;
#if HIPSPH_PEC64_EARLY
        const PecStart p0 = pec_start(C, t, dt, damping);
#endif
        double drho, ax, ay;
        if (W.template rates<MODE>(P, K, ncx, ncy, t, bt, drho, ax, ay)) {
            P.drho[t] = drho;
            P.ax[t] = ax;
            P.ay[t] = ay;
        } else {
            drho = P.drho[t];
            ax = P.ax[t];
            ay = P.ay[t];
        }
        v.add(C.hc.on ? C.hc.h : C.s.h[t], ax, ay);
#if !HIPSPH_PEC64_EARLY
        const PecStart p0 = pec_start(C, t, dt, damping);
#endif
        pec_finish(C, t, p0, ax, ay, drho, dt, damping);
    }
    v.publish_slots(C.dslots, lds);
}

// The batched ensemble (one thread per slot, and the persistent work-queue
// form), as the float pass's k_pair_batch_uniform[_queue].
template <int KERNEL>
__global__ __launch_bounds__(256) void k_pair_batch_uniform64(const BInst *inst, const int *instOf, Uniform64Args P,
                                                              const Uniform64Const *Ks) {
    __shared__ unsigned s_list[uniform64_list<KERNEL>() * 256];
    const int t = xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (t >= P.n) return;
    uniform64_target_batch<KERNEL>(inst, instOf, P, Ks, t, s_list);
}

template <int KERNEL>
__global__ __launch_bounds__(256) void k_pair_batch_uniform64_queue(const BInst *inst, const int *instOf,
                                                                    Uniform64Args P, const Uniform64Const *Ks,
                                                                    int *queue) {
    __shared__ unsigned s_list[uniform64_list<KERNEL>() * 256];
    __shared__ int s_tile;
    const int ntiles = (int)((P.n + (long long)blockDim.x - 1) / blockDim.x);
    const int xcd = (int)(blockIdx.x % kXcds);
    const int per = (ntiles + kXcds - 1) / kXcds;
    const int lo = xcd * per;
    const int hi = lo + per < ntiles ? lo + per : ntiles;
    int *ctr = queue + xcd * kQueueStride;
    for (;;) {
        if (threadIdx.x == 0) s_tile = lo + atomicAdd(ctr, 1);
        __syncthreads();
        const int tile = s_tile;
        __syncthreads();  // every lane has read s_tile before lane 0 writes the next
        if (tile >= hi) break;
        const int t = tile * (int)blockDim.x + (int)threadIdx.x;
        if (t < P.n) uniform64_target_batch<KERNEL>(inst, instOf, P, Ks, t, s_list);
    }
    if (threadIdx.x == 0) {
        __threadfence();
        if (atomicAdd(queue + kXcds * kQueueStride, 1) == (int)gridDim.x - 1)
            for (int k = 0; k <= kXcds; ++k) atomicExch(queue + k * kQueueStride, 0);
    }
}


// The batched ensemble with PEC's corrector and the dt partials fused in:
// one workgroup per chunk (slots cs[c] .. cs[c + 1], at most 256 of one
// instance), so the instance's grid, constants and integrator fields are the
// same for the whole workgroup. The chunk's dt partials go to its instance's
// in C.part, where the batch's corrector puts them. An instance
// that is not active keeps its state; its fluid still enters the partials.
template <int KERNEL, int MODE>
__global__ __launch_bounds__(256) void k_pair_batch_uniform64_pec(const BInst *inst, const int *cs, const int *chunkInst, int NC,
                                                       Uniform64Args P, const Uniform64Const *Ks, PecArgs C) {
    __shared__ unsigned s_list[uniform64_list<KERNEL>() * 256];
    __shared__ double lds[kDtQ * 16];
    const int c = xcd_remap(blockIdx.x, gridDim.x);
    if (c >= NC) return;  // the whole workgroup
    const int k = chunkInst[c], entry = C.entry[c];
    const BInst &I = inst[k];
    DtVars v;
    const int t = cs[c] + (int)threadIdx.x;
    if (t < cs[c + 1]) {
        const double4 bt = P.B[t];
        if (!not_fluid64(bt.w)) {
            double drho, ax, ay;
            if (I.active) {
                const double dt = I.dt, damping = I.damping;
                PecArgs Ci = C;
                Ci.strict = I.strict;
#if HIPSPH_PEC64_EARLY
                const PecStart p0 = pec_start(Ci, t, dt, damping);
#endif
                if (uniform64_rates<KERNEL, MODE>(
                        P, Ks[k], (int)I.grid.ncx, (int)I.grid.ncy, I.cellBase, t, bt, s_list, drho, ax, ay)) {
                    P.drho[t] = drho;
                    P.ax[t] = ax;
                    P.ay[t] = ay;
                } else {
                    drho = P.drho[t];
                    ax = P.ax[t];
                    ay = P.ay[t];
                }
#if !HIPSPH_PEC64_EARLY
                const PecStart p0 = pec_start(Ci, t, dt, damping);
#endif
                pec_finish(Ci, t, p0, ax, ay, drho, dt, damping);
            } else {
                ax = P.ax[t];
                ay = P.ay[t];
            }
            v.add(I.uh_on ? I.uh : C.s.h[t], ax, ay);
        }
    }
    v.publish(C.part, entry, lds);
    if (c == 0 && threadIdx.x == 0 && C.mark) *C.mark = 1;
}

// ---------------------------------------------------------------------------
// G lanes per target (sph_pair_group.h)
// ---------------------------------------------------------------------------
template <int KERNEL, int MODE>
struct Uniform64Group {
    using RecA = double2;
    using Term = double;
    using Sum = PlainSum;
    static constexpr bool kDesc = true, kCount = true;  // counts every neighbour of a target outside the grid
    static constexpr int NQ = 5;  // drho, momentum and wall force along x and y
    const Uniform64Args &P;
    const Uniform64Const &K;
    double X, Y;
    double vx0, vy0, rho0, prs;  // the target's B record
    bool counts;
    __device__ __forceinline__ RecA load(unsigned u) const { return at32(P.A, u); }
    __device__ __forceinline__ bool test(const RecA &a, unsigned, bool &counted) const {
        const double dx = X - a.x, dy = Y - a.y;
        const double r2 = dx * dx + dy * dy;
        if (counts) {  // SolverTools.py:166-169
            const double lim = (K.qmax * K.h) * (K.qmax * K.h);
            counted = r2 < lim * (1.0 - 1e-12);
            if (!counted && !(r2 > lim * (1.0 + 1e-12))) counted = exact_q_test(X, Y, K.h, a.x, a.y, K.h, K.qmax);
        }
        return r2 <= K.lim2 && r2 > kPairNone;
    }
    // uniform64_rates' expressions for one listed pair. All five quantities are
    // returned together: stores into out from the fluid's and the
    // wall's branch became stores through a selected address, and out
    // 32 bytes of scratch memory.
    __device__ __forceinline__ void terms(unsigned u, double *out) const {
        double d = 0.0, a0 = 0.0, a1 = 0.0, f0 = 0.0, f1 = 0.0;
        pair(u, d, a0, a1, f0, f1);
        out[0] = d;
        out[1] = a0;
        out[2] = a1;
        out[3] = f0;
        out[4] = f1;
    }
    __device__ __forceinline__ void pair(unsigned u, double &d, double &a0, double &a1, double &f0, double &f1) const {
        const double2 a = at32(P.A, u);
        const double4 b = at32(P.B, u);
        const double dx = X - a.x, dy = Y - a.y;
        const double xij2 = dx * dx + dy * dy;
        double half;
        const double r = pair_root(xij2, half);
        if (!not_fluid64(b.w)) {
            const double qq = pair_quotient(r, K.h, K.hinv);
            double dwx, dwy;
            if (KERNEL == SPH_KERNEL_GAUSSIAN) {
                double f;
                if (!gauss_factor(xij2, K.h, K.ih2, K.g2, f)) return;
                dwx = f * dx;
                dwy = f * dy;
            } else {
                double grad;
                if (KERNEL == SPH_KERNEL_WENDLAND) {
                    if ((qq >= 2.0) || (r < 1e-10)) return;
                    const double inner = 1.0 - 0.5 * qq;
                    grad = ipow(inner, 5.0) * (-14.0 / 3.0) * qq * (1 + 2.5 * qq);
                } else {
                    if ((qq > 2.0) || (r < 1e-10)) return;
                    grad = (qq > 1.0) ? -0.75 * ((2.0 - qq) * (2.0 - qq)) : -3.0 * qq * (1.0 - 0.75 * qq);
                }
                const double hr = K.h * r;
                const double norm = pair_quotient(K.alpha_k * grad, hr, pair_recip(hr, half * K.hinv2));
                dwx = norm * dx;
                dwy = norm * dy;
            }
            const double vx = vx0 - b.x, vy = vy0 - b.y;
            const double dot = vx * dwx + vy * dwy;
            if constexpr ((MODE & kEquations) != kMomentum) d = K.m * dot;
            if constexpr ((MODE & kEquations) == kContinuity) return;
            const double dv = vx * dx + vy * dy;
            double PI_ij = 0.0;
            if (dv < 0) {
                const double rhoij = 0.5 * (rho0 + b.z);
                const double rr = KERNEL == SPH_KERNEL_GAUSSIAN ? xij2 : r * r;
                const double muij = K.h * dv / (rr + K.c01);
                const double ppij = muij * (K.beta * muij - K.alpha * K.cij);
                PI_ij = ppij / rhoij;
            }
            const double factor = prs + b.w + PI_ij;
            a0 = -K.m * factor * dwx;
            a1 = -K.m * factor * dwy;
        } else if ((MODE & kEquations) != kContinuity && !(r > K.r0) && r > 1e-12) {
            const double frac = K.r0 / r;
            const double tmp = wall_pow<MODE>(frac, K.p1) - wall_pow<MODE>(frac, K.p2);
            const double fac = K.D * tmp;
            f0 = fac * dx / (r * r);
            f1 = fac * dy / (r * r);
        }
    }
};

// The rates of target t by its G lanes, in the first of them; false: it has no
// neighbour (or walks is false).
template <int KERNEL, int MODE, int G>
__device__ inline bool uniform64_group_rates(const Uniform64Args &P, const Uniform64Const &K, int ncx, int ncy,
                                             const double2 &at, int2 c, const double4 &bt, bool walks, int l,
                                             GroupMem<Uniform64Group<KERNEL, MODE>, G> &M, double &drho, double &ax,
                                             double &ay) {
    using UG = Uniform64Group<KERNEL, MODE>;
    // a target whose own cell is in the grid finds itself (q = 0)
    const bool inside = c.x >= 0 && c.x < ncx && c.y >= 0 && c.y < ncy;
    const UG ug{P, K, at.x, at.y, bt.x, bt.y, bt.z, bt.w, !inside};
    GroupSums<UG, G> acc;
    int cnt;
    group_sums<UG, G>(ug, P.cellStart, c, ncx, ncy, 0, walks, l, M, acc, cnt);
    drho = acc.template get<0>();
    const double a0 = acc.template get<1>(), a1 = acc.template get<2>();
    const double f0 = acc.template get<3>(), f1 = acc.template get<4>();
    ax = a0 + f0;
    ay = (MODE & kEquations) == kContinuity ? 0.0 : (a1 - K.g) + f1;  // WCSPH.py:169, then SolverTools.py:170-171
    return walks && (inside || cnt != 0);  // SolverTools.py:166-169
}

template <int KERNEL, int MODE, int G>
__global__ __launch_bounds__(256) void k_group_uniform64(const Ctrl *ctrl, Uniform64Args P, Uniform64Const K) {
    __shared__ GroupMem<Uniform64Group<KERNEL, MODE>, G> mem[256 / G];
    const int i = threadIdx.x / G, l = threadIdx.x % G;
    const int t = xcd_remap(blockIdx.x, gridDim.x) * (256 / G) + i;
    const int t0 = t < P.n ? t : P.n - 1;
    const double4 bt = P.B[t0];  // the target's records together with the control block
    const double2 at = P.A[t0];
    const int2 c = P.cxy[t0];
    if (!ctrl->active) return;
    const bool walks = t < P.n && !not_fluid64(bt.w);
    const Grid &g = ctrl->grid;
    double drho, ax, ay;
    const bool any = uniform64_group_rates<KERNEL, MODE, G>(P, K, (int)g.ncx, (int)g.ncy, at, c, bt, walks, l, mem[i],
                                                            drho, ax, ay);
    if (!any || l != 0) return;
    if constexpr ((MODE & kEquations) != kMomentum) P.drho[t] = drho;
    if constexpr ((MODE & kEquations) != kContinuity) {
        P.ax[t] = ax;
        P.ay[t] = ay;
    }
}

// k_pair_uniform64_pec with G lanes per target; the group's first lane
// corrects.
template <int KERNEL, int MODE, int G>
__global__ __launch_bounds__(256) void k_group_uniform64_pec(Ctrl *ctrl, Uniform64Args P, Uniform64Const K,
                                                             PecArgs C) {
    __shared__ GroupMem<Uniform64Group<KERNEL, MODE>, G> mem[256 / G];
    __shared__ double lds[kDtQ * 16];
    const int i = threadIdx.x / G, l = threadIdx.x % G;
    const int t = xcd_remap(blockIdx.x, gridDim.x) * (256 / G) + i;
    const int t0 = t < P.n ? t : P.n - 1;
    const double4 bt = P.B[t0];  // the target's records together with the control block
    const double2 at = P.A[t0];
    const int2 c = P.cxy[t0];
    const int q = C.perm[t0];
    if (!ctrl->active) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctrl->dt_parts = kDtSlots;
        ctrl->pec_parts = 1;
    }
    const bool walks = t < P.n && !not_fluid64(bt.w);
    const Grid &g = ctrl->grid;
    const double dt = ctrl->dt, damping = ctrl->damping;
    const bool corrects = walks && l == 0;
    PecStart p0{};
    if (corrects) p0 = pec_start_from(C, q, dt, damping);  // in flight under the walk
    double drho, ax, ay;
    const bool any = uniform64_group_rates<KERNEL, MODE, G>(P, K, (int)g.ncx, (int)g.ncy, at, c, bt, walks, l, mem[i],
                                                              drho, ax, ay);
    DtVars v;
    if (corrects) {
        if (any) {
            P.drho[t] = drho;
            P.ax[t] = ax;
            P.ay[t] = ay;
        } else {
            drho = P.drho[t];
            ax = P.ax[t];
            ay = P.ay[t];
        }
        v.add(C.hc.on ? C.hc.h : C.s.h[t], ax, ay);
        pec_finish(C, t, p0, ax, ay, drho, dt, damping);
    }
    v.publish_slots(C.dslots, lds);
}

}  // namespace
}  // namespace hipsph
