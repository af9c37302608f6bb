// sph_common.h — device code shared by the single-simulation engine and the
// batched ensemble: workgroup reductions, the PEC half-step expressions, the
// Tait pressure, and the cell-sort pipeline (prefix scan of bin counts,
// scatter, per-bin rank sort). Included by more than one translation unit:
// everything is in an anonymous namespace, so each gets its own copy.
#pragma once
#include <type_traits>

#include "sph_internal.h"

namespace hipsph {
namespace {

// Host: calls f with the kernel id as a compile-time constant
// (std::integral_constant<int, id>), for launchers instantiated per kernel.
template <typename F>
inline void with_kernel(int kernel, F &&f) {
    switch (kernel) {
        case SPH_KERNEL_WENDLAND: f(std::integral_constant<int, SPH_KERNEL_WENDLAND>{}); break;
        case SPH_KERNEL_GAUSSIAN: f(std::integral_constant<int, SPH_KERNEL_GAUSSIAN>{}); break;
        default: f(std::integral_constant<int, SPH_KERNEL_CUBIC>{}); break;
    }
}

// ---------------------------------------------------------------------------
// reductions (wavefront shuffles, then LDS across the 4 waves of a block)
// ---------------------------------------------------------------------------
template <typename T, typename Op>
__device__ inline T wave_reduce(T v, Op op) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = op(v, __shfl_xor(v, o, 64));
    return v;
}

template <typename T, typename Op>
__device__ inline T block_reduce(T v, Op op, T *lds) {
    v = wave_reduce(v, op);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) lds[w] = v;
    __syncthreads();
    if (w == 0) {
        v = (lane < (int)(blockDim.x >> 6)) ? lds[lane] : Op::identity();
        v = wave_reduce(v, op);
    }
    __syncthreads();
    return v;  // valid in wave 0
}

struct AddOp {
    __device__ static double identity() { return 0.0; }
    __device__ double operator()(double a, double b) const { return a + b; }
};

template <class T>
__device__ inline T max_of(T a, T b) {
    return b > a ? b : a;
}

// Cross-lane moves of the vector ALU (an LDS permute each otherwise), for types of 4
// and 8 bytes: x of another lane of the same row of 16 lanes (a DPP control), and
// the upper lanes of a exchanged with the lower ones of b, over the
// wavefront's halves (ROWS 32) or each half's rows (16).
template <class T, class F>
__device__ inline T by_words(T x, F &&f) {
    if constexpr (sizeof(T) == 4) {
        const unsigned r = f(__builtin_bit_cast(unsigned, x));
        return __builtin_bit_cast(T, r);
    } else {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
        const unsigned lo = f((unsigned)b), hi = f((unsigned)(b >> 32));
        return __builtin_bit_cast(T, (unsigned long long)hi << 32 | lo);
    }
}
template <int CTRL, class T>
__device__ inline T row_move(T x) {
    return by_words(x, [](unsigned w) { return (unsigned)__builtin_amdgcn_mov_dpp((int)w, CTRL, 0xf, 0xf, false); });
}
template <int ROWS>
__device__ inline void row_swap(unsigned &a, unsigned &b) {
    if constexpr (ROWS == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    }
}
template <int ROWS, class T>
__device__ inline void row_swap(T &a, T &b) {
    if constexpr (sizeof(T) == 4) {
        unsigned x = __builtin_bit_cast(unsigned, a), y = __builtin_bit_cast(unsigned, b);
        row_swap<ROWS>(x, y);
        a = __builtin_bit_cast(T, x);
        b = __builtin_bit_cast(T, y);
    } else {
        const auto x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
        unsigned x0 = (unsigned)x, x1 = (unsigned)(x >> 32), y0 = (unsigned)y, y1 = (unsigned)(y >> 32);
        row_swap<ROWS>(x0, y0);
        row_swap<ROWS>(x1, y1);
        a = __builtin_bit_cast(T, (unsigned long long)x1 << 32 | x0);
        b = __builtin_bit_cast(T, (unsigned long long)y1 << 32 | y0);
    }
}
constexpr int kRor8 = 0x128, kRor4 = 0x124, kRor2 = 0x122, kRor1 = 0x121;  // rotations of a row
constexpr int kHalfMirror = 0x141, kQuadXor2 = 0x4e, kQuadXor1 = 0xb1;
template <class T>
__device__ inline T lane_value(T x, int lane) {  // of a lane that is the same for the wavefront
    return by_words(x, [&](unsigned w) { return (unsigned)__builtin_amdgcn_readlane((int)w, lane); });
}
// Of the lane before (lane 0: its own).
__device__ inline int lane_before(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x138, 0xf, 0xf, false); }
// The sum over the lanes up to this one; unsigned, since two sums packed into
// one word use its top bit.
template <int CTRL, int ROWS>
__device__ inline unsigned scan_step(unsigned x) {
    return x + (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
}
__device__ inline unsigned wave_scan(unsigned x) {
    x = scan_step<0x111, 0xf>(x);  // within the rows
    x = scan_step<0x112, 0xf>(x);
    x = scan_step<0x114, 0xf>(x);
    x = scan_step<0x118, 0xf>(x);
    x = scan_step<0x142, 0xa>(x);  // a row's last lane into the next row
    return scan_step<0x143, 0xc>(x);  // the lower half's into the upper
}

// f over the values of all lanes, in all of them: the pairs of an xor tree of
// 32, 16, ... 1 (f commutes), so a sum has that tree's bits.
template <class T, class F>
__device__ inline T row_fold(T x, F &&f) {
    x = f(x, row_move<kRor8>(x));
    x = f(x, row_move<kRor4>(x));
    x = f(x, row_move<kRor2>(x));
    return f(x, row_move<kRor1>(x));
}
template <class T, class F>
__device__ inline T wave_fold(T x, F &&f) {
    T y = x;
    row_swap<32>(x, y);
    x = f(x, y);
    y = x;
    row_swap<16>(x, y);
    return row_fold(f(x, y), f);
}
template <class T>
__device__ inline T wave_max(T x) {
    return wave_fold(x, [](T a, T b) { return max_of(a, b); });
}

// The maximum over each group of 64 / P lanes, in all of them (P: 4 or 8).
template <int P, class T>
__device__ inline T group_max(T x) {
    if constexpr (P == 8) {
        x = max_of(x, row_move<kHalfMirror>(x));
        x = max_of(x, row_move<kQuadXor2>(x));
        return max_of(x, row_move<kQuadXor1>(x));
    } else {
        return row_fold(x, [](T a, T b) { return max_of(a, b); });
    }
}
// The maxima over the wavefront of P quantities (4 or 8): that of quantity q in
// the q-th group of 64 / P lanes. Each exchange halves the quantities a lane
// carries: eight take 10 exchanges instead of 48.
template <int P, class T>
__device__ inline T wave_maxima(T (&m)[P]) {
#pragma unroll
    for (int q = 0; q < P / 2; ++q) {
        row_swap<32>(m[q], m[q + P / 2]);
        m[q] = max_of(m[q], m[q + P / 2]);
    }
#pragma unroll
    for (int q = 0; q < P / 4; ++q) {
        row_swap<16>(m[q], m[q + P / 4]);
        m[q] = max_of(m[q], m[q + P / 4]);
    }
    if constexpr (P == 8) {
        const bool up = threadIdx.x & 8;
        const T mine = up ? m[1] : m[0], other = up ? m[0] : m[1];
        m[0] = max_of(mine, row_move<kRor8>(other));
    }
    return group_max<P>(m[0]);
}

// Fold NQ (at most 8) quantities over a whole workgroup (up to 16
// wavefronts). kind: 0 min, 1 max, 2 a count of which only zero or not is
// kept: all are taken as maxima (the minima negated), inside a wavefront by
// wave_maxima (as 96 LDS permutes per wavefront they kept a CU's LDS pipe busy for 3
// us in the bounds kernels); one LDS round, then wavefront 0
// folds the wavefronts' values, a group of lanes per quantity. block_maxima: the
// maximum of quantity q in the q-th group of fold_lanes lanes of wavefront 0.
// block_fold: the results in all lanes of wavefront 0. lds holds P * 16 doubles, P
// the next of 4 and 8.
template <int NQ>
constexpr int fold_lanes() {
    return NQ <= 4 ? 16 : 8;
}
template <int NQ>
__device__ inline double block_maxima(const double (&v)[NQ], const int (&kind)[NQ], double *lds) {
    constexpr int P = NQ <= 4 ? 4 : 8, L = fold_lanes<NQ>();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    double m[P];
#pragma unroll
    for (int q = 0; q < P; ++q) m[q] = q < NQ ? (kind[q < NQ ? q : 0] == 0 ? -v[q < NQ ? q : 0] : v[q < NQ ? q : 0]) : -INFINITY;
    const double top = wave_maxima<P>(m);
    if (lane % L == 0) lds[(lane / L) * 16 + w] = top;
    __syncthreads();
    if (w != 0) return 0.0;
    double x = -INFINITY;
#pragma unroll
    for (int u = 0; u < 16; u += L)
        if (u + lane % L < nw) x = max_of(x, lds[(lane / L) * 16 + u + lane % L]);
    return group_max<P>(x);
}
template <int NQ>
__device__ inline void block_fold(double (&v)[NQ], const int (&kind)[NQ], double *lds) {
    const double x = block_maxima<NQ>(v, kind, lds);
    if (threadIdx.x >= 64) return;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const double r = lane_value(x, q * fold_lanes<NQ>());
        v[q] = kind[q] == 0 ? -r : r;
    }
}

// Per-workgroup partials of NQ quantities in one LDS round (block_fold):
// thread 0 stores part[q * R + k]. lds as block_fold's.
template <int NQ>
__device__ inline void block_partials(double (&v)[NQ], const int (&kind)[NQ], double *lds, double *part, int R,
                                      int k) {
    block_fold<NQ>(v, kind, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) part[q * R + k] = v[q];
    }
}

// Doubles as unsigned integers of the same order (no NaN), and back.
__device__ inline unsigned long long order_key(double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x + 0.0);  // -0.0 as 0.0
    return b ^ ((b >> 63) ? ~0ull : 0x8000000000000000ull);
}
__device__ inline double order_value(unsigned long long k) {
    return __longlong_as_double((long long)(k ^ ((k >> 63) ? 0x8000000000000000ull : ~0ull)));
}

// A workgroup's maxima of NQ quantities (block_maxima) as order keys into
// p[0 .. NQ), or raised there (shared).
template <int NQ>
__device__ inline void publish_maxima(const double (&v)[NQ], const int (&kind)[NQ], double *lds, unsigned long long *p,
                                      bool shared) {
    const double x = block_maxima<NQ>(v, kind, lds);
    const int t = threadIdx.x, q = t / fold_lanes<NQ>();
    if (t >= 64 || t % fold_lanes<NQ>() || q >= NQ) return;
    if (shared)
        atomicMax(p + q, order_key(x));
    else
        p[q] = order_key(x);
}

// src/Integrators/PEC.py:32-59 (useXSPH = False branch), one particle. The
// fused step evaluates the same expressions inside the neighbour update.
__device__ inline double pec_half_pos(double x, double v, double dt) { return x + 0.5 * dt * v; }
__device__ inline double pec_half_vel(double v, double a, double dt, double damping) {
#pragma clang fp contract(off)  // the integrator's arithmetic in every unit that inlines it
    return (v + 0.5 * dt * a) / (1 + 0.5 * damping);
}

// src/Integrators/PEC.py:61-89, one fluid particle from its start-of-step
// state (x0 ... rho0), the velocity that moved it in the predictor (mvx, mvy:
// the half-step velocity, or the XSPH velocity with useXSPH) and this step's
// rates: writes x, y, vx, vy, rho of slot j.
__device__ inline void pec_correct(const State &s, int j, double x0, double y0, double vx0, double vy0, double rho0,
                                   double mvx, double mvy, double ax, double ay, double drho, double dt,
                                   double damping, int strict) {
#pragma clang fp contract(off)
    double mid_x = x0 + 0.5 * dt * mvx;
    double mid_y = y0 + 0.5 * dt * mvy;
    double mid_vx = (vx0 + 0.5 * dt * ax) / (1 + 0.5 * damping);
    double mid_vy = (vy0 + 0.5 * dt * ay) / (1 + 0.5 * damping);
    s.x[j] = 2 * mid_x - x0;
    s.y[j] = 2 * mid_y - y0;
    s.vx[j] = 2 * mid_vx - vx0;
    s.vy[j] = 2 * mid_vy - vy0;
    double mid_rho = rho0 + 0.5 * dt * drho;
    double r = 2 * mid_rho - rho0;
    if (strict && r < 0.0) r = 0.0;
    s.rho[j] = r;
}

// The corrector of fluid slot j after a lean reorder: the start-of-step state
// from the previous buffer at the particle's previous slot, the half-step
// velocity formed again there (the predictor's expression). Loaded by
// pec_start (before the pair walk, so that the gathers are in flight under
// it), applied by pec_finish.
struct PecStart {
    double x0, y0, vx0, vy0, rho0, vxh, vyh;
};
__device__ inline PecStart pec_start_from(const PecArgs &C, int q, double dt, double damping) {
    PecStart p;
    p.x0 = C.o.x[q];
    p.y0 = C.o.y[q];
    p.vx0 = C.o.vx[q];
    p.vy0 = C.o.vy[q];
    p.rho0 = C.o.rho[q];
    p.vxh = pec_half_vel(p.vx0, C.o.ax[q], dt, damping);
    p.vyh = pec_half_vel(p.vy0, C.o.ay[q], dt, damping);
    return p;
}
__device__ inline PecStart pec_start(const PecArgs &C, int j, double dt, double damping) {
    return pec_start_from(C, C.perm[j], dt, damping);
}
__device__ inline void pec_finish(const PecArgs &C, int j, const PecStart &p, double ax, double ay, double drho,
                                  double dt, double damping) {
    pec_correct(C.s, j, p.x0, p.y0, p.vx0, p.vy0, p.rho0, p.vxh, p.vyh, ax, ay, drho, dt, damping, C.strict);
}

// time step: src/Equations/TimeStep.py:58-90 computeVars over the fluid
// (min h, max |a|^2, count, non-finite count), one workgroup's partials.
struct DtVars {
    double mn = INFINITY, mx = -INFINITY, cnt = 0.0, bad = 0.0;
    __device__ void add(double h, double ax, double ay) {
#pragma clang fp contract(off)
        double a2 = ax * ax + ay * ay;
        if (h < mn) mn = h;
        if (a2 > mx) mx = a2;
        if (!(a2 == a2)) bad += 1.0;
        cnt += 1.0;
    }
    // this workgroup's partials as entry k of R (one LDS round, plain
    // stores: part[q * R + k]); lds holds kDtQ * 16 doubles
    __device__ void store(double *part, int R, int k, double *lds) {
        const int kind[kDtQ] = {0, 1, 2, 2};
        double v[kDtQ] = {mn, mx, cnt, bad};
        block_partials<kDtQ>(v, kind, lds, part, R, k);
    }
    __device__ void publish(double *part, double *lds) { store(part, gridDim.x, blockIdx.x, lds); }
    // a batch tile's, into entry e of its instance's (kDtQ order keys, the
    // minimum as a maximum), or into ~e, which other tiles share
    __device__ void publish(unsigned long long *part, int e, double *lds) {
        const int kind[kDtQ] = {0, 1, 2, 2};
        const double v[kDtQ] = {mn, mx, cnt, bad};
        publish_maxima<kDtQ>(v, kind, lds, part + (size_t)kDtQ * (e < 0 ? ~e : e), e < 0);
    }
    // into the dt slots (one h for every particle: min h is not folded).
    // |a|^2 >= 0 orders as its bits. lds holds 4 * 16 doubles.
    __device__ void publish_slots(unsigned long long *d, double *lds) {
        const int kind[3] = {1, 2, 2};
        double v[3] = {mx, cnt, bad};
        block_fold<3>(v, kind, lds);
        if (threadIdx.x == 0 && v[1] > 0.0) {
            unsigned long long *p = d + (size_t)(blockIdx.x % kDtSlotCount) * kDtStride;
            if (v[0] >= 0.0) atomicMax(p, (unsigned long long)__double_as_longlong(v[0]));
            atomicOr(p + 1, kDtAny | (v[2] > 0.0 ? kDtBad : 0ull));
        }
    }
};
// Solver._minTimeStep (src/Solver.py:210-230): courant (TimeStep.py:47-49),
// force (:51-56), min(c, f) (:45), from the folded fluid reduction v. Also
// opens the step: the reference's loop condition `while self.t <
// self.duration` (src/Solver.py:366) and `self.t += self.dt` (:409) move
// here, so a step needs no host. It also bounds how far
// this step's predictor puts any particle from where the last update binned
// it (disp, for the border-cell bounds): after the fused PEC pass of the last
// step (ctrl->pec_parts; dt0 its dt, V = ctrl->vbound its velocity bound at the
// start, A0 = ctrl->abound its predictor's rates, A1 this fold's), a fluid
// particle binned at x + dt0 v / 2 was corrected to x + dt0 vh, with |vh| <=
// V + dt0 A0 / 2 (damping only shrinks it), and its new velocity v' has
// |v'| <= V + dt0 A1, so per axis it now lies within dt0 (V + dt0 A0 / 2) +
// dt0 V / 2 of where it was binned and this step's predictor moves it dt |v'|
// / 2 further; V + dt0 A1 bounds the next step's start. Anything else (other
// partials, non-finite rates, a halted step, a second call on the same
// partials) leaves +inf: the next update scans every particle. Changes nothing
// itself. C: the control block, or a batch instance with its ensemble's
// pec_parts.
struct DtIn {  // the control fields of the decision, loaded before the fold
    double t, dt, dt_c, dt_f, duration, fixed_dt, co, V, A0;
    long long step;
    unsigned flags;
    int advance_t, pec;
    template <typename C>
    __device__ DtIn(const C &c, int pec_parts)
        : t(c.t), dt(c.dt), dt_c(c.dt_c), dt_f(c.dt_f), duration(c.duration), fixed_dt(c.fixed_dt), co(c.co),
          V(c.vbound), A0(c.abound), step(c.step), flags(c.flags), advance_t(c.advance_t), pec(pec_parts) {}
};
__device__ inline DtNext dt_decide(const DtIn &in, const double *v, double gamma_c, double gamma_f) {
    DtNext x;
    x.t = in.t;
    x.dt = in.dt;
    x.dt_c = in.dt_c;
    x.dt_f = in.dt_f;
    x.step = in.step;
    x.disp = x.vbound = x.abound = INFINITY;
    x.flags = 0;
    x.active = 0;
    const double mn = v[0], mx = v[1], cnt = v[2], bad = v[3];
    const unsigned halt = SPH_FLAG_CAPACITY | SPH_FLAG_NONFINITE | SPH_FLAG_NO_FLUID | SPH_FLAG_ZERO_DENSITY;
    if ((in.flags & halt) || !(x.t < in.duration)) return x;
    if (cnt == 0) {
        x.flags = SPH_FLAG_NO_FLUID;
        return x;
    }
    if (bad != 0) x.flags |= SPH_FLAG_NONFINITE;
    double dt, c, f;
    if (in.fixed_dt > 0.0) {
        dt = in.fixed_dt;  // src/Solver.py:370-372
        c = 0.0;
        f = 0.0;
    } else {
        const double max_c = in.co;  // c = co for every fluid particle (WCSPH.py:110-129)
        c = gamma_c * mn / max_c;
        f = (mx < 1e-12) ? 1e10 : gamma_f * sqrt(mn / mx);
        dt = (f < c) ? f : c;
        if (dt < 1e-6) x.flags |= SPH_FLAG_DT_SMALL;  // src/Solver.py:220-224
    }
    const double dt0 = x.dt;
    x.dt = dt;
    x.dt_c = c;
    x.dt_f = f;
    if (in.advance_t) x.t = x.t + dt;
    x.step = x.step + 1;
    x.active = 1;
    if (bad == 0) {
        const double A1 = sqrt(mx);
        x.abound = A1;
        if (in.pec) {
            const double V1 = in.V + dt0 * A1;
            const double d = dt0 * (in.V + 0.5 * dt0 * in.A0) + 0.5 * dt0 * in.V + 0.5 * dt * V1;
            if (d == d) x.disp = d;  // NaN: +inf
            x.vbound = V1;
        }
    }
    return x;
}

// _get_cell_size :103-110 and _get_number_of_cells :112-127 from the folded
// bounds. Returns the halt flag (0: the grid is valid).
__device__ inline unsigned derive_grid(const double *v, double scale, long long cap, Grid &g) {
    const double xmn = v[0], xmx = v[1], ymn = v[2], ymx = v[3], hmn = v[4], hmx = v[5], bad = v[6];
    g.xmin = xmn;
    g.xmax = xmx;
    g.ymin = ymn;
    g.ymax = ymx;
    double cell_size = hmn * scale;
    if (cell_size < 1e-6) cell_size = 1.0;
    g.cs = cell_size;
    g.uniform_h = hmn == hmx;
    double cell_size1 = 1. / cell_size;
    double fx = ceil(cell_size1 * (xmx - xmn));
    double fy = ceil(cell_size1 * (ymx - ymn));
    if (bad != 0.0 || !(fx < 2.0e9) || !(fy < 2.0e9)) return SPH_FLAG_NONFINITE;
    long long ncx = (long long)fx, ncy = (long long)fy;
    if (ncx < 1) ncx = 1;
    if (ncy < 1) ncy = 1;
    g.ncx = ncx;
    g.ncy = ncy;
    g.ncells = ncx * ncy;
    return g.ncells > cap ? SPH_FLAG_CAPACITY : 0u;
}

__device__ inline double pec_half_rho(double rho, double drho, double dt, int strict) {
    double r = rho + 0.5 * dt * drho;
    if (strict && r < 0.0) r = 0.0;
    return r;
}

// src/Integrators/NewmarkBeta.py:41-66, one coupled particle: the predictor
// x + v dt + a (1/2 - beta) dt^2, v + a (1 - gamma) dt and the corrector
// x + a beta dt^2, v + a gamma dt, left to right, dt^2 the product dt dt (a
// power with the integer literal 2 in the numba source).
__device__ inline double nm_pred_pos(double x, double v, double a, double beta, double dt) {
    return x + v * dt + a * (0.5 - beta) * (dt * dt);
}
__device__ inline double nm_pred_vel(double v, double a, double gamma, double dt) { return v + a * (1 - gamma) * dt; }
__device__ inline double nm_corr_pos(double x, double a, double beta, double dt) { return x + a * beta * (dt * dt); }
__device__ inline double nm_corr_vel(double v, double a, double gamma, double dt) { return v + a * gamma * dt; }

// Runs of equal bins in lane order. A run also breaks where the reference
// index drops (consecutive slots from two old cells), so every run is in
// reference-index order; a bin that receives two runs is flagged for
// bin_place. leader: the first lane of this lane's run; next: the lane after
// its last.
__device__ inline void bin_run(int b, int id, int &leader, int &next) {
    const int lane = threadIdx.x & 63;
    const int prev = lane_before(b), prev_id = lane_before(id);
    const unsigned long long heads = __ballot(lane == 0 || b != prev || id < prev_id);
    const unsigned long long upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
    leader = 63 - __clzll(heads & upto);
    const unsigned long long after = heads & ~upto;
    next = after ? __ffsll((long long)after) - 1 : 64;
}

// Exclusive prefix scan of counts[0 .. ncells] into cellStart, in tiles of
// kScanTile bins: the keys kernels add their particles to their tiles' sums
// as well, so each tile's workgroup reads the sums before it and its own
// counts in one round of loads. (A kernel of its own for the tile sums took
// 4.6 us and its launch.) A workgroup's particles lie in one tile or two: those
// of its first particle's tile are added up in LDS, and the sums
// lie kTileStride apart, since the atomics of a line go one after another
// (one per wavefront on packed sums: the 1M dam break's keys take 41 us instead of
// 16). Called by the whole workgroup;
// tile: that of the thread's particle, or -1 (not the first thread's).
constexpr int kTileStride = 4;
__device__ inline void tile_add(int *tileSums, int tile) {
    __shared__ int s_tile, s_sum;
    if (threadIdx.x == 0) {
        s_tile = tile;
        s_sum = 0;
    }
    __syncthreads();
    const unsigned long long same = __ballot(tile == s_tile);
    if ((threadIdx.x & 63) == 0 && same) atomicAdd(&s_sum, __popcll(same));
    const int other = tile == s_tile ? -1 : tile;
    if (__ballot(other >= 0)) {
        int leader, next;
        bin_run(other, 0, leader, next);
        if ((int)(threadIdx.x & 63) == leader && other >= 0)
            atomicAdd(&tileSums[(size_t)other * kTileStride], next - leader);
    }
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&tileSums[(size_t)s_tile * kTileStride], s_sum);
}
__device__ inline unsigned block_scan_excl(unsigned v, unsigned *lds, unsigned *total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned s = wave_scan(v);
    if (lane == 63) lds[w] = s;
    __syncthreads();
    int nw = blockDim.x >> 6;
    unsigned off = 0, tot = 0;
    for (int k = 0; k < nw; ++k) {
        const unsigned ws = lds[k];
        if (k < w) off += ws;
        tot += ws;
    }
    __syncthreads();
    *total = tot;
    return off + s - v;
}
__device__ inline int block_scan_excl(int v, int *lds, int *total) {
    unsigned tot;
    const unsigned ex = block_scan_excl((unsigned)v, reinterpret_cast<unsigned *>(lds), &tot);
    *total = (int)tot;
    return (int)ex;
}

// Tile `tile` of the scan of nbins counts, from `first` on (workgroups of
// kBlock threads, four bins each; counts and cellStart from a multiple of four bins,
// with whole rows of four). Clears its counts for the next update. lds holds 16 ints.
__device__ inline void scan_tile(int *counts, const int *tileSums, int *cellStart, long long nbins, long long tile,
                                 int first, int *lds) {
    const long long b0 = tile * kScanTile + (long long)threadIdx.x * kScanItems;
    int4 c = b0 < nbins ? *reinterpret_cast<const int4 *>(counts + b0) : make_int4(0, 0, 0, 0);
    int pre = 0;
    constexpr int U = 4;  // loads in flight
    for (long long j = threadIdx.x; j < tile; j += U * kBlock) {
        int t[U];
#pragma unroll
        for (int u = 0; u < U; ++u) t[u] = j + u * kBlock < tile ? tileSums[(j + u * kBlock) * kTileStride] : 0;
#pragma unroll
        for (int u = 0; u < U; ++u) pre += t[u];
    }
    int tot, sum;
    block_scan_excl(pre, lds, &tot);
    if (b0 + 1 >= nbins) c.y = 0;  // past the last bin
    if (b0 + 2 >= nbins) c.z = 0;
    if (b0 + 3 >= nbins) c.w = 0;
    const int v[kScanItems] = {c.x, c.y, c.z, c.w};
    int ex = block_scan_excl(c.x + c.y + c.z + c.w, lds, &sum) + tot + first;
    if (b0 < nbins) *reinterpret_cast<int4 *>(counts + b0) = make_int4(0, 0, 0, 0);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (b0 + k < nbins) cellStart[b0 + k] = ex;
        ex += v[k];
    }
    // the end of the last bin
    if (b0 < nbins && b0 + kScanItems >= nbins) cellStart[nbins] = ex;
}

__global__ __launch_bounds__(kBlock) void k_scan(const Ctrl *ctrl, int *counts, const int *tileSums, int *cellStart) {
    if (!ctrl->active) return;
    __shared__ int lds[16];
    const long long nbins = ctrl->grid.ncells + 1;
    for (long long tile = blockIdx.x; tile * kScanTile < nbins; tile += gridDim.x)
        scan_tile(counts, tileSums, cellStart, nbins, tile, 0, lds);
}

// Share i of S of the exclusive scan of counts[0 .. nbins) (16-byte aligned)
// into cellStart: the workgroup sums what lies before its share itself, the
// counts or, in a grid of more than kPlainBins (whose keys left them), the
// tiles' sums, and scans its share, four bins per thread. lds holds 16 ints.
constexpr int kPlainBins = 1 << 17;
__device__ inline void scan_share(const int *counts, const int *tileSums, int *cellStart, int nbins, int i, int S,
                                  unsigned *lds) {
    const bool tiles = nbins > kPlainBins;
    const int unit = tiles ? kScanTile : 4;
    const int share = ((nbins + S - 1) / S + unit - 1) / unit * unit;
    const long long at = (long long)i * share;
    if (at >= nbins) return;
    const int b0 = (int)at, b1 = nbins - b0 > share ? b0 + share : nbins;
    unsigned pre = 0;
    const int step = 4 * (int)blockDim.x;
    if (tiles) {
        for (int j = threadIdx.x; j < b0 / kScanTile; j += blockDim.x) pre += (unsigned)tileSums[(size_t)j * kTileStride];
    } else {
        constexpr int U = 8;  // loads in flight per thread
        for (int j = 4 * (int)threadIdx.x; j < b0; j += U * step) {  // b0 is a multiple of 4
            int4 c[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                c[u] = j + u * step < b0 ? *reinterpret_cast<const int4 *>(counts + j + u * step)
                                         : make_int4(0, 0, 0, 0);
#pragma unroll
            for (int u = 0; u < U; ++u) pre += (unsigned)(c[u].x + c[u].y + c[u].z + c[u].w);
        }
    }
    unsigned run, tot;
    block_scan_excl(pre, lds, &run);  // run: the sum before the share
    for (int b = b0; b < b1; b += step) {
        const int k = b + 4 * (int)threadIdx.x;
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = k + u < b1 ? counts[k + u] : 0;
        int ex = (int)(block_scan_excl((unsigned)(v[0] + v[1] + v[2] + v[3]), lds, &tot) + run);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (k + u < b1) cellStart[k + u] = ex;
            ex += v[u];
        }
        run += tot;
    }
}

constexpr int kScanThreads = 1024;  // of the kernels that use scan_share

// Each particle's place from its bin's offset and its rank there: perm0 maps
// places to slots. Inside a bin the order is that of the ranks' atomics;
// bin_place orders it. Also zeroes the tile sums for the next update. The bounds slots, folded by now, are cleared for the next
// update too, active or not (a halted step's k_bounds may have filled them).
__global__ void k_place(const Ctrl *ctrl, const int *cellStart, const int *bin, const int *rank, int *perm0, int n,
                        int *tiles, unsigned long long *bslots) {
    if (blockIdx.x == 0 && threadIdx.x < kBoundsSlots * kBoundsStride) bslots[threadIdx.x] = 0;
    if (!ctrl->active) return;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    for (long long j = t; j * kScanTile <= ctrl->grid.ncells; j += (long long)gridDim.x * blockDim.x)
        tiles[j * kTileStride] = 0;
    if (t < n) perm0[cellStart[bin[t]] + rank[t]] = t;
}

// The place of the particle that k_place put at t, with its bin in order of
// the reference index (what the reference's head-inserted lists are ordered
// by, descending there; the pair pass walks the bin backwards): the bin's
// start plus the number of smaller indices in it. Only a bin filled by more
// than one run of k_keys (binflag[b] holds this update's epoch) can be out
// of order. The places of a bin are consecutive, so its indices are mostly in
// other lanes of the wavefront and are compared there; a bin that crosses
// into the next wavefront reads them through perm0. (A kernel of its own for
// the flagged bins took 8.9 us on the 1M dam break and its permuted indices
// 1.4 us in the scatter; here the reorder takes 39.9 us instead of 34.0.)
// Called by every thread with t < n of a wavefront of consecutive t together (my: its particle's
// index).
__device__ inline int bin_place(int t, int my, long long b, const int *cellStart, const int *binflag, int epoch,
                                const int *perm0, const int *id) {
    const int lane = threadIdx.x & 63, t0 = t - lane;
    const bool flagged = binflag[b] == epoch;
    int s = t, e = t;
    if (flagged) {
        s = cellStart[b];
        e = cellStart[b + 1];
    }
    const bool inside = s >= t0 && e <= t0 + 64;
    const int len = flagged && inside ? e - s : 0;
    int r = 0;
    for (int j = 0; __ballot(j < len) != 0; ++j) {  // every lane takes part in every exchange
        const int other = __shfl(my, (s - t0 + j) & 63, 64);
        r += j < len && other < my;
    }
    if (!flagged) return t;
    if (inside) return s + r;
    int j = s;
    for (; j + 4 <= e; j += 4) {
        int q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = perm0[j + u];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = id[q[u]];
#pragma unroll
        for (int u = 0; u < 4; ++u) r += q[u] < my;
    }
    for (; j < e; ++j) r += id[perm0[j]] < my;
    return s + r;
}

// _bin's cell of a position (src/Tools/NNLinkedList.py:146-176): floor of
// the true quotient per axis, clamped only for the int conversion (any
// clamped value is far outside the grid). The keys kernels and the reorders
// both call it, so a particle's stored cell is the one it was binned by.
__device__ inline int2 cell_of(double x, double y, const Grid &g) {
    double fx = floor((x - g.xmin) / g.cs);
    double fy = floor((y - g.ymin) / g.cs);
    // clamped so the integer conversion is defined; NaN goes below the grid
    fx = !(fx >= -1.0e9) ? -1.0e9 : (fx > 1.0e9 ? 1.0e9 : fx);
    fy = !(fy >= -1.0e9) ? -1.0e9 : (fy > 1.0e9 ? 1.0e9 : fy);
    return make_int2((int)(long long)fx, (int)(long long)fy);
}

// The border-cell bounds (after a fused PEC step; see border_bounds_may in
// the engine): the margin test, 2 disp under the cell size by far more than
// the rounding of positions and cell arithmetic (false for +inf and NaN), on
// a grid of at least 3 x 3 cells (the caller's test).
__device__ inline bool border_margin_ok(const Grid &g, double disp) {
    const double slack = 1e-12 * (fabs(g.xmin) + fabs(g.xmax) + fabs(g.ymin) + fabs(g.ymax));
    return 2.0 * disp * (1.0 + 1e-6) + slack < g.cs * (1.0 - 1e-6);
}

// The slots of the border cells of grid g (bins from cb, offsets in
// cellStart), shared by nthreads threads (tid in [0, nthreads), nthreads a
// multiple of 64): rows 0, ncy - 2, ncy - 1 and the out-of-grid bin, one
// slot range, thread-strided (it also holds what a flat key carries past the
// last row); and for each row r <= ncy - 3 the run of columns ncx - 2,
// ncx - 1 of row r and column 0 of row r + 1 (consecutive keys: one slot
// range, one wavefront; it also holds what a flat key carries past the last
// column into the next row). take(slot) for each.
// The first slot of each kind is known on construction (-1: none), so that
// a caller can load it while it still decides; rest takes the others.
struct BorderWalk {
    const int *start;
    long long ncx, ncy, cb;
    int tid, nthreads, a0, la, b0, lab, s0 = 0, s1 = 0;
    __device__ BorderWalk(const int *cellStart, long long cb_, const Grid &g, int tid_, int nthreads_)
        : start(cellStart), ncx(g.ncx), ncy(g.ncy), cb(cb_), tid(tid_), nthreads(nthreads_) {
        a0 = start[cb];
        const int a1 = start[cb + ncx], b1 = start[cb + g.ncells + 1];
        b0 = start[cb + (ncy - 2) * ncx];
        if ((tid >> 6) <= ncy - 3) run(tid >> 6, s0, s1);
        la = a1 - a0;
        lab = la + (b1 - b0);
    }
    __device__ void run(long long r, int &x0, int &x1) const {
        x0 = start[cb + r * ncx + ncx - 2];
        x1 = start[cb + (r + 1) * ncx + 1];
    }
    __device__ int at(int j) const { return j < la ? a0 + j : b0 + (j - la); }
    __device__ int first_row() const { return tid < lab ? at(tid) : -1; }
    __device__ int first_run() const { return s0 + (tid & 63) < s1 ? s0 + (tid & 63) : -1; }
    template <class F>
    __device__ void rest(F &&take) const {
        for (int j = tid + nthreads; j < lab; j += nthreads) take(at(j));
        const int lane = tid & 63;
        for (int i = s0 + lane + 64; i < s1; i += 64) take(i);
        for (long long r = (tid + nthreads) >> 6; r <= ncy - 3; r += nthreads >> 6) {
            int x0, x1;
            run(r, x0, x1);
            for (int i = x0 + lane; i < x1; i += 64) take(i);
        }
    }
};

// Tait pressure + Pb (src/Equations/TaitEOS.py:6-31; WCSPH.py:131-149).
__device__ inline double tait_p(double rho, int8_t label, double gamma, double B, double rho0, double Pb) {
    double p = 0.0;
    if (label == kFluid) {
        double ratio = ipow(rho / rho0, gamma);
        p = (ratio - 1.0) * B;
    }
    return p + Pb;
}

// The packed pair-pass records of slot t in format fmt (kRecFp64,
// kRecFp32, kRecUniform): w = m for fluid and -label otherwise; p / rho^2
// with p the Tait pressure + Pb (src/Tools/SolverTools.py:122-127,
// src/Equations/Momentum.py:28,36). Returns p / rho^2.
__device__ inline double write_pair_records(int t, double x, double y, double vx, double vy, double rho, double m,
                                            double h, int8_t lab, const Phys &ph, int fmt, void *recA, void *recB) {
    const double p = tait_p(rho, lab, ph.gamma, ph.B, ph.rho0, ph.Pb);
    const double pr = p / (rho * rho);
    const double w = lab == kFluid ? m : -(double)lab;
    if (fmt == kRecUniform) {
        ((double2 *)recA)[t] = make_double2(x, y);
        ((float4 *)recB)[t] = make_float4((float)vx, (float)vy, (float)rho,
                                          lab == kFluid ? (float)pr : __int_as_float(0x7fc00000));
    } else if (fmt == kRecUniform64) {
        ((double2 *)recA)[t] = make_double2(x, y);
        ((double4 *)recB)[t] = make_double4(vx, vy, rho, lab == kFluid ? pr : __longlong_as_double(0x7ff8000000000000ll));
    } else if (fmt == kRecFp32) {
        Rec<float>::A ra;
        ra.x = x;
        ra.y = y;
        ra.h = (float)h;
        ra.w = (float)w;
        ra.vx = (float)vx;
        ra.vy = (float)vy;
        ((Rec<float>::A *)recA)[t] = ra;
        ((Rec<float>::B *)recB)[t] = Rec<float>::B{(float)rho, (float)pr};
    } else {
        ((Rec<double>::A *)recA)[t] = Rec<double>::A{x, y, h, w};
        ((Rec<double>::B *)recB)[t] = Rec<double>::B{vx, vy, rho, pr};
    }
    return pr;
}

// ---------------------------------------------------------------------------
// staged walks of the uniform pair passes
// ---------------------------------------------------------------------------
// Staged walk: the A records of the slot ranges a workgroup's targets walk,
// one range per row offset, are copied to LDS once (coalesced) and the walk
// and the flush read them there (the scattered 16-byte loads of the walk
// kept the vector memory path of the float pass 80 % busy); a workgroup
// whose ranges hold more than STAGE_CAP records walks global memory instead.
// 1024 (16 KB; the 1M dam break's workgroups need about 800): 5 workgroups
// per CU, as many as the fused float pass's 81 registers allow. Staging B as
// well (3 workgroups per CU) or a shorter list (a flush mid-walk in most
// threads) cost more than the walk saves. Workgroups of at most 256 threads.
#ifndef HIPSPH_STAGE_CAP
#define HIPSPH_STAGE_CAP 1024
#endif
constexpr int kStageCap = HIPSPH_STAGE_CAP;
static_assert(kStageCap > 0 && kStageCap < 65536, "LDS indices are 16-bit");

// Which diagonal neighbour cells of a target at (X, Y) in cell c lie wholly
// beyond the listing radius (r^2 > lim2 for every point of the cell): bit 0
// below left, 1 below right, 2 above left, 3 above right. With cells 2h wide
// and the radius 2h, about a fifth of them (the target near its cell's
// centre); their particles could only be candidates that fail the test, so
// skipping them leaves every sum as it was. Distances to the cell edges are
// taken 1e-9 cs short of the computed ones, far more than the rounding of
// cell_of's floor((x - xmin) / cs) can move a particle. (The staged float
// walk skips them; in the double walk the extra registers cost more than
// the skipped candidates save.)
__device__ inline unsigned far_corners(double X, double Y, int2 c, const Grid &g, double lim2) {
    const double e = 1e-9 * g.cs;
    const double x0 = g.xmin + g.cs * c.x, y0 = g.ymin + g.cs * c.y;
    double l = X - x0 - e, r = x0 + g.cs - X - e, b = Y - y0 - e, a = y0 + g.cs - Y - e;
    l = l > 0.0 ? l * l : 0.0;
    r = r > 0.0 ? r * r : 0.0;
    b = b > 0.0 ? b * b : 0.0;
    a = a > 0.0 ? a * a : 0.0;
    return (l + b > lim2 ? 1u : 0u) | (r + b > lim2 ? 2u : 0u) | (l + a > lim2 ? 4u : 0u) | (r + a > lim2 ? 8u : 0u);
}

// The runs of slots target c walks in rows c.y - 1, c.y, c.y + 1 (index d =
// 0, 1, 2): [rs[d], re[d]), empty for a row outside the grid; the diagonal
// cells in `far` (far_corners) are left out of the runs of rows 0 and 2.
template <typename Args>
__device__ inline void row_runs(const Args &P, int ncx, int ncy, long long base, int2 c, unsigned far, int rs[3],
                                int re[3]) {
    const int lo = c.x - 1 > 0 ? c.x - 1 : 0;
    const int hi = c.x + 1 < ncx - 1 ? c.x + 1 : ncx - 1;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int cy = c.y + d - 1;
        rs[d] = 0;
        re[d] = 0;
        if (lo <= hi && ncy > cy && cy > -1) {
            const unsigned f = d == 0 ? far : (d == 2 ? far >> 2 : 0u);
            const int l = (f & 1u) && lo == c.x - 1 ? lo + 1 : lo;
            const int h = (f & 2u) && hi == c.x + 1 ? hi - 1 : hi;
            const long long row = base + (long long)ncx * cy;
            rs[d] = P.cellStart[row + l];
            re[d] = P.cellStart[row + h + 1];
        }
    }
}

// The workgroup's staging plan: row range d is [smin[d], smin[d] + len[d])
// of the slots, held from LDS record off[d] on.
struct Stage {
    int smin[3], len[3], off[3], total;
};

// Folds every thread's row runs (empty for a thread without a walk) into
// the workgroup's ranges. Ends with a barrier; every thread returns the same
// plan.
__device__ inline Stage stage_plan(const int rs[3], const int re[3], int *s_red) {
    int v[8];  // all as maxima
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const bool any = rs[d] < re[d];
        v[d] = any ? -rs[d] : -0x7fffffff;
        v[3 + d] = any ? re[d] : -0x7fffffff;
    }
    v[6] = v[7] = -0x7fffffff;
    const int top = wave_maxima<8>(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if (lane % 8 == 0 && lane < 48) s_red[(lane / 8) * 4 + w] = lane < 24 ? -top : top;
    __syncthreads();
    Stage S;
    int off = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int mn = 0x7fffffff, mx = -0x7fffffff;
        for (int k = 0; k < nw; ++k) {
            const int a = s_red[d * 4 + k], b = s_red[(3 + d) * 4 + k];
            mn = a < mn ? a : mn;
            mx = b > mx ? b : mx;
        }
        S.smin[d] = mn;
        S.len[d] = mx > mn ? mx - mn : 0;
        S.off[d] = off;
        off += S.len[d];
    }
    S.total = off;
    return S;
}

// Copies the planned ranges of A into LDS. Ends with a barrier.
template <typename Args>
__device__ inline void stage_copy(const Args &P, const Stage &S, double2 *sA) {
#pragma unroll
    for (int d = 0; d < 3; ++d)
        for (int i = threadIdx.x; i < S.len[d]; i += blockDim.x)
            sA[S.off[d] + i] = at32(P.A, (unsigned)(S.smin[d] + i));
    __syncthreads();
}

}  // namespace
}  // namespace hipsph
