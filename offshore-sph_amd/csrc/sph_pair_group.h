// sph_pair_group.h — the pair passes with G lanes per target, for states too
// small to fill the chip with one thread per target.
//
// One thread per target walks about 61 candidates and evaluates about 20
// contributors one after another: a serial chain of 20 to 30 us whatever the
// size, on a fraction of the 256 CUs (5k particles: 28 workgroups). Here a
// group of G consecutive lanes shares a target:
//   * the walk: lane l tests the candidates l, l + G, ... of each segment of
//     the same walk (the double pass's nine cells, the float pass's three row
//     runs); a ballot gives each kept candidate its place in the target's list
//     in LDS, so the list is the one the single thread would build;
//   * the terms: lane l evaluates the listed pairs l, l + G, ...;
//   * the sums: the G pairs' terms go through LDS and lane q % G adds quantity
//     q of all of them in list order, so every sum has the order, and the bits,
//     of the one-thread pass. A pair that adds nothing there adds a zero here.
// All lanes of a wavefront take part in every ballot: loops run until no
// group of the wavefront needs them. It costs about twice the instructions
// per target, so the launchers use it only below a size (group_lanes).
#pragma once
#include "sph_common.h"
#include "sph_pair_impl.h"

namespace hipsph {
namespace {

// LDS written by some lanes of a wavefront and read by others: the DS unit
// keeps a wavefront's order, the compiler has to as well.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The candidates of target cell c in the order of the one-thread pass, as
// one sequence of n: candidate i is slot x - i (DESC) or x + i, x the sum of
// the steps of the segments up to the one i falls in (selecting among values
// in an array instead made the compiler select their addresses and put the
// array in scratch memory). DESC: the nine cells, x shift outer, y shift inner
// (src/Tools/NNLinkedList.py:50-56), each from its highest slot down; else the
// three row runs, ascending. A cell the grid does not have is empty.
template <bool DESC>
struct Candidates {
    static constexpr int N = DESC ? 9 : 3;
    int first[N], step[N], n = 0;
    __device__ __forceinline__ Candidates(const int *cellStart, int2 c, int ncx, int ncy, long long base, bool walks) {
        // offsets of the cells c.x - 1 .. c.x + 2 of each row; the loads stay
        // inside the row's bins, an absent cell's are not used
        int o[3][4];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int cy = c.y + d - 1;
            const bool row_ok = walks && cy > -1 && cy < ncy;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int cx = c.x - 1 + k;
                cx = cx < 0 ? 0 : (cx > ncx ? ncx : cx);
                o[d][k] = row_ok ? cellStart[base + (long long)ncx * cy + cx] : 0;
            }
        }
        int before = 0;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            first[k] = n;
            int x;
            if constexpr (DESC) {
                const int a = k / 3, d = k % 3;  // the x and y shifts + 1
                const bool ok = c.x + a - 1 > -1 && c.x + a - 1 < ncx;
                x = o[d][a + 1] - 1 + n;
                n += ok ? o[d][a + 1] - o[d][a] : 0;
            } else {
                // a run over the row's cells inside the grid: lo .. hi
                const bool ok = (c.x - 1 > 0 ? c.x - 1 : 0) <= (c.x + 1 < ncx - 1 ? c.x + 1 : ncx - 1);
                x = o[k][0] - n;
                n += ok ? o[k][3] - o[k][0] : 0;
            }
            step[k] = x - before;
            before = x;
        }
    }
    __device__ __forceinline__ unsigned slot(int i) const {
        int x = step[0];
#pragma unroll
        for (int k = 1; k < N; ++k) x += i >= first[k] ? step[k] : 0;
        return (unsigned)(DESC ? x - i : x + i);
    }
};

// LDS of one target: its list and the G terms of every quantity being summed.
template <class P, int G>
struct GroupMem {
    static constexpr int L = 64;  // list entries; flushed when G more might not fit
    unsigned list[L];
    typename P::Term term[P::NQ][G + 1];
};

// A lane's sums: those of the quantities l, l + G, ...
template <class P, int G>
struct GroupSums {
    static constexpr int N = (P::NQ + G - 1) / G;
    typename P::Sum s[N];
    // quantity Q, in the group's first lane
    template <int Q>
    __device__ __forceinline__ double get() const {
        const double v = s[Q / G].get();
        if constexpr (Q % G == 0)
            return v;
        else
            return row_move<0x100 | Q % G>(v);  // of the lane Q % G further on
    }
};

// The walk and the sums of one target by its G lanes (lane l): P gives the
// test of a candidate and the terms of a listed pair. After it, acc
// holds the sums, and cnt the candidates P counted as
// neighbours. Called by every lane of the wavefront; walks is false for a
// group without a target. The records of the next two rounds of candidates
// are in flight while one is tested. One place each tests and flushes: with
// the loops over segments unrolled the compiler kept the flush a function,
// its captures in scratch memory, and the double pass took four times as long.
template <class P, int G>
__device__ __forceinline__ void group_sums(const P &p, const int *cellStart, int2 c, int ncx, int ncy, long long base,
                                  bool walks, int l, GroupMem<P, G> &M, GroupSums<P, G> &acc, int &cnt) {
    using Term = typename P::Term;
    const Candidates<P::kDesc> S(cellStart, c, ncx, ncy, base, walks);
    const int shift = (threadIdx.x & 63) - l;  // the group's first lane
    const unsigned below = (1u << l) - 1u, mask = (1u << G) - 1u;
    int nl = 0;
    cnt = 0;
    typename P::RecA a0{}, a1{};
    unsigned u0 = S.slot(l), u1 = S.slot(G + l);
    if (l < S.n) a0 = p.load(u0);
    if (G + l < S.n) a1 = p.load(u1);
    for (int i0 = 0;; i0 += G) {
        const bool more = __ballot(i0 < S.n) != 0;
        if (more) {
            const typename P::RecA a = a0;
            const unsigned u = u0;
            const int i = i0 + l;
            a0 = a1;
            u0 = u1;
            u1 = S.slot(i + 2 * G);
            if (i + 2 * G < S.n) a1 = p.load(u1);
            bool counted = false;
            const bool in = i < S.n && p.test(a, u, counted);
            const unsigned m = (unsigned)(__ballot(in) >> shift) & mask;
            if constexpr (P::kCount) cnt += __popc((unsigned)(__ballot(i < S.n && counted) >> shift) & mask);
            if (in) M.list[nl + __popc(m & below)] = u;
            nl += __popc(m);
        }
        if (more && __ballot(nl > GroupMem<P, G>::L - G) == 0) continue;
        // the listed pairs' terms, summed in list order
        wave_sync();
        for (int k0 = 0; __ballot(k0 < nl) != 0; k0 += G) {
            Term out[P::NQ];
#pragma unroll
            for (int q = 0; q < P::NQ; ++q) out[q] = Term(0);
            if (k0 + l < nl) p.terms(M.list[k0 + l], out);
#pragma unroll
            for (int q = 0; q < P::NQ; ++q) M.term[q][l] = out[q];
            wave_sync();
#pragma unroll
            for (int j = 0; j < GroupSums<P, G>::N; ++j) {
                const int q = j * G + l;
                if (q < P::NQ) {
                    Term v[G];
#pragma unroll
                    for (int k = 0; k < G; ++k) v[k] = M.term[q][k];
#pragma unroll
                    for (int k = 0; k < G; ++k) acc.s[j].add(v[k]);
                }
            }
            wave_sync();
        }
        nl = 0;
        if (!more) break;
    }
}

// Plain sums in list order.
struct PlainSum {
    double s = 0.0;
    __device__ void add(double v) { s += v; }
    __device__ double get() const { return s; }
};

// ---------------------------------------------------------------------------
// the general pass (any h and masses; XSPH)
// ---------------------------------------------------------------------------
// Quantities: 0 drho, 1 and 2 momentum, 3 and 4 wall force, 5 and 6 XSPH. The
// terms are contribute's, each taken by a one-term sum (0 + v: v itself).
template <typename R, int KERNEL, int MODE, bool XS>
struct GeneralGroup {
    using RecA = typename Rec<R>::A;
    using Term = R;
    using Sum = Acc<R>;
    static constexpr bool kDesc = sizeof(R) == 8, kCount = true;
    static constexpr int NQ = XS ? 7 : 5;
    const PairArgs<R> &P;
    const Target<R> &T;
    const Phys &ph;
    bool implied;
    __device__ __forceinline__ RecA load(unsigned u) const { return P.A[u]; }
    // scan_cell's candidate test
    __device__ __forceinline__ bool test(const RecA &a, unsigned u, bool &counted) const {
        constexpr double kEps = sizeof(R) == 8 ? 1e-12 : 1e-5;
        const R qmax = (R)ph.qmax, ks = (R)support_q<KERNEL>();
        const R r0sq = (R)ph.r0 * (R)ph.r0 * R(1.0 + kEps);
        const R dx = (R)(T.X - a.x), dy = (R)(T.Y - a.y);
        const R r2 = dx * dx + dy * dy;
        const R hij = R(0.5) * (T.h + (R)a.h);
        const R sh = ks * hij;
        const R sup2 = a.w >= R(0) ? sh * sh * R(1.0 + kEps)
                                   : (XS ? fmax(sh * sh * R(1.0 + kEps), r0sq) : r0sq);
        bool in = true;
        if (!implied || !(a.w >= R(0))) {
            const R qh = qmax * hij;
            const R lim = qh * qh;
            in = r2 < lim * R(1.0 - kEps);
            if (!in && !(r2 > lim * R(1.0 + kEps))) {
                const double hj = sizeof(R) == 8 ? (double)a.h : P.H[u];
                in = exact_q_test(T.X, T.Y, T.H, a.x, a.y, hj, ph.qmax);
            }
            counted = in;
        }
        const bool apart = XS ? (r2 > R(0) || (int)u != T.slot) : r2 > R(0);
        return in && apart && !(r2 > sup2) && ((MODE & kEquations) != kContinuity || a.w >= R(0));
    }
    __device__ __forceinline__ void terms(unsigned u, R *out) const {
        Sums<R> S;
        contribute<R, KERNEL, MODE, XS>(P, T, ph, u, P.A[u], S);
        out[0] = S.arho.s;
        out[1] = S.a0.s;
        out[2] = S.a1.s;
        out[3] = S.f0.s;
        out[4] = S.f1.s;
        if constexpr (XS) {
            out[5] = S.xs0.s;
            out[6] = S.xs1.s;
        }
    }
};

template <typename R, int KERNEL, int MODE, bool XS, int G>
__global__ __launch_bounds__(256) void k_pair_group(const Ctrl *ctrl, PairArgs<R> P, Phys ph) {
    using GG = GeneralGroup<R, KERNEL, MODE, XS>;
    __shared__ GroupMem<GG, G> mem[256 / G];
    const int i = threadIdx.x / G, l = threadIdx.x % G;
    const int t = xcd_remap(blockIdx.x, gridDim.x) * (256 / G) + i;
    const int t0 = t < P.n ? t : P.n - 1;
    const typename Rec<R>::A at = P.A[t0];  // the target's records together with the control block
    const typename Rec<R>::B bt = P.B[t0];
    const int2 c = P.cxy[t0];
    const double H = sizeof(R) == 8 ? (double)at.h : P.H[t0];
    if (!ctrl->active) return;
    const Grid &g = ctrl->grid;
    const int ncx = (int)g.ncx, ncy = (int)g.ncy;
    const bool walks = t < P.n && at.w >= R(0);  // walls are not targets
    Target<R> T;
    T.X = at.x;
    T.Y = at.y;
    T.H = H;
    T.h = (R)at.h;
    T.vx = (R)rec_vx(at, bt);
    T.vy = (R)rec_vy(at, bt);
    T.rho = (R)bt.rho;
    T.slf = (R)bt.prs;
    T.slot = t;
    const bool implied = !walks || cutoff_implied<KERNEL>(nullptr, ph.qmax, c, ncx, ncy, T.H);
    const GG gg{P, T, ph, implied};
    GroupSums<GG, G> acc;
    int cnt = 0;
    group_sums<GG, G>(gg, P.cellStart, c, ncx, ncy, 0, walks, l, mem[i], acc, cnt);
    const double arho = acc.template get<0>(), a0 = acc.template get<1>(), a1 = acc.template get<2>();
    const double f0 = acc.template get<3>(), f1 = acc.template get<4>();
    double xs0 = 0.0, xs1 = 0.0;
    if constexpr (XS) {
        xs0 = acc.template get<5>();
        xs1 = acc.template get<6>();
    }
    if (!walks || l != 0) return;
    if (!implied && cnt == 0) return;  // SolverTools.py:166-169: no neighbours, keep the previous values
    if constexpr ((MODE & kEquations) != kMomentum) P.drho[t] = arho;
    if constexpr ((MODE & kEquations) != kContinuity) {
        P.ax[t] = a0 + f0;
        P.ay[t] = (a1 - ph.g) + f1;  // WCSPH.py:169, then SolverTools.py:170-171
    }
    if constexpr (XS) {  // WCSPH.compute_velocity: xsph = v + correction (WCSPH.py:180-186)
        const double vxi = sizeof(R) == 8 ? (double)T.vx : P.VX[t];
        const double vyi = sizeof(R) == 8 ? (double)T.vy : P.VY[t];
        P.xsx[t] = vxi + xs0;
        P.xsy[t] = vyi + xs1;
    }
}

template <typename R, int MODE, bool XS = false>
void launch_group_mode(const Ctrl *ctrl, const PairArgs<R> &P, const Phys &ph, int lanes, hipStream_t s) {
    const int nb = xcd_blocks((long long)P.n * lanes, 256);
    with_kernel(ph.kernel, [&](auto kk) {
        with_group(lanes, [&](auto gg) {
            k_pair_group<R, decltype(kk)::value, MODE, XS, decltype(gg)::value><<<nb, 256, 0, s>>>(ctrl, P, ph);
        });
    });
}

template <typename R, bool EXACT>
hipError_t launch_pair(const Ctrl *ctrl, const PairArgs<R> &P, const Phys &ph, int threads, int mode, hipStream_t s) {
    const bool xs = P.xsx != nullptr;  // XSPH velocity requested (fused and momentum passes only)
    const bool whole = whole_exponent(ph.p1) && whole_exponent(ph.p2);
    const int lanes = P.count || !whole ? 0 : group_lanes(P.n, sizeof(R) == 8, false, ph.kernel);
    if (lanes) {
        if (mode == kContinuity)
            launch_group_mode<R, kContinuity | kIntPow>(ctrl, P, ph, lanes, s);
        else if (mode == kMomentum)
            xs ? launch_group_mode<R, kMomentum | kIntPow, true>(ctrl, P, ph, lanes, s)
               : launch_group_mode<R, kMomentum | kIntPow>(ctrl, P, ph, lanes, s);
        else
            xs ? launch_group_mode<R, kFused | kIntPow, true>(ctrl, P, ph, lanes, s)
               : launch_group_mode<R, kFused | kIntPow>(ctrl, P, ph, lanes, s);
        return hipGetLastError();
    }
    if (threads != 64 && threads != 128 && threads != 256) threads = kPairThreads;
    const int nb = xcd_blocks(P.n, threads);
    with_pow(whole, [&](auto ww) {
        constexpr int W = decltype(ww)::value;
        if (mode == kContinuity)
            launch_pair_mode<R, EXACT, kContinuity | W>(ctrl, P, ph, nb, threads, s);
        else if (mode == kMomentum)
            xs ? launch_pair_mode<R, EXACT, kMomentum | W, true>(ctrl, P, ph, nb, threads, s)
               : launch_pair_mode<R, EXACT, kMomentum | W>(ctrl, P, ph, nb, threads, s);
        else
            xs ? launch_pair_mode<R, EXACT, kFused | W, true>(ctrl, P, ph, nb, threads, s)
               : launch_pair_mode<R, EXACT, kFused | W>(ctrl, P, ph, nb, threads, s);
    });
    return hipGetLastError();
}

}  // namespace
}  // namespace hipsph
