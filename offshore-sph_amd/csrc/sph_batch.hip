// sph_batch.hip — many independent WCSPH simulations advanced together.
//
// A batch holds K instances of uneven particle counts (an ensemble of dam
// breaks with different geometry, resolution and constants). All instances
// share one concatenated, cell-ordered state and one segmented cell grid, and
// every stage of the step is ONE launch covering all instances:
//   * instance k owns particle slots [off_k, off_k + n_k) for good (its
//     particles only ever move among its own slots) and room for its most
//     cells from a fixed bin on, so each instance's offsets are scanned from
//     off_k without the others;
//   * every workgroup works on one instance (tiles of 256 slots, chunks of
//     1,024 or 4,096 for the bounds), whose control block it reads once;
//   * reductions (bounds, dt) leave partials per chunk or tile, and the
//     kernel that needs the result folds its instance's in every workgroup,
//     as the single engine's k_bounds and k_keys do (24 dam breaks, 0.72M
//     particles: the update's five kernels take 42 us; 72 with kernels of
//     their own for the folds, the bins' bases and the bin sort, LDS permutes
//     in the folds and a scan that read every count again);
//   * every instance has its own control block (BInst): clock, dt, grid,
//     halt flags and constants (alpha, c0, B, r0, D ...).
// A step needs no host round trip, like the single simulation's. The
// arithmetic per particle is the single engine's, in the same order, so an
// instance evolves exactly as it would alone.
//
// Built with -ffp-contract=off (as sph_engine.hip).
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstring>
#include <vector>

#include "sph_ctx.h"
#include "sph_common.h"

using namespace hipsph;

namespace {

// Two segmentations of the slots, each segment inside one instance: chunks
// of chunk_slots for the bounds reduction (one workgroup of kChunkThreads), tiles
// of kTile for everything else (one 256-thread workgroup per tile).
constexpr int kChunkThreads = 512;
// 1,024 slots, or 4,096 in a batch of more than 2,048 such chunks: each
// workgroup folds its instance's dt partials again, and when the border cells
// are enough few of its threads have a particle (256 dam breaks, 7.7M
// particles: 7,500 workgroups took 76 us).
inline int chunk_slots(long long n) { return n > 2048 * 1024 ? 4096 : 1024; }
constexpr int kTile = 256;
// Entries of dt partials (tiles) and bounds partials (chunks) an instance has
// at most: every workgroup of the next kernel reads all of its instance's, so
// without a limit that grows with the square of its size. An instance of more
// shares them by atomic maxima, cleared after their readers. Steps in us without
// and with a limit (and the scan's workgroups by size): one FP32C instance of 4M
// particles 764, 556; of 1M 190, 148; 2 of 2M 639, 554; 24 of 30k 127, 127.
constexpr int kDtEntries = 512, kBoundsEntries = 128;
static_assert(kTile == 256, "the fused batch pair pass runs one 256-thread workgroup per tile");

struct BState {  // the concatenated cell-ordered state (as State)
    State s;
};

// ---------------------------------------------------------------------------
// per-instance dt (src/Solver.py:210-230, src/Equations/TimeStep.py:40-90)
// ---------------------------------------------------------------------------
// segment c (a tile) covers [cs[c], cs[c + 1]) inside one instance
__global__ void kb_dt_partial(const int *cs, const int *segInst, const int *entry, const BInst *inst, State s,
                              unsigned long long *part, Ctrl *view) {
    __shared__ double lds[kDtQ * 16];
    const int c = blockIdx.x, e = entry[c];
    if (c == 0 && threadIdx.x == 0) view->pec_parts = 0;
    const BInst &I = inst[segInst[c]];
    DtVars v;
    for (int t = cs[c] + threadIdx.x; t < cs[c + 1]; t += blockDim.x)
        if (s.label[t] == kFluid) v.add(I.uh_on ? I.uh : s.h[t], s.ax[t], s.ay[t]);
    v.publish(part, e, lds);
}

// One workgroup's fold of its instance's dt partials; the result is valid in
// thread 0. lds holds kDtQ * 16 doubles.
__device__ inline void bdt_fold(const unsigned long long *part, const BInst &I, double (&v)[kDtQ], double *lds) {
    const int kind[kDtQ] = {0, 1, 2, 2};
    v[0] = INFINITY;
    v[1] = -INFINITY;
    v[2] = v[3] = 0.0;
    for (int j = threadIdx.x; j < I.dtn; j += blockDim.x) {
        const ulonglong2 *p = reinterpret_cast<const ulonglong2 *>(part + (size_t)kDtQ * (I.dt0 + j));
        const ulonglong2 a = p[0], b = p[1];
        v[0] = -max_of(-v[0], order_value(a.x));
        v[1] = max_of(v[1], order_value(a.y));
        v[2] = max_of(v[2], order_value(b.x));
        v[3] = max_of(v[3], order_value(b.y));
    }
    block_fold<kDtQ>(v, kind, lds);
}

// The decision takes effect (dt_commit, for an instance).
__device__ inline void bdt_commit(BInst &I, const DtNext &x) {
    I.disp = x.disp;
    I.vbound = x.vbound;
    I.abound = x.abound;
    if (x.flags) atomicOr(&I.flags, x.flags);
    I.active = x.active;
    if (!x.active) return;
    I.dt = x.dt;
    I.dt_c = x.dt_c;
    I.dt_f = x.dt_f;
    I.t = x.t;
    I.step = x.step;
}

// ---------------------------------------------------------------------------
// neighbour update over the segmented grid (src/Tools/NNLinkedList.py)
// ---------------------------------------------------------------------------
struct BPos {  // what it is formed from, loaded before dt is known
    double x, y, vx, vy;
    int8_t lab;
};
__device__ inline BPos bpos_load(const State &a, int i, bool pred) {
    return BPos{a.x[i], a.y[i], pred ? a.vx[i] : 0.0, pred ? a.vy[i] : 0.0, a.label[i]};
}
__device__ inline void bupd_pos(const BPos &p, bool pred, double dt, double &x, double &y) {
    const bool f = pred && p.lab == kFluid;
    x = f ? pec_half_pos(p.x, p.vx, dt) : p.x;
    y = f ? pec_half_pos(p.y, p.vy, dt) : p.y;
}

// Per chunk (of one instance's slots): the fold of the instance's dt
// partials and its decision (every workgroup needs dt; the first chunk's
// leaves it in I.nx for kb_keys), then the chunk's bounds into an entry of its
// instance's partials (kBoundsVQ order keys, as maxima), or one that it shares
// (~entry). With PEC's predictor the full scan also finds the
// largest |vx|, |vy| (kb_keys keeps it as the instance's vbound). With
// cellStart (the fused PEC step) and an instance whose carried bound allows
// it (as the single engine's k_bounds), the instance's chunks share the walk
// of its border cells instead.
__global__ __launch_bounds__(kChunkThreads) void kb_bounds(const int *cs, const int *chunkInst, const int *entry,
                                                           const int *chunk0, BInst *inst, State a, int pec,
                                                           const unsigned long long *part_d, unsigned long long *part,
                                                           const int *cellStart, Ctrl *view) {
    __shared__ double lds[kBoundsVQ * 16];
    __shared__ double s_dt, s_disp;
    __shared__ int s_active;
    const int c = blockIdx.x;
    const int k = chunkInst[c], e = entry[c];
    if (c == 0 && threadIdx.x == 0) view->epoch += 1;
    BInst &I = inst[k];
    const bool pred = pec != 0;
    // the first particles of either scan, in flight under the dt fold
    const Grid g = I.grid;
    const bool may = cellStart && pred && I.uh_on && g.ncx >= 3 && g.ncy >= 3;
    const int tid = (c - chunk0[k]) * (int)blockDim.x + (int)threadIdx.x;
    const int nthreads = (chunk0[k + 1] - chunk0[k]) * (int)blockDim.x;
    constexpr int U = 2;
    int slot[U];
    BPos p[U];
    if (may) {
        const BorderWalk W(cellStart, I.cellBase, g, tid, nthreads);
        slot[0] = W.first_row();
        slot[1] = W.first_run();
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = cs[c] + (int)threadIdx.x + u * kChunkThreads;
            slot[u] = i < cs[c + 1] ? i : -1;
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (slot[u] >= 0) p[u] = bpos_load(a, slot[u], pred);
    {
        const DtIn in(I, view->pec_parts);
        double v[kDtQ];
        bdt_fold(part_d, I, v, lds);
        if (threadIdx.x == 0) {
            const DtNext x = dt_decide(in, v, I.gamma_c, I.gamma_f);
            s_dt = x.dt;
            s_disp = x.disp;
            s_active = x.active;
            if (c == chunk0[k]) I.nx = x;
        }
        __syncthreads();
    }
    if (!s_active) return;
    const double dt = s_dt;
    double xmn = INFINITY, xmx = -INFINITY, ymn = INFINITY, ymx = -INFINITY, hmn = INFINITY, hmx = -INFINITY;
    double bad = 0.0, vmx = -INFINITY;
    auto take = [&](int i, const BPos &q) {
        double xi, yi;
        bupd_pos(q, pred, dt, xi, yi);
        const double hi = I.uh_on ? I.uh : a.h[i];
        if (!(xi - xi == 0.0) || !(yi - yi == 0.0)) bad += 1.0;
        xmn = xi < xmn ? xi : xmn;
        xmx = xi > xmx ? xi : xmx;
        ymn = yi < ymn ? yi : ymn;
        ymx = yi > ymx ? yi : ymx;
        hmn = hi < hmn ? hi : hmn;
        hmx = hi > hmx ? hi : hmx;
    };
    if (may && border_margin_ok(g, s_disp)) {
        if (c == chunk0[k] && threadIdx.x == 0) I.border_updates += 1;
        hmn = hmx = I.uh;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (slot[u] >= 0) take(slot[u], p[u]);
        BorderWalk(cellStart, I.cellBase, g, tid, nthreads).rest([&](int i) { take(i, bpos_load(a, i, pred)); });
    } else {
        auto speed = [&](const BPos &q) {
            if (!pred) return;
            const double ux = fabs(q.vx), uy = fabs(q.vy);
            const double w = (isfinite(ux) && isfinite(uy)) ? (ux > uy ? ux : uy) : INFINITY;
            vmx = w > vmx ? w : vmx;
        };
        const int end = cs[c + 1];
        int i0 = cs[c] + (int)threadIdx.x;
        if (!may) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (slot[u] >= 0) {
                    take(slot[u], p[u]);
                    speed(p[u]);
                }
            i0 += U * kChunkThreads;
        }
        for (; i0 < end; i0 += U * kChunkThreads) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + u * kChunkThreads < end) p[u] = bpos_load(a, i0 + u * kChunkThreads, pred);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + u * kChunkThreads < end) {
                    take(i0 + u * kChunkThreads, p[u]);
                    speed(p[u]);
                }
        }
    }
    const int kind[kBoundsVQ] = {0, 1, 0, 1, 0, 1, 2, 1};
    const double v[kBoundsVQ] = {xmn, xmx, ymn, ymx, hmn, hmx, bad, vmx};
    __syncthreads();  // lds held the dt fold
    publish_maxima<kBoundsVQ>(v, kind, lds, part + (size_t)kBoundsVQ * (e < 0 ? ~e : e), e < 0);
}

// _bin :129-141 with the instance's grid; rank by runs as k_keys does. One
// tile per workgroup, which derives its instance's grid from the bounds'
// partials itself (32 lanes per quantity) and clears a dt entry that is shared; the instance's first tile moves the grid and the dt decision into
// its control block, whose fields no workgroup reads here (they take I.nx and
// their own grid). An instance that is not active is left where it is.
__global__ __launch_bounds__(kTile) void kb_keys(const int *ts, const int *tileInst, const int *entry,
                                                 const int *tile0, BInst *inst, State a, int pec, const unsigned long long *part,
                                                 unsigned long long *part_d, int *counts, int *bin, int *rank, int *binflag, int *tileSums, Ctrl *view) {
    __shared__ double s_v[kBoundsVQ];
    __shared__ Grid s_g;
    __shared__ unsigned s_halt;
    const int c = blockIdx.x;
    if (c == 0 && threadIdx.x == 0) view->pec_parts = 0;  // kb_bounds has read it
    const int k = tileInst[c], e = entry[c];
    BInst &I = inst[k];
    const bool first = c == tile0[k];
    // loaded together with the instance's control block
    const int t = ts[c] + (int)threadIdx.x;
    const bool in = t < ts[c + 1];
    const int lane = threadIdx.x & 63;
    const int t0 = in ? t : ts[c];
    const BPos p = bpos_load(a, t0, pec != 0);
    const int id = in ? a.id[t0] : 0x7fffffff;
    if (e < 0 && ~e == I.dt0 + c - tile0[k] && threadIdx.x < kDtQ)  // its entry's first tile
        part_d[(size_t)kDtQ * ~e + threadIdx.x] = 0;                // kb_bounds has folded it
    if (!I.nx.active) {
        if (first && threadIdx.x == 0) bdt_commit(I, I.nx);
        return;
    }
    const int epoch = view->epoch;
    double x, y;
    bupd_pos(p, pec != 0, I.nx.dt, x, y);
    {  // 32 lanes per quantity fold the instance's bounds, all as maxima
        const int q = threadIdx.x >> 5;
        unsigned long long u = 0;
        for (int j = threadIdx.x & 31; j < I.bn; j += 32) u = max_of(u, part[(size_t)kBoundsVQ * (I.b0 + j) + q]);
        unsigned long long u2 = u;
        row_swap<16>(u, u2);
        u = group_max<4>(max_of(u, u2));
        if ((threadIdx.x & 31) == 0) s_v[q] = q == 0 || q == 2 || q == 4 ? -order_value(u) : order_value(u);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        Grid g;
        const unsigned halt = derive_grid(s_v, I.scale, I.cap, g);
        s_halt = halt;
        s_g = g;
        if (first) {
            bdt_commit(I, I.nx);
            if (s_v[7] >= 0.0) I.vbound = s_v[7];  // a full scan's velocity bound
            if (halt) {
                atomicOr(&I.flags, halt);
                I.active = 0;
            } else {
                I.grid = g;
            }
        }
    }
    __syncthreads();
    if (s_halt) return;
    const Grid &g = s_g;
    int b = -1;
    if (in) {
        const int2 cc = cell_of(x, y, g);
        const long long key = (long long)cc.x + g.ncx * (long long)cc.y;
        if (key >= 0 && key < g.ncells) {
            b = (int)(I.cellBase + key);
        } else {  // as k_keys: the overflow bin, and the instance's flag
            b = (int)(I.cellBase + g.ncells);
            atomicOr(&I.flags, (unsigned)SPH_FLAG_OOB_KEY);
        }
    }
    int leader, next;
    bin_run(b, id, leader, next);
    int base = 0;
    if (lane == leader && b >= 0) {
        base = atomicAdd(&counts[b], next - leader);
        if (base != 0) binflag[b] = epoch;
    }
    tile_add(tileSums, b < 0 ? -1 : I.tileBase + (b - (int)I.cellBase) / kScanTile);
    base = __shfl(base, leader, 64);
    if (in) {
        bin[t] = b;
        rank[t] = base + (lane - leader);
    }
}

// Each instance's offsets, scanned from its first slot by scan_groups
// workgroups, a tile of bins each at a time: those of row blockIdx.y, or, with
// the tables, wg0[k] ... wg0[k + 1] - 1 of the x axis (the others hold 65,535
// workgroups, a batch up to 2^20 instances), whose instances wgInst gives.
// As many as keep the chip busy with few instances, or one for every 2,048
// slots (about 800 bins of a dam break) of a large one: with 64 whatever
// its size the scan of one instance of 4M particles took 111 us, now 17.
constexpr int kScanAlike = 4096;  // most workgroups in rows of as many for each instance
inline int scan_groups(int K, long long n, long long tiles) {
    const long long few = K < 2048 ? (K > 32 ? 2048 / K : 64) : 1;
    return (int)std::min(tiles, std::max(few, n / 2048));
}
__global__ __launch_bounds__(kBlock) void kb_scan(const BInst *inst, int *counts, const int *tileSums, int *cellStart,
                                                  const int *wgInst, const int *wg0) {
    __shared__ int lds[16];
    int k = (int)blockIdx.y, first = (int)blockIdx.x, w = (int)gridDim.x;
    if (wgInst) {
        k = wgInst[first];
        w = wg0[k + 1] - wg0[k];
        first -= wg0[k];
    }
    const BInst &I = inst[k];
    if (!I.active) return;
    const long long nbins = I.grid.ncells + 1;
    for (long long tile = first; tile * kScanTile < nbins; tile += w)
        scan_tile(counts + I.cellBase, tileSums + (size_t)I.tileBase * kTileStride, cellStart + I.cellBase, nbins,
                  tile, I.off, lds);
}

// Each particle's place (k_place); an instance that is not active keeps its
// order. Also zeroes the instance's tile sums for the next update, and its
// bounds entries if it shares them, active or not.
__global__ __launch_bounds__(kTile) void kb_place(const int *ts, const int *tileInst, const int *tile0,
                                                  const BInst *inst, const int *cellStart, const int *bin,
                                                  const int *rank, int *perm0, int *tileSums,
                                                  unsigned long long *part_b) {
    const int c = blockIdx.x, k = tileInst[c];
    const BInst &I = inst[k];
    const int t = ts[c] + (int)threadIdx.x;
    const bool in = t < ts[c + 1];
    const int active = I.active, shares = I.shares, first = tile0[k];  // one trip to memory
    if (shares && c == first)
        for (int j = threadIdx.x; j < kBoundsVQ * I.bn; j += kTile) part_b[(size_t)kBoundsVQ * I.b0 + j] = 0;
    if (!active) {
        if (in) perm0[t] = t;
        return;
    }
    const int j = c - first, nt = tile0[k + 1] - first;
    for (long long q = j * kTile + (int)threadIdx.x; q * kScanTile <= I.grid.ncells; q += (long long)nt * kTile)
        tileSums[(I.tileBase + q) * kTileStride] = 0;
    if (in) perm0[cellStart[bin[t]] + rank[t]] = t;
}

// Permute the state into the new order with the PEC predictor of active
// instances fused in, and write the pair records (as k_reorder). With PEC the
// reorder is lean as k_reorder's for the fluid of active instances: no
// x0 ... rho0 (kb_correct gathers them from the source buffer), no half-step
// x, y, vx, vy, rho (kb_correct forms the half-step velocity again and
// overwrites the rest), no rates of a particle inside its instance's grid
// (written by the pair pass).
__global__ __launch_bounds__(kTile) void kb_reorder(const int *ts, const int *tileInst, BInst *inst, State a, State b,
                                                    const int *perm0, int *perm, const int *cellStart,
                                                    const int *binflag, int2 *cxy_s, int fmt, void *recA, void *recB,
                                                    int pec, const Ctrl *view) {
    const int c = blockIdx.x, k = tileInst[c];
    int t = ts[c] + (int)threadIdx.x;
    if (t >= ts[c + 1]) return;
    const BInst &I = inst[k];
    const int s = perm0[t];
    const int id = a.id[s];
    const bool hs = I.uh_on;  // m and h stay in place (and m is not read: the uniform records have none)
    double x = a.x[s], y = a.y[s], vx = a.vx[s], vy = a.vy[s], rho = a.rho[s];
    const double m = hs ? 0.0 : a.m[s], h = hs ? I.uh : a.h[s];
    const double ax = a.ax[s], ay = a.ay[s], drho = a.drho[s];
    const int8_t lab = a.label[s];
    const bool skip = I.active && pec && lab == kFluid;
    if (skip) {
        const double dt = I.dt;
        x = pec_half_pos(x, vx, dt);
        y = pec_half_pos(y, vy, dt);
        vx = pec_half_vel(vx, ax, dt, I.damping);
        vy = pec_half_vel(vy, ay, dt, I.damping);
        rho = pec_half_rho(rho, drho, dt, I.strict);
    }
    // x0 ... rho0 are not kept: nothing in a batch step reads them
    // the raw cell the keys used (0, 0 in an inactive instance)
    const Grid &g = I.grid;
    int2 cc = make_int2(0, 0);
    if (I.active) {
        cc = cell_of(x, y, g);
        const long long key = (long long)cc.x + g.ncx * (long long)cc.y;  // kb_keys' bin
        t = bin_place(t, id, I.cellBase + (key >= 0 && key < g.ncells ? key : g.ncells), cellStart, binflag, view->epoch,
                      perm0, a.id);
    }
    perm[t] = s;
    if (!skip) {
        b.x[t] = x;
        b.y[t] = y;
        b.vx[t] = vx;
        b.vy[t] = vy;
        b.rho[t] = rho;
    }
    if (!hs) {
        b.m[t] = m;
        b.h[t] = h;
    }
    b.label[t] = lab;
    b.id[t] = id;
    if (!skip || !(cc.x >= 0 && cc.x < g.ncx && cc.y >= 0 && cc.y < g.ncy && h > 0.0 && I.qmax >= 0.0)) {
        b.ax[t] = ax;
        b.ay[t] = ay;
        b.drho[t] = drho;
    }
    cxy_s[t] = cc;
    const double pr = write_pair_records(t, x, y, vx, vy, rho, m, h, lab, inst_phys(I), fmt, recA, recB);
    if (I.active && lab == kFluid && !isfinite(pr)) atomicOr(&inst[k].flags, (unsigned)SPH_FLAG_ZERO_DENSITY);
}

// Per instance (one workgroup each): min and max h over its particles and
// min and max m over its fluid, in out[4k .. 4k+3].
__global__ void kb_hm_range(const BInst *inst, State st, double *out) {
    __shared__ double lds[4 * 16];
    const int k = blockIdx.x, s0 = inst[k].off, s1 = s0 + inst[k].n;
    double v[4] = {INFINITY, -INFINITY, INFINITY, -INFINITY};
    for (int i = s0 + threadIdx.x; i < s1; i += blockDim.x) {
        const double h = st.h[i];
        v[0] = h < v[0] ? h : v[0];
        v[1] = h > v[1] ? h : v[1];
        if (st.label[i] == kFluid) {
            const double m = st.m[i];
            v[2] = m < v[2] ? m : v[2];
            v[3] = m > v[3] ? m : v[3];
        }
    }
    const int kind[4] = {0, 1, 0, 1};
    block_fold<4>(v, kind, lds);
    if (threadIdx.x == 0)
        for (int q = 0; q < 4; ++q) out[4 * k + q] = v[q];
}

// PEC.correct / Euler (fluid of active instances) + the next dt partials.
// PEC's start-of-step values come from the buffer before the reorder, at the
// particle's previous slot perm[j] (the lean reorder did not copy them).
__global__ void kb_correct(const int *cs, const int *chunkInst, const int *entry, const BInst *inst, State s, State o,
                           const int *perm, int euler, unsigned long long *part, Ctrl *view) {
    __shared__ double lds[kDtQ * 16];
    const int c = blockIdx.x, e = entry[c];
    if (c == 0 && threadIdx.x == 0) view->pec_parts = 0;
    const BInst &I = inst[chunkInst[c]];
    const double dt = I.dt, damping = I.damping;
    DtVars v;
    for (int j = cs[c] + threadIdx.x; j < cs[c + 1]; j += blockDim.x) {
        if (s.label[j] != kFluid) continue;
        const double ax = s.ax[j], ay = s.ay[j];
        v.add(I.uh_on ? I.uh : s.h[j], ax, ay);
        if (!I.active) continue;
        if (!euler) {
            const int q = perm[j];
            const double x0 = o.x[q], y0 = o.y[q], vx0 = o.vx[q], vy0 = o.vy[q], rho0 = o.rho[q];
            const double vxh = pec_half_vel(vx0, o.ax[q], dt, damping);  // as kb_reorder formed it
            const double vyh = pec_half_vel(vy0, o.ay[q], dt, damping);
            double mid_x = x0 + 0.5 * dt * vxh;
            double mid_y = y0 + 0.5 * dt * vyh;
            double mid_vx = (vx0 + 0.5 * dt * ax) / (1 + 0.5 * damping);
            double mid_vy = (vy0 + 0.5 * dt * ay) / (1 + 0.5 * damping);
            s.x[j] = 2 * mid_x - x0;
            s.y[j] = 2 * mid_y - y0;
            s.vx[j] = 2 * mid_vx - vx0;
            s.vy[j] = 2 * mid_vy - vy0;
            double mid_rho = rho0 + 0.5 * dt * s.drho[j];
            double r = 2 * mid_rho - rho0;
            if (I.strict && r < 0.0) r = 0.0;
            s.rho[j] = r;
        } else {
            double vx = s.vx[j], vy = s.vy[j];
            s.x[j] = s.x[j] + dt * vx + 0.5 * dt * dt * ax;
            s.y[j] = s.y[j] + dt * vy + 0.5 * dt * dt * ay;
            s.vx[j] = vx + dt * ax;
            s.vy[j] = vy + dt * ay;
            s.rho[j] = s.rho[j] + dt * s.drho[j];
        }
    }
    v.publish(part, e, lds);
}

__global__ void kb_upload(State d, sph_state_t in, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    d.x[i] = d.x0[i] = in.x[i];
    d.y[i] = d.y0[i] = in.y[i];
    d.vx[i] = d.vx0[i] = in.vx[i];
    d.vy[i] = d.vy0[i] = in.vy[i];
    d.rho[i] = d.rho0[i] = in.rho[i];
    d.ax[i] = in.ax ? in.ax[i] : 0.0;
    d.ay[i] = in.ay ? in.ay[i] : 0.0;
    d.drho[i] = in.drho ? in.drho[i] : 0.0;
    d.m[i] = in.m[i];
    d.h[i] = in.h[i];
    d.label[i] = in.label[i];
    d.id[i] = i;
}

// m0, h0: the upload's buffer, where an instance with uh_on keeps m and h at
// slot = id.
__global__ void kb_download(State s, sph_state_t out, const BInst *inst, const int *instOf, int n,
                            const double *m0, const double *h0) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int i = s.id[t];
    const BInst &I = inst[instOf[t]];
    if (out.x) out.x[i] = s.x[t];
    if (out.y) out.y[i] = s.y[t];
    if (out.vx) out.vx[i] = s.vx[t];
    if (out.vy) out.vy[i] = s.vy[t];
    if (out.rho) out.rho[i] = s.rho[t];
    if (out.ax) out.ax[i] = s.ax[t];
    if (out.ay) out.ay[i] = s.ay[t];
    if (out.drho) out.drho[i] = s.drho[t];
    if (out.m) out.m[i] = I.uh_on ? m0[i] : s.m[t];
    if (out.h) out.h[i] = I.uh_on ? h0[i] : s.h[t];
    if (out.label) out.label[i] = s.label[t];
    if (out.p) out.p[i] = tait_p(s.rho[t], s.label[t], I.gamma, I.B, I.rho0, I.Pb);
}

// The bins an instance of at most cap cells needs, with the overflow bin and
// the end of its slots, in whole 16-byte rows of counts; and its scan tiles.
inline long long bin_room(long long cap) { return (cap + 2 + 3) / 4 * 4; }
inline long long tile_room(long long cap) { return (cap + 1 + kScanTile - 1) / kScanTile; }

inline int nblk_b(long long n, int bs = kBlock) {
    long long b = (n + bs - 1) / bs;
    return (int)(b < 1 ? 1 : b);
}

}  // namespace

// ---------------------------------------------------------------------------
// the batch object
// ---------------------------------------------------------------------------
struct sph_batch {
    int K = 0, n = 0, NC = 0;
    int kernel = 0, precision = 0, integrator = 0;
    std::vector<sph_params_t> P;
    State buf[2];
    void *arena[2] = {nullptr, nullptr};
    int cur = 0;
    BInst *inst = nullptr;
    Ctrl *view = nullptr;
    int *instOf = nullptr, *cs = nullptr, *chunkInst = nullptr, *chunk0 = nullptr;
    int NT = 0;  // tiles: starts ts (NT + 1), instance of each, first tile of each instance (K + 1)
    int *ts = nullptr, *tileInst = nullptr, *tile0 = nullptr;
    dim3 scan;  // the scan's workgroups: a row for each instance, or by the tables
    int *wgInst = nullptr, *wg0 = nullptr;
    int *bin = nullptr, *rank = nullptr, *perm0 = nullptr, *perm = nullptr;
    int2 *cxy_s = nullptr;
    int *counts = nullptr, *cellStart = nullptr, *binflag = nullptr, *tileSums = nullptr;
    unsigned long long *part_b = nullptr, *part_d = nullptr;  // bounds and dt partials
    int *bEntry = nullptr, *dtEntry = nullptr;  // of each chunk and tile (~: shared)
    size_t part_d_bytes = 0;
    void *recA = nullptr, *recB = nullptr;
    long long capBins = 0;
    bool dt_fresh = false;
    bool loaded = false;  // a state was uploaded: every id indexes its instance
    int pair_threads = 256;
    int list_len = 0;  // 0: the single-simulation pass's length
    int persistent = 0;    // the pair pass as a persistent work-queue kernel
    int border_bounds = 1;  // the fused PEC step's bounds from the border cells when the carried bound allows
    // every instance has one h for all its particles and one fluid mass and
    // allows the uniform pass (found at upload): records kRecUniform(64) and
    // the uniform pair pass, each instance's constants in uniK
    bool uni = false;
    bool whole = true;  // every instance's wall force exponents are whole numbers
    void *uniK = nullptr;
    double *hm = nullptr;  // per-instance h and fluid-mass ranges (4 per instance)
    int *queue = nullptr;  // its counters (9 x 32 ints), zero between launches
    int cus = 0;           // compute units of the batch's device
    int queue_grid = 0;    // its grid (0: to be sized before the next launch)
    bool timing = false;
    std::vector<hipEvent_t> ev;
    size_t n_ev = 0;
    std::vector<int> offs;
};

namespace {

void free_batch(sph_batch *b) {
    if (!b) return;
    for (int k = 0; k < 2; ++k) {
        if (b->arena[k]) hipFree(b->arena[k]);
    }
    void *ptrs[] = {b->inst, b->view, b->instOf, b->cs, b->chunkInst, b->chunk0, b->ts, b->tileInst, b->tile0,
                    b->wgInst, b->wg0, b->bEntry, b->dtEntry, b->bin, b->rank, b->perm,
                    b->perm0, b->cxy_s, b->counts, b->cellStart, b->binflag, b->tileSums,
                    b->part_b, b->part_d, b->recA, b->recB, b->queue, b->uniK, b->hm};
    for (void *p : ptrs)
        if (p) hipFree(p);
    for (auto e : b->ev) hipEventDestroy(e);
    delete b;
}

// The persistent pair pass's grid: one resident occupancy of the device
// (hipOccupancy for the chosen kernel, list and workgroup size). Host only;
// sized before a step is launched.
void size_queue(sph_batch *b) {
    if (!b->persistent || b->queue_grid > 0) return;
    const int per = b->uni ? (b->precision == SPH_PREC_FP32C ? pair_batch_uniform_occupancy_fp32(b->kernel)
                                                             : pair_batch_uniform_occupancy_fp64(b->kernel))
                    : b->precision == SPH_PREC_FP32C
                        ? pair_batch_queue_occupancy_fp32c(b->kernel, b->list_len, b->pair_threads)
                        : pair_batch_queue_occupancy_fp64(b->kernel, b->list_len, b->pair_threads);
    b->queue_grid = (b->cus > 0 ? b->cus : kXcds) * per;
}

int b_nn(sph_batch *b, hipStream_t s) {
    const int pec = b->integrator == SPH_INTEGRATOR_PEC;
    State a = b->buf[b->cur], c = b->buf[1 - b->cur];
    if (!b->dt_fresh)
        kb_dt_partial<<<b->NT, kBlock, 0, s>>>(b->ts, b->tileInst, b->dtEntry, b->inst, a, b->part_d, b->view);
    // the border-cell bounds only in the fused PEC step's update
    const bool fused = b->uni && !b->persistent && pec;
    kb_bounds<<<b->NC, kChunkThreads, 0, s>>>(b->cs, b->chunkInst, b->bEntry, b->chunk0, b->inst, a, pec, b->part_d,
                                              b->part_b, fused && b->border_bounds ? b->cellStart : nullptr, b->view);
    kb_keys<<<b->NT, kTile, 0, s>>>(b->ts, b->tileInst, b->dtEntry, b->tile0, b->inst, a, pec, b->part_b, b->part_d,
                                    b->counts, b->bin, b->rank, b->binflag, b->tileSums, b->view);
    kb_scan<<<b->scan, kBlock, 0, s>>>(b->inst, b->counts, b->tileSums, b->cellStart, b->wgInst, b->wg0);
    kb_place<<<b->NT, kTile, 0, s>>>(b->ts, b->tileInst, b->tile0, b->inst, b->cellStart, b->bin, b->rank, b->perm0,
                                     b->tileSums, b->part_b);
    const int fmt = b->precision == SPH_PREC_FP32C ? (b->uni ? kRecUniform : kRecFp32)
                                                   : (b->uni ? kRecUniform64 : kRecFp64);
    kb_reorder<<<b->NT, kTile, 0, s>>>(b->ts, b->tileInst, b->inst, a, c, b->perm0, b->perm, b->cellStart, b->binflag,
                                       b->cxy_s, fmt, b->recA, b->recB, pec, b->view);
    HIPCHK(hipGetLastError());
    b->cur = 1 - b->cur;
    return 0;
}

// An event around the pair pass (timing on).
int b_mark(sph_batch *b, hipStream_t s) {
    if (b->n_ev >= b->ev.size()) {
        hipEvent_t e;
        HIPCHK(hipEventCreate(&e));
        b->ev.push_back(e);
    }
    HIPCHK(hipEventRecord(b->ev[b->n_ev++], s));
    return 0;
}

int b_pair(sph_batch *b, hipStream_t s) {
    State st = b->buf[b->cur];
    PairIn in{b->recA, b->recB, st.h, b->cxy_s, b->cellStart};
    PairOut out{st.ax, st.ay, st.drho, nullptr, 0};
    int *q = b->persistent ? b->queue : nullptr;
    hipError_t e;
    if (b->uni)  // the uniform pass: its own workgroup size (256) and list length
        e = b->precision == SPH_PREC_FP32C
                ? launch_pair_batch_fp32u(b->inst, b->instOf, in, out, b->uniK, b->kernel, b->n, q, b->queue_grid, s)
                : launch_pair_batch_fp64u(b->inst, b->instOf, in, out, b->uniK, b->kernel, b->n, q, b->queue_grid, s);
    else
        e = b->precision == SPH_PREC_FP32C
                ? launch_pair_batch_fp32c(b->inst, b->instOf, in, out, b->kernel, b->n, b->pair_threads, b->list_len,
                                          q, b->queue_grid, s)
                : launch_pair_batch_fp64(b->inst, b->instOf, in, out, b->kernel, b->n, b->pair_threads, b->list_len,
                                         q, b->queue_grid, s);
    if (e != hipSuccess) return fail(SPH_EHIP, "batch pair launch: %s", hipGetErrorString(e));
    return 0;
}

// The uniform pair pass with PEC's corrector and the tiles' dt partials
// fused in: one workgroup per tile (one instance each).
int b_pair_pec(sph_batch *b, hipStream_t s) {
    State st = b->buf[b->cur];
    PairIn in{b->recA, b->recB, st.h, b->cxy_s, b->cellStart};
    PairOut out{st.ax, st.ay, st.drho, nullptr, 0};
    const PecArgs pec{st, b->buf[1 - b->cur], b->perm, b->part_d, nullptr, HmConst{}, 0, b->dtEntry,
                      &b->view->pec_parts};
    hipError_t e = b->precision == SPH_PREC_FP32C
                       ? launch_pair_batch_fp32u_pec(b->inst, b->ts, b->tileInst, b->NT, in, out, b->uniK, b->kernel,
                                                     b->n, b->whole, pec, s)
                       : launch_pair_batch_fp64u_pec(b->inst, b->ts, b->tileInst, b->NT, in, out, b->uniK, b->kernel,
                                                     b->n, b->whole, pec, s);
    if (e != hipSuccess) return fail(SPH_EHIP, "batch pair launch: %s", hipGetErrorString(e));
    return 0;
}

int b_step(sph_batch *b, hipStream_t s) {
    int rc;
    if ((rc = b_nn(b, s))) return rc;
    // timed: the pair pass and the corrector, fused or apart
    if (b->timing && (rc = b_mark(b, s))) return rc;
    if (b->uni && !b->persistent && b->integrator == SPH_INTEGRATOR_PEC) {
        if ((rc = b_pair_pec(b, s))) return rc;
    } else {
        if ((rc = b_pair(b, s))) return rc;
        kb_correct<<<b->NT, kBlock, 0, s>>>(b->ts, b->tileInst, b->dtEntry, b->inst, b->buf[b->cur], b->buf[1 - b->cur],
                                            b->perm, b->integrator == SPH_INTEGRATOR_EULER, b->part_d, b->view);
        HIPCHK(hipGetLastError());
    }
    if (b->timing && (rc = b_mark(b, s))) return rc;
    b->dt_fresh = true;
    return 0;
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

int sph_batch_create(const sph_params_t *params, int32_t ninst, sph_batch_t **out) {
    if (!params || !out) return fail(SPH_EINVAL, "NULL argument");
    *out = nullptr;
    if (ninst < 1 || ninst > (1 << 20)) return fail(SPH_EINVAL, "ninst=%d out of range", ninst);
    long long ntot = 0, capTot = 0, tiles = 0;
    for (int k = 0; k < ninst; ++k) {
        const sph_params_t &P = params[k];
        if (P.n <= 0) return fail(SPH_EINVAL, "instance %d: n=%lld", k, (long long)P.n);
        if (P.kernel != params[0].kernel || P.precision != params[0].precision ||
            P.integrator != params[0].integrator)
            return fail(SPH_EINVAL, "instance %d: kernel, precision and integrator must agree across the batch", k);
        if (P.kernel < 0 || P.kernel > 2) return fail(SPH_EINVAL, "unknown kernel id %d", P.kernel);
        if (P.precision != SPH_PREC_FP64 && P.precision != SPH_PREC_FP32C)
            return fail(SPH_EINVAL, "unknown precision %d", P.precision);
        if (P.integrator != SPH_INTEGRATOR_PEC && P.integrator != SPH_INTEGRATOR_EULER)
            return fail(SPH_EINVAL, "unknown integrator %d", P.integrator);
        if (P.use_xsph || P.use_summation_density || P.dynamic_h || P.coupled_integrator)
            return fail(SPH_EUNSUPPORTED, "a batch runs the plain WCSPH step (no XSPH, summation density, dynamic h or coupled integrator)");
        if (!(P.scale > 0) || !(P.qmax > 0) || !(P.rho0 > 0))
            return fail(SPH_EINVAL, "instance %d: scale, qmax and rho0 must be positive", k);
        ntot += P.n;
        const long long cap = P.cell_capacity > 0 ? P.cell_capacity : P.n * 8 + 4096;
        capTot += bin_room(cap);
        tiles += tile_room(cap);
    }
    if (ntot > (1LL << 30)) return fail(SPH_EINVAL, "%lld particles in the batch (max 2^30)", ntot);
    if (capTot > (1LL << 31) - 16) return fail(SPH_EINVAL, "too many cells in the batch");
    sph_batch *b = new (std::nothrow) sph_batch;
    if (!b) return fail(SPH_ENOMEM, "host allocation failed");
    b->K = ninst;
    b->n = (int)ntot;
    b->kernel = params[0].kernel;
    b->precision = params[0].precision;
    b->integrator = params[0].integrator;
    b->P.assign(params, params + ninst);
    b->capBins = capTot;
    const size_t n = (size_t)ntot;
    // chunk and tile tables
    std::vector<int> cs, chunkInst, chunk0, ts, tileInst, tile0, dtEntry, bEntry;
    size_t ND = 0, NB = 0;  // entries of dt and of bounds partials
    std::vector<BInst> hI(ninst);
    const int chunk = chunk_slots(ntot);
    long long off = 0, base = 0;
    int tbase = 0;
    for (int k = 0; k < ninst; ++k) {
        const sph_params_t &P = params[k];
        const int c0 = (int)cs.size();
        chunk0.push_back(c0);
        for (long long c = 0; c < P.n; c += chunk) {
            cs.push_back((int)(off + c));
            chunkInst.push_back(k);
        }
        tile0.push_back((int)ts.size());
        for (long long c = 0; c < P.n; c += kTile) {
            ts.push_back((int)(off + c));
            tileInst.push_back(k);
        }
        BInst &I = hI[k];
        std::memset(&I, 0, sizeof I);
        const int nt = (int)ts.size() - tile0.back(), nc = (int)cs.size() - c0;
        I.dt0 = (int)ND;
        I.dtn = std::min(nt, kDtEntries);
        for (int j = 0; j < nt; ++j) dtEntry.push_back(nt <= kDtEntries ? I.dt0 + j : ~(I.dt0 + j % kDtEntries));
        ND += I.dtn;
        I.b0 = (int)NB;
        I.bn = std::min(nc, kBoundsEntries);
        I.shares = nc > kBoundsEntries;
        for (int j = 0; j < nc; ++j) bEntry.push_back(nc <= kBoundsEntries ? I.b0 + j : ~(I.b0 + j % kBoundsEntries));
        NB += I.bn;
        I.disp = I.vbound = I.abound = INFINITY;
        I.off = (int)off;
        I.n = (int)P.n;
        I.active = 1;
        I.advance_t = 1;
        I.cap = P.cell_capacity > 0 ? P.cell_capacity : P.n * 8 + 4096;
        I.cellBase = base;
        I.tileBase = tbase;
        tbase += (int)tile_room(I.cap);
        base += bin_room(I.cap);
        I.duration = P.duration;
        I.fixed_dt = P.fixed_dt;
        I.damping = P.damping;
        I.rho0 = P.rho0;
        I.gamma = P.gamma;
        I.co = P.co;
        I.B = P.B;
        I.Pb = P.Pb;
        I.alpha = P.alpha;
        I.beta = P.beta;
        I.r0 = P.r0;
        I.D = P.D;
        I.p1 = P.p1;
        I.p2 = P.p2;
        I.g = P.gravity;
        I.qmax = P.qmax;
        I.scale = P.scale;
        I.gamma_c = P.gamma_c;
        I.gamma_f = P.gamma_f;
        I.strict = P.strict;
        b->whole = b->whole && whole_exponent(P.p1) && whole_exponent(P.p2);
        I.kernel = P.kernel;
        b->offs.push_back((int)off);
        off += P.n;
    }
    b->offs.push_back((int)off);
    cs.push_back((int)off);
    chunk0.push_back((int)chunkInst.size());
    b->NC = (int)chunkInst.size();
    ts.push_back((int)off);
    tile0.push_back((int)tileInst.size());
    b->NT = (int)tileInst.size();
    // the scan's workgroups: as many for each instance where that is few enough
    std::vector<int> wg0{0}, wgInst;
    int most = 1;
    for (int k = 0; k < ninst; ++k) {
        const int w = scan_groups(ninst, hI[k].n, tile_room(hI[k].cap));
        most = std::max(most, w);
        wg0.push_back(wg0.back() + w);
    }
    if ((long long)most * ninst <= kScanAlike) {
        b->scan = dim3(most, ninst);
    } else {
        b->scan = dim3(wg0.back());
        wgInst.resize(wg0.back());
        for (int k = 0; k < ninst; ++k) std::fill(wgInst.begin() + wg0[k], wgInst.begin() + wg0[k + 1], k);
    }
    std::vector<int> instOf(n);
    for (int k = 0; k < ninst; ++k)
        for (int i = b->offs[k]; i < b->offs[k + 1]; ++i) instOf[i] = k;
    const size_t nd = 15;
    const size_t bytes = n * (nd * sizeof(double) + sizeof(int) + 8) + 1024;
    bool ok = true;
    for (int k = 0; k < 2 && ok; ++k) {
        ok = hipMalloc(&b->arena[k], bytes) == hipSuccess;
        if (!ok) break;
        char *p = (char *)b->arena[k];
        double **fields[] = {&b->buf[k].x,  &b->buf[k].y,   &b->buf[k].vx,   &b->buf[k].vy, &b->buf[k].rho,
                             &b->buf[k].ax, &b->buf[k].ay,  &b->buf[k].drho, &b->buf[k].x0, &b->buf[k].y0,
                             &b->buf[k].vx0, &b->buf[k].vy0, &b->buf[k].rho0, &b->buf[k].m, &b->buf[k].h};
        for (double **f : fields) {
            *f = (double *)p;
            p += n * sizeof(double);
        }
        b->buf[k].id = (int *)p;
        p += n * sizeof(int);
        b->buf[k].label = (int8_t *)p;
    }
    const size_t ra = b->precision == SPH_PREC_FP32C ? sizeof(Rec<float>::A) : sizeof(Rec<double>::A);
    // the uniform forms' records (16-B A, float4 / double4 B) fit in these
    const size_t rb = b->precision == SPH_PREC_FP32C ? sizeof(float4) : sizeof(Rec<double>::B);
    static_assert(sizeof(Rec<float>::A) >= sizeof(double2) && sizeof(Rec<double>::A) >= sizeof(double2) &&
                      sizeof(Rec<double>::B) >= sizeof(double4) && sizeof(float4) >= sizeof(Rec<float>::B),
                  "record buffers hold every format");
    const size_t uk = b->precision == SPH_PREC_FP32C ? uniform_const_size_fp32() : uniform_const_size_fp64();
    const size_t part_b_bytes = sizeof(unsigned long long) * kBoundsVQ * NB;
    b->part_d_bytes = sizeof(unsigned long long) * kDtQ * ND;
    ok = ok && hipMalloc(&b->inst, sizeof(BInst) * ninst) == hipSuccess &&
         hipMalloc(&b->view, sizeof(Ctrl)) == hipSuccess && hipMalloc(&b->instOf, sizeof(int) * n) == hipSuccess &&
         hipMalloc(&b->cs, sizeof(int) * cs.size()) == hipSuccess &&
         hipMalloc(&b->chunkInst, sizeof(int) * chunkInst.size()) == hipSuccess &&
         hipMalloc(&b->chunk0, sizeof(int) * chunk0.size()) == hipSuccess &&
         hipMalloc(&b->ts, sizeof(int) * ts.size()) == hipSuccess &&
         hipMalloc(&b->tileInst, sizeof(int) * tileInst.size()) == hipSuccess &&
         hipMalloc(&b->tile0, sizeof(int) * tile0.size()) == hipSuccess &&
         hipMalloc(&b->wg0, sizeof(int) * wg0.size()) == hipSuccess &&
         (wgInst.empty() || hipMalloc(&b->wgInst, sizeof(int) * wgInst.size()) == hipSuccess) &&
         hipMalloc(&b->bin, sizeof(int) * n) == hipSuccess && hipMalloc(&b->rank, sizeof(int) * n) == hipSuccess &&
         hipMalloc(&b->perm, sizeof(int) * n) == hipSuccess && hipMalloc(&b->perm0, sizeof(int) * n) == hipSuccess &&
         hipMalloc(&b->cxy_s, sizeof(int2) * n) == hipSuccess &&
         hipMalloc(&b->counts, sizeof(int) * (capTot + 1)) == hipSuccess &&
         hipMalloc(&b->cellStart, sizeof(int) * (capTot + 2)) == hipSuccess &&
         hipMalloc(&b->binflag, sizeof(int) * (capTot + 1)) == hipSuccess &&
         hipMalloc(&b->tileSums, sizeof(int) * kTileStride * tiles) == hipSuccess &&
         hipMemset(b->tileSums, 0, sizeof(int) * kTileStride * tiles) == hipSuccess &&
         hipMalloc(&b->part_b, part_b_bytes) == hipSuccess &&
         hipMalloc(&b->part_d, b->part_d_bytes) == hipSuccess &&
         hipMalloc(&b->bEntry, sizeof(int) * bEntry.size()) == hipSuccess &&
         hipMalloc(&b->dtEntry, sizeof(int) * dtEntry.size()) == hipSuccess &&
         hipMemset(b->part_b, 0, part_b_bytes) == hipSuccess &&
         hipMalloc(&b->recA, ra * n) == hipSuccess && hipMalloc(&b->recB, rb * n) == hipSuccess &&
         hipMalloc(&b->queue, sizeof(int) * kQueueInts) == hipSuccess &&
         hipMalloc(&b->uniK, uk * ninst) == hipSuccess && hipMalloc(&b->hm, sizeof(double) * 4 * ninst) == hipSuccess;
    if (!ok) {
        free_batch(b);
        return fail(SPH_ENOMEM, "device allocation for a batch of %lld particles failed", ntot);
    }
    Ctrl v;
    std::memset(&v, 0, sizeof v);
    v.active = 1;
    ok = hipMemcpy(b->inst, hI.data(), sizeof(BInst) * ninst, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->view, &v, sizeof v, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->instOf, instOf.data(), sizeof(int) * n, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->cs, cs.data(), sizeof(int) * cs.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->chunkInst, chunkInst.data(), sizeof(int) * chunkInst.size(), hipMemcpyHostToDevice) ==
             hipSuccess &&
         hipMemcpy(b->chunk0, chunk0.data(), sizeof(int) * chunk0.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->ts, ts.data(), sizeof(int) * ts.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->tileInst, tileInst.data(), sizeof(int) * tileInst.size(), hipMemcpyHostToDevice) ==
             hipSuccess &&
         hipMemcpy(b->tile0, tile0.data(), sizeof(int) * tile0.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->bEntry, bEntry.data(), sizeof(int) * bEntry.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->dtEntry, dtEntry.data(), sizeof(int) * dtEntry.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->wg0, wg0.data(), sizeof(int) * wg0.size(), hipMemcpyHostToDevice) == hipSuccess &&
         (wgInst.empty() ||
          hipMemcpy(b->wgInst, wgInst.data(), sizeof(int) * wgInst.size(), hipMemcpyHostToDevice) == hipSuccess) &&
         hipMemset(b->counts, 0, sizeof(int) * (capTot + 1)) == hipSuccess &&
         hipMemset(b->cellStart, 0, sizeof(int) * (capTot + 2)) == hipSuccess &&
         hipMemset(b->binflag, 0, sizeof(int) * (capTot + 1)) == hipSuccess &&
         hipMemset(b->queue, 0, sizeof(int) * kQueueInts) == hipSuccess;
    int dev = 0;
    if (ok && hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&b->cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        b->cus = 0;
    if (!ok) {
        free_batch(b);
        return fail(SPH_EHIP, "batch initialisation failed");
    }
    *out = b;
    return 0;
}

int sph_batch_destroy(sph_batch_t *b) {
    if (!b) return 0;
    hipDeviceSynchronize();
    free_batch(b);
    return 0;
}

int sph_batch_upload(sph_batch_t *b, const sph_state_t *st, void *stream) {
    if (!b || !st || !st->x || !st->y || !st->vx || !st->vy || !st->rho || !st->m || !st->h || !st->label)
        return fail(SPH_EINVAL, "upload needs x, y, vx, vy, rho, m, h and label");
    hipStream_t s = (hipStream_t)stream;
    b->cur = 0;
    b->dt_fresh = false;
    // the last state's partials, which shared entries would keep
    HIPCHK(hipMemsetAsync(b->part_d, 0, b->part_d_bytes, s));
    kb_upload<<<nblk_b(b->n), kBlock, 0, s>>>(b->buf[0], *st, b->n);
    HIPCHK(hipGetLastError());
    b->loaded = true;
    HIPCHK(hipStreamSynchronize(s));
    std::vector<BInst> hI(b->K);
    HIPCHK(hipMemcpy(hI.data(), b->inst, sizeof(BInst) * b->K, hipMemcpyDeviceToHost));
    for (auto &I : hI) {
        I.t = 0.0;
        I.step = 0;
        I.dt = I.dt_c = I.dt_f = 0.0;
        I.flags = 0;
        I.active = 1;
        I.disp = I.vbound = I.abound = INFINITY;
    }
    HIPCHK(hipMemcpy(b->inst, hI.data(), sizeof(BInst) * b->K, hipMemcpyHostToDevice));
    // the uniform pass when every instance has one h and one fluid mass and
    // its parameters allow it; a batch has no dynamic h, so this holds until
    // the next upload
    kb_hm_range<<<b->K, kBlock, 0, s>>>(b->inst, b->buf[0], b->hm);
    HIPCHK(hipGetLastError());
    std::vector<double> hm(4 * (size_t)b->K);
    HIPCHK(hipMemcpyAsync(hm.data(), b->hm, sizeof(double) * hm.size(), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    bool uni = b->n <= kUniformMaxN;  // the records of all instances, addressed with 32-bit byte offsets
    for (int k = 0; k < b->K && uni; ++k) {
        const double *v = &hm[4 * (size_t)k];
        uni = v[0] == v[1] && v[2] == v[3] && uniform_eligible(b->P[k], v[0]);
    }
    if (uni) {
        const bool f32 = b->precision == SPH_PREC_FP32C;
        const size_t uk = f32 ? uniform_const_size_fp32() : uniform_const_size_fp64();
        std::vector<unsigned char> blk(uk * (size_t)b->K);
        for (int k = 0; k < b->K; ++k) {
            const UniformParams u = make_uniform_params(b->P[k], hm[4 * (size_t)k], hm[4 * (size_t)k + 2]);
            if (f32) uniform_const_fp32(u, blk.data() + uk * k);
            else uniform_const_fp64(u, blk.data() + uk * k);
        }
        HIPCHK(hipMemcpy(b->uniK, blk.data(), blk.size(), hipMemcpyHostToDevice));
    }
    // m and h stay in place for the uniform pass (the upload's buffer, slot =
    // id): every instance's one h in its control block
    for (int k = 0; k < b->K; ++k) {
        hI[k].uh_on = uni ? 1 : 0;
        hI[k].uh = uni ? hm[4 * (size_t)k] : 0.0;
    }
    HIPCHK(hipMemcpy(b->inst, hI.data(), sizeof(BInst) * b->K, hipMemcpyHostToDevice));
    if (uni != b->uni) {  // another record format and pair kernel
        b->uni = uni;
        b->queue_grid = 0;
    }
    return 0;
}

int sph_batch_pair_form(sph_batch_t *b, int32_t *form) {
    if (!b || !form) return fail(SPH_EINVAL, "NULL argument");
    if (!b->loaded) return fail(SPH_ESTATE, "no state: call sph_batch_upload first");
    *form = b->precision == SPH_PREC_FP32C ? (b->uni ? SPH_PAIR_FP32C_UNIFORM : SPH_PAIR_FP32C)
                                           : (b->uni ? SPH_PAIR_FP64_UNIFORM : SPH_PAIR_FP64);
    return 0;
}

int sph_batch_download(sph_batch_t *b, const sph_state_t *st, void *stream) {
    if (!b || !st) return fail(SPH_EINVAL, "NULL argument");
    if (!b->loaded) return fail(SPH_ESTATE, "no state: call sph_batch_upload first");
    kb_download<<<nblk_b(b->n), kBlock, 0, (hipStream_t)stream>>>(b->buf[b->cur], *st, b->inst, b->instOf, b->n,
                                                                  b->buf[0].m, b->buf[0].h);
    HIPCHK(hipGetLastError());
    return 0;
}

// Launched one by one, whatever use_graph, as sph_step.
int sph_batch_step(sph_batch_t *b, int64_t nsteps, int32_t use_graph, void *stream) {
    (void)use_graph;
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    if (nsteps < 0) return fail(SPH_EINVAL, "nsteps < 0");
    if (!b->loaded) return fail(SPH_ESTATE, "no state: call sph_batch_upload first");
    size_queue(b);
    for (int64_t k = 0; k < nsteps; ++k) {
        int rc = b_step(b, (hipStream_t)stream);
        if (rc) return rc;
    }
    return 0;
}

int sph_batch_status(sph_batch_t *b, double *out_d, int64_t *out_i, void *stream) {
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    HIPCHK(hipStreamSynchronize((hipStream_t)stream));
    std::vector<BInst> hI(b->K);
    HIPCHK(hipMemcpy(hI.data(), b->inst, sizeof(BInst) * b->K, hipMemcpyDeviceToHost));
    for (int k = 0; k < b->K; ++k) {
        if (out_d) {
            out_d[4 * k + 0] = hI[k].t;
            out_d[4 * k + 1] = hI[k].dt;
            out_d[4 * k + 2] = hI[k].dt_c;
            out_d[4 * k + 3] = hI[k].dt_f;
        }
        if (out_i) {
            out_i[2 * k + 0] = hI[k].step;
            out_i[2 * k + 1] = hI[k].flags;
        }
    }
    return 0;
}

int sph_batch_set_tuning(sph_batch_t *b, int32_t pair_threads) {
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    if (pair_threads != 64 && pair_threads != 128 && pair_threads != 256)
        return fail(SPH_EINVAL, "pair_threads must be 64, 128 or 256");
    if (pair_threads != b->pair_threads) {
        b->pair_threads = pair_threads;
        b->queue_grid = 0;
    }
    return 0;
}

int sph_batch_set_list_len(sph_batch_t *b, int32_t list_len) {
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    if (list_len != 0 && list_len != 16 && list_len != 24 && list_len != 32)
        return fail(SPH_EINVAL, "list_len must be 0, 16, 24 or 32");
    if (list_len != b->list_len) {
        b->list_len = list_len;
        b->queue_grid = 0;
    }
    return 0;
}

int sph_batch_set_persistent(sph_batch_t *b, int32_t on) {
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    if (on != 0 && on != 1) return fail(SPH_EINVAL, "persistent must be 0 or 1");
    if (on != b->persistent) {
        b->persistent = on;
        b->queue_grid = 0;
    }
    return 0;
}

int sph_batch_set_border_bounds(sph_batch_t *b, int32_t on) {
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    b->border_bounds = on ? 1 : 0;
    return 0;
}

int sph_batch_border_count(sph_batch_t *b, int64_t *counts, void *stream) {
    if (!b || !counts) return fail(SPH_EINVAL, "NULL argument");
    HIPCHK(hipStreamSynchronize((hipStream_t)stream));
    std::vector<BInst> hI(b->K);
    HIPCHK(hipMemcpy(hI.data(), b->inst, sizeof(BInst) * b->K, hipMemcpyDeviceToHost));
    for (int k = 0; k < b->K; ++k) counts[k] = hI[k].border_updates;
    return 0;
}

int sph_batch_timing_enable(sph_batch_t *b, int32_t on) {
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    b->timing = on != 0;
    b->n_ev = 0;
    return 0;
}

int sph_batch_timing_read(sph_batch_t *b, double *avg_ms_pair, int64_t *count, int32_t reset) {
    if (!b) return fail(SPH_EINVAL, "batch is NULL");
    HIPCHK(hipDeviceSynchronize());
    double tot = 0.0;
    int64_t k = 0;
    for (size_t i = 0; i + 1 < b->n_ev; i += 2) {
        float ms = 0.f;
        HIPCHK(hipEventElapsedTime(&ms, b->ev[i], b->ev[i + 1]));
        tot += ms;
        ++k;
    }
    if (avg_ms_pair) *avg_ms_pair = k ? tot / k : 0.0;
    if (count) *count = k;
    if (reset) b->n_ev = 0;
    return 0;
}

}  // extern "C"
