// SSSP epoch kernels for gfx950.
//
//  * Pull epoch (Bellman-Ford, in place): dist[u] = min(dist[u],
//    min_{(v,w)} dist[v]+w), the arithmetic of epoch_sssp_pull_cpu_one_to_one
//    (src/kernels/cpu/sssp.cuh:155-182) with int32 weights and a saturating
//    sentinel.  Vertex mappings: thread / wavefront / workgroup per vertex
//    (counterparts of src/kernels/gpu/sssp.cuh:120-281) and the fused
//    degree-bucketed plan (hub chunks with atomicMin, workgroup, wavefront,
//    16-lane, 4-lane and 1-lane groups in one launch).
//  * Push epoch: relax the out-edges of the active frontier with atomicMin and
//    append improved vertices (deduplicated through a bitmap) to the next
//    frontier, wavefront-aggregated.
//  * Device-driven loop (step / control / compact launches per epoch, see
//    frontier.h): the controller picks the next direction (pull when the
//    frontier's degree sum exceeds m/alpha) and stops the loop when nothing
//    changed, so the host only enqueues launches.
#include <algorithm>
#include <cmath>
#include <functional>
#include <vector>
#include <cstring>

#include "frontier.h"

namespace hc {

// ---------------------------------------------------------------------------
// Row reductions
// ---------------------------------------------------------------------------

__device__ __forceinline__ bool changed_bit(const Staged<uint32_t> &bm, int32_t v) {
    return (bm[v >> 5] >> (v & 31)) & 1u;
}

// Minimum candidate over edges [b, e) taken G apart starting at b+lane.
// Trips of four edges per lane with predicated loads (a short row is one
// trip of parallel loads, not a serial tail), and the next trip's ids and
// weights are loaded before this trip's distance gathers, so each trip costs
// about one memory round trip instead of two.
// FILTER: only neighbours set in `changed` (the vertices whose distance
// changed in the previous epoch) are gathered; the others cannot lower the
// row below its current value.  `gathered` counts the gathers.
// Neighbour distances through a 16-bit mirror: half the bytes per gathered
// entry, so twice as many vertices fit each cache.  0xFFFF: unreached;
// 0xFFFE: too large for 16 bits, read the int32 array.  The mirror is
// rebuilt from the int32 distances before every pull epoch and written
// during the sweep by whoever lowers an entry; a row lowered concurrently by
// several hub chunks may keep a stale (larger) mirror entry until the next
// rebuild, which costs nothing in exactness: the row is marked changed, so
// another epoch runs, and it starts from a fresh mirror.
struct Dist16Reader {
    const uint16_t *h;
    const int32_t *full;
    __device__ __forceinline__ int32_t operator[](int32_t v) const {
        const uint32_t x = h[v];
        return x < 0xFFFEu ? int32_t(x) : (x == 0xFFFFu ? HC_INF_DIST : full[v]);
    }
};

__device__ __forceinline__ uint16_t dist16(int32_t d) {
    return d >= HC_INF_DIST ? uint16_t(0xFFFF) : (d >= 0xFFFE ? uint16_t(0xFFFE) : uint16_t(d));
}

template <int G, bool FILTER, typename DR, typename OffT>
__device__ __forceinline__ int32_t row_min(const GraphView<OffT> &g,
                                           const DR &dist,
                                           const Staged<uint32_t> &changed,
                                           OffT b, OffT e, int lane, uint32_t &gathered) {
    int32_t m = HC_INF_DIST;
    OffT i = b + OffT(lane);
    if (i >= e) return m;
    int32_t v[4], w[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const OffT k = i + OffT(r * G);
        v[r] = k < e ? ldnt(&g.adj[k]) : -1;
        w[r] = k < e ? ldnt(&g.wt[k]) : 0;
    }
    for (;;) {
        const OffT ni = i + OffT(4 * G);
        int32_t nv[4] = {-1, -1, -1, -1}, nw[4] = {0, 0, 0, 0};
        if (ni < e) {  // short rows skip the prefetch instructions entirely
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const OffT k = ni + OffT(r * G);
                nv[r] = k < e ? ldnt(&g.adj[k]) : -1;
                nw[r] = k < e ? ldnt(&g.wt[k]) : 0;
            }
        }
        bool use[4];
#pragma unroll
        for (int r = 0; r < 4; r++) use[r] = v[r] >= 0 && (!FILTER || changed_bit(changed, v[r]));
        int32_t d[4];
#pragma unroll
        for (int r = 0; r < 4; r++) d[r] = use[r] ? dist[v[r]] : HC_INF_DIST;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            m = min(m, relax(d[r], w[r]));
            gathered += use[r] ? 1u : 0u;
        }
        if (ni >= e) break;
        for (int r = 0; r < 4; r++) {
            v[r] = nv[r];
            w[r] = nw[r];
        }
        i = ni;
    }
    return m;
}

// Workgroup minimum for any blockDim that is a multiple of 64 (<= 1024).
// The leading barrier keeps the LDS slots from being overwritten while a
// previous call is still reading them (the reuse race of
// src/kernels/gpu/sssp.cuh:259-275).
__device__ __forceinline__ int32_t block_min(int32_t m) {
    __shared__ int32_t s_min[16];
    m = group_min<64>(m);
    __syncthreads();
    if (lane_id() == 0) s_min[threadIdx.x / kWave] = m;
    __syncthreads();
    int32_t r = s_min[0];
    const int nw = blockDim.x / kWave;
    for (int i = 1; i < nw; i++) r = min(r, s_min[i]);
    return r;
}

// ---------------------------------------------------------------------------
// Fused degree-bucketed pull sweep
// ---------------------------------------------------------------------------

// Lowers dist[u] to m when that is lower; chg: this call lowered it.  For
// rows that several groups of one sweep may lower (hub chunks, the column
// blocks of a row): atomicMin decides, a stale `cur` only costs an atomic.
__device__ __forceinline__ void lower_shared_row(int32_t *dist, uint16_t *d16, int32_t u,
                                                 int32_t cur, int32_t m, bool &chg) {
    if (m < cur) {
        const int32_t old = atomicMin(&dist[u], m);
        chg = m < old;
        // Two groups lowering one row may store their mirror values out of
        // order; a stale (larger) entry only weakens this epoch, and the row
        // is marked changed, so the next epoch starts from a rebuild.
        if (chg && d16) d16[u] = dist16(m);
    }
}

// One row of class c per group of G lanes.  SHARED: other groups of the
// sweep may lower the same row (column-blocked sweeps), so the row is
// lowered with atomicMin.
template <int G, bool FILTER, bool SHARED = false, typename DR, typename OffT>
__device__ __forceinline__ void pull_group(const PlanDev &p, int c, int k,
                                           const GraphView<OffT> &g,
                                           const DR &rd,
                                           const Staged<uint32_t> &changed,
                                           int32_t *__restrict__ dist, uint16_t *d16,
                                           bool &chg, int32_t &u, uint32_t &gathered,
                                           int64_t &deg) {
    constexpr int PER = kBlock / G;
    const int gid = threadIdx.x / G, lane = threadIdx.x % G;
    const int idx = k * PER + gid;
    if (idx < p.cnt[c]) {
        int32_t uu = p.list[c] ? p.list[c][idx] : p.beg[c] + idx;
        const OffT b = g.rbeg(uu), e = g.rend(uu);
        // The row's own distance is read with its bounds, before the
        // gathers: in a pull epoch only this group writes it (unless SHARED).
        const int32_t cur = lane == 0 ? dist[uu] : 0;
        int32_t m = row_min<G, FILTER>(g, rd, changed, b, e, lane, gathered);
        if (G > 1) m = group_min<G>(m);
        if (lane == 0) {
            if (SHARED) {
                lower_shared_row(dist, d16, uu, cur, m, chg);
            } else if (m < cur) {
                dist[uu] = m;
                if (d16) d16[uu] = dist16(m);
                chg = true;
            }
            u = uu;
            deg = int64_t(e - b);
        }
    }
}


// One pull sweep over the plan's units (grid-stride).  LOOP: changed
// vertices are set in the next-frontier bitmap and counted (first setting
// only: hub chunks may lower the same vertex twice); otherwise changes are
// counted for the epoch API.
// Neighbour distances are read through `rd` (hub entries from the LDS
// snapshot); the row's own distance is read and written in global memory.
// A stale snapshot only delays an improvement to a later epoch: values only
// decrease, and an epoch without any change had nothing stale to read.
// FILTER: gather only neighbours in `changed` (see row_min); `gathered`
// counts the gathers.
template <bool LOOP, bool FILTER, typename DR, typename OffT>
__device__ __forceinline__ void sssp_pull_sweep(const PlanDev &p, const GraphView<OffT> &g,
                                const DR &rd, const Staged<uint32_t> &changed,
                                int32_t *__restrict__ dist, uint16_t *d16, uint32_t *next_bm,
                                uint32_t &cnt, unsigned long long &edges_acc,
                                uint32_t &gathered) {
    const int total = p.unit_start[kNumClasses];
    for (int unit = blockIdx.x; unit < total; unit += gridDim.x) {
        int c = 0;
        while (unit >= p.unit_start[c + 1]) c++;
        const int k = unit - p.unit_start[c];
        bool chg = false;
        int32_t u = 0;
        int64_t deg = -1;  // the row's degree when its bounds were read here
        if (c <= 1) {
            int32_t uu;
            OffT b, e;
            if (c == 0) {
                HubChunk h = p.chunks[k];
                uu = h.u;
                b = OffT(h.b);
                e = OffT(h.e);
            } else {
                uu = p.list[1] ? p.list[1][k] : p.beg[1] + k;
                b = g.rbeg(uu);
                e = g.rend(uu);
                deg = int64_t(e - b);
            }
            int32_t m = block_min(row_min<kBlock, FILTER>(g, rd, changed, b, e, threadIdx.x,
                                                          gathered));
            if (threadIdx.x == 0) {
                if (c == 0) {
                    lower_shared_row(dist, d16, uu, dist[uu], m, chg);
                } else {
                    int32_t cur = dist[uu];
                    if (m < cur) {
                        dist[uu] = m;
                        if (d16) d16[uu] = dist16(m);
                        chg = true;
                    }
                }
                u = uu;
            }
        } else if (c == 2) {
            pull_group<64, FILTER>(p, c, k, g, rd, changed, dist, d16, chg, u, gathered, deg);
        } else if (c == 3) {
            pull_group<16, FILTER>(p, c, k, g, rd, changed, dist, d16, chg, u, gathered, deg);
        } else if (c == 4) {
            pull_group<4, FILTER>(p, c, k, g, rd, changed, dist, d16, chg, u, gathered, deg);
        } else {
            pull_group<1, FILTER>(p, c, k, g, rd, changed, dist, d16, chg, u, gathered, deg);
        }
        if (LOOP && c == 0) {
            // Several chunks may lower the same hub: count its bit once.
            if (wave_set_bit(next_bm, u, chg)) {
                cnt++;
                edges_acc += (unsigned long long)(g.rend(u) - g.rbeg(u));
            }
        } else if (LOOP) {
            // Any other row is swept by one group only.
            wave_or_bits(next_bm, u, chg);
            if (chg) {
                cnt++;
                edges_acc += (unsigned long long)(deg >= 0 ? deg : int64_t(g.rend(u) - g.rbeg(u)));
            }
        } else {
            cnt += chg ? 1u : 0u;
        }
    }
}

// One pull sweep over the column blocks of the graph (see colblock.hip):
// units (block k, plan unit) in block-major order, so the grid gathers from
// one block of distances at a time.  `cb` views the blocked arrays with the
// offsets of block 0; block k's slices start (n+1) k offsets later.  Plan
// classes are by mean slice degree and have no hub chunks.  A row may be
// lowered by several blocks in one sweep: atomicMin, and `counted` (the
// next-frontier bitmap, or the epoch API's seen bitmap) counts it once;
// edges_acc adds its full degree.
template <typename DR, typename OffT>
__device__ __forceinline__ void sssp_pull_sweep_cb(const PlanDev &p, const GraphView<OffT> &g,
                                   const GraphView<OffT> &cb, int K, const DR &rd,
                                   int32_t *__restrict__ dist, uint16_t *d16,
                                   uint32_t *counted, uint32_t &cnt,
                                   unsigned long long &edges_acc, uint32_t &gathered) {
    const int U = p.unit_start[kNumClasses];
    const int total = U * K;
    const Staged<uint32_t> nochg = unstaged<uint32_t>(nullptr);
    for (int unit = blockIdx.x; unit < total; unit += gridDim.x) {
        const int k = unit / U;
        const int pu = unit - k * U;
        GraphView<OffT> gk = cb;
        gk.off = cb.off + (size_t)k * ((size_t)g.n + 1);
        int c = 1;
        while (pu >= p.unit_start[c + 1]) c++;
        const int kk = pu - p.unit_start[c];
        bool chg = false;
        int32_t u = 0;
        int64_t deg = -1;
        if (c == 1) {
            const int32_t uu = p.list[1] ? p.list[1][kk] : p.beg[1] + kk;
            const int32_t m = block_min(row_min<kBlock, false>(gk, rd, nochg, gk.rbeg(uu),
                                                               gk.rend(uu), threadIdx.x,
                                                               gathered));
            if (threadIdx.x == 0) {
                lower_shared_row(dist, d16, uu, dist[uu], m, chg);
                u = uu;
            }
        } else if (c == 2) {
            pull_group<64, false, true>(p, c, kk, gk, rd, nochg, dist, d16, chg, u, gathered, deg);
        } else if (c == 3) {
            pull_group<16, false, true>(p, c, kk, gk, rd, nochg, dist, d16, chg, u, gathered, deg);
        } else if (c == 4) {
            pull_group<4, false, true>(p, c, kk, gk, rd, nochg, dist, d16, chg, u, gathered, deg);
        } else {
            pull_group<1, false, true>(p, c, kk, gk, rd, nochg, dist, d16, chg, u, gathered, deg);
        }
        if (wave_set_bit(counted, u, chg)) {
            cnt++;
            edges_acc += (unsigned long long)(g.rend(u) - g.rbeg(u));
        }
    }
}

// ---------------------------------------------------------------------------
// Push expansion of the frontier
// ---------------------------------------------------------------------------

constexpr int kPushTrip = 4;  // edges a lane of a push epoch has in flight
// Rows up to this degree take kSmallLanes lanes (two trips at most); with one
// edge in flight per lane they would want a wavefront from 17 edges on.
constexpr int32_t kPushMid = 64;

// Edges of a push epoch: the CSR's two arrays, or the weight-sorted pairs (FAR:
// with buckets).
template <typename OffT, bool FAR = false>
struct CsrEdges {
    static constexpr bool kSorted = false, kFar = FAR;
    const int32_t *adj, *wt;
    __device__ __forceinline__ int2 get(OffT i) const { return int2{adj[i], wt[i]}; }
    __device__ __forceinline__ int32_t floor(int32_t) const { return 0; }
};
template <typename OffT, bool FAR>
struct SortedEdges {
    static constexpr bool kSorted = true, kFar = FAR;
    SortedView v;
    __device__ __forceinline__ int2 get(OffT i) const { return v.e[i]; }
    __device__ __forceinline__ int32_t floor(int32_t w) const { return v.floor(w); }
};

// Relaxes the out-edges [b, e) of u (G lanes, kPushTrip edges a lane in
// flight: a trip is a chain of dependent accesses -- pair, distance, minimum,
// staging slot -- and its latency bounds the epoch); a lowered neighbour joins
// the next frontier.  Sorted edges: only those that land below `reach` are
// relaxed (HC_INF_DIST: all), and the scan stops at the first key that cannot.
// Buckets: a neighbour lowered to `thresh` or more joins the far bitmap instead
// (`nfar` counts those settings).  `lowest` is the smallest value written;
// `pairs` and `gathered` count the edges and distances read where the scan may
// stop early.
template <int G, typename ER, typename OffT>
__device__ __forceinline__ void push_range(const GraphView<OffT> &g, const ER &er,
                                           int32_t *__restrict__ dist,
                                           const FrontierBufs &fb, StepCtl *ctl,
                                           const PushOut &out,
                                           int nxt, uint32_t *wbm, int32_t u, OffT b,
                                           OffT e, int lane, uint32_t &cnt,
                                           unsigned long long &edges_acc, int32_t reach,
                                           int32_t thresh, int32_t &lowest, uint32_t &nfar,
                                           uint32_t &pairs, uint32_t &gathered) {
    const int32_t du = dist[u];
    for (OffT i = b + OffT(lane); i < e; i += OffT(kPushTrip * G)) {
        int2 x[kPushTrip];
        bool in[kPushTrip];
#pragma unroll
        for (int r = 0; r < kPushTrip; r++) {
            const OffT k = i + OffT(r * G);
            in[r] = k < e;
            x[r] = in[r] ? er.get(k) : int2{0, 0};
        }
        if (ER::kSorted && ER::kFar) pairs += (uint32_t)min((e - 1 - i) / OffT(G) + 1, OffT(kPushTrip));
        if (ER::kSorted && relax(du, er.floor(x[0].y)) >= reach) break;
        int32_t nd[kPushTrip], d[kPushTrip], old[kPushTrip];
#pragma unroll
        for (int r = 0; r < kPushTrip; r++) {
            nd[r] = in[r] ? relax(du, x[r].y) : HC_INF_DIST;
            d[r] = nd[r] < reach ? dist[x[r].x] : 0;
            if (ER::kSorted && ER::kFar) gathered += nd[r] < reach ? 1u : 0u;
        }
#pragma unroll
        for (int r = 0; r < kPushTrip; r++)
            old[r] = nd[r] < d[r] ? atomicMin(&dist[x[r].x], nd[r]) : 0;
        int32_t v[kPushTrip];
        bool lowered[kPushTrip];
#pragma unroll
        for (int r = 0; r < kPushTrip; r++) {
            v[r] = x[r].x;
            lowered[r] = nd[r] < old[r];
            if (lowered[r]) lowest = min(lowest, nd[r]);
            if (ER::kFar && lowered[r] && nd[r] >= thresh) {
                atomicOr(&fb.far[v[r] >> 5], 1u << (v[r] & 31));
                nfar++;
                lowered[r] = false;
            }
            if (!out.dedup && lowered[r]) {
                // The first edge to set v's bit appends v, now.
                const uint32_t bit = 1u << (v[r] & 31);
                lowered[r] = !(atomicOr(&wbm[v[r] >> 5], bit) & bit);
                if (lowered[r]) {
                    cnt++;
                    edges_acc += (unsigned long long)(g.rend(v[r]) - g.rbeg(v[r]));
                }
            }
        }
        // Deferred: a lowered neighbour is a candidate; the staging keeps
        // its first copy (bit `wbm`) and counts it there.
        push_out_append(out, g, fb, ctl, nxt, lowered, v, cnt, edges_acc);
    }
}

template <typename ER, typename OffT>
__device__ __forceinline__ void sssp_push_sweep(const GraphView<OffT> &g, const ER &er,
                                int32_t *__restrict__ dist,
                                const FrontierBufs &fb, StepCtl *ctl,
                                const PushOut &out, int cur,
                                int nxt, uint32_t *wbm, uint32_t &cnt,
                                unsigned long long &edges_acc, int32_t &lowest,
                                uint32_t &nfar, uint32_t &pairs, uint32_t &gathered) {
    const int32_t thresh = ER::kFar ? ctl->thresh : HC_INF_DIST;
    const int32_t reach = ER::kSorted && !ctl->far_on ? thresh : HC_INF_DIST;
    const uint32_t nch = fb.cnt[cur][3], n0 = fb.cnt[cur][0],
                   n1 = fb.cnt[cur][1], n2 = fb.cnt[cur][2];
    const uint32_t u1 = nch + n0;
    const uint32_t u2 = u1 + (n1 + kWavesPerBlock - 1) / kWavesPerBlock;
    const uint32_t total = u2 + (n2 + kSmallPerUnit - 1) / kSmallPerUnit;
    // An upper bound of the staged count: the workgroup synchronizes to check
    // for room only when the next unit could overfill the buffer.
    uint32_t staged = 0;
    for (uint32_t unit = blockIdx.x; unit < total; unit += gridDim.x) {
        const uint32_t umax = push_unit_max(unit, nch, u2, ctl);
        if (staged + umax > out.cap)
            staged = push_out_make_room(out, g, fb, ctl, nxt, umax, cnt, edges_acc);
        staged += umax;
        if (unit < nch) {
            HubChunk h = fb.ch[cur][unit];
            push_range<kBlock>(g, er, dist, fb, ctl, out, nxt, wbm, h.u, OffT(h.b), OffT(h.e),
                               threadIdx.x, cnt, edges_acc, reach, thresh, lowest, nfar,
                               pairs, gathered);
        } else if (unit < u1) {
            int32_t u = fb.q[cur][0][unit - nch];
            push_range<kBlock>(g, er, dist, fb, ctl, out, nxt, wbm, u, g.rbeg(u), g.rend(u),
                               threadIdx.x, cnt, edges_acc, reach, thresh, lowest, nfar,
                               pairs, gathered);
        } else if (unit < u2) {
            uint32_t idx = (unit - u1) * kWavesPerBlock + threadIdx.x / kWave;
            if (idx < n1) {
                int32_t u = fb.q[cur][1][idx];
                push_range<kWave>(g, er, dist, fb, ctl, out, nxt, wbm, u, g.rbeg(u), g.rend(u),
                                  lane_id(), cnt, edges_acc, reach, thresh, lowest, nfar,
                               pairs, gathered);
            }
        } else {
            uint32_t idx = (unit - u2) * kSmallPerUnit + threadIdx.x / kSmallLanes;
            if (idx < n2) {
                int32_t u = fb.q[cur][2][idx];
                push_range<kSmallLanes>(g, er, dist, fb, ctl, out, nxt, wbm, u, g.rbeg(u),
                                        g.rend(u), threadIdx.x % kSmallLanes, cnt,
                                        edges_acc, reach, thresh, lowest, nfar,
                               pairs, gathered);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Sweeps over the weight-sorted adjacency
// ---------------------------------------------------------------------------

// Distances that bound a sorted sweep (fields of the control block).
struct RowBounds {
    int32_t low, base, thresh;
};

// A settling sweep is taken when the bucket's degree sum times this exceeds
// the edges not yet done (uniform, 8M vertices, three sources: 4.09 / 4.22 / 4.27
// ms with 1, 4.08 / 4.21 / 4.25 with 2, 4.20 / 4.01 / 3.91 with 8; 1M and 4M
// vertices the same with all).
constexpr long long kSettleShare = 2;
// Within a bucket, a frontier of more than m / kBucketSweep edges is relaxed
// by a sweep over the rows instead of a push (the same graph: 4.75 ms with 2, 4.21
// with 8, 6.17 with 32).
constexpr long long kBucketSweep = 8;
// A bucket whose frontiers hold more than kLightEdges + n / 8 edges is heavy: it
// is worth two or three passes over the vertices and their launches, which a
// light one is not (3D grid of 256^3 vertices, weights 1..3, about 500 buckets:
// 30.9 ms with the limit at kLightEdges + n / 32, 16.6 at n / 8, 36.2 with
// none light).  On graphs without locality a bucket holds up to forty times as
// many as the one before it, and most of the last light one's edges are relaxed
// for nothing (uniform, 8M vertices: 40 us), so growth counts.
constexpr long long kLightEdges = 1ll << 18;

// What a sorted sweep does with a row.
enum RowJob {
    kRowPull,    // lower the row; a lowered row is changed
    kRowBucket,  // buckets: lower the row to a value below thresh; a lowered row is changed
    kRowSettle,  // buckets: lower a row at or above base; below thresh it joins the frontier
    kRowScatter  // buckets: push the edges of a row in [low, thresh) that leave the bucket
};

// Per-thread results of a sweep.
struct RowSums {
    uint32_t cnt = 0;                  // rows put into the next frontier
    unsigned long long edges = 0;      // and their degree sum
    uint32_t pairs = 0;                // sorted edges read
    uint32_t gathered = 0;             // distances read for them
    uint32_t left = 0;                 // promotions: rows reached and left at or above thresh;
                                       // pushes: settings of the far bitmap
    int32_t lowest = HC_INF_DIST;      // smallest value written (promotions: left at or above thresh)
};

// One trip of sorted_row_min: R edges a lane from edge i.  False when the
// scan is over.
template <int G, int R, typename OffT>
__device__ __forceinline__ bool sorted_trip(const SortedView &sv, const int32_t *dist, OffT i,
                                            OffT e, int lane, int32_t low, int32_t &best,
                                            int32_t &m, uint32_t &pairs, uint32_t &gathered) {
    int2 x[R];
    bool in[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const OffT k = i + OffT(r * G + lane);
        in[r] = k < e;
        x[r] = in[r] ? sv.e[k] : int2{0, 0};
        pairs += in[r] ? 1u : 0u;
    }
    int32_t d[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const bool use = in[r] && low + x[r].y < best;
        d[r] = use ? dist[x[r].x] : HC_INF_DIST;
        gathered += use ? 1u : 0u;
    }
#pragma unroll
    for (int r = 0; r < R; r++) m = min(m, relax(d[r], x[r].y));
    if (G > 1) m = group_min<G>(m);
    best = min(best, m);
    // The last lane's last edge has the trip's heaviest key.
    bool more = in[R - 1] && low + sv.floor(x[R - 1].y) < best;
    if (G > 1) more = __shfl(more ? 1 : 0, G - 1, G) != 0;
    return more;
}

// Smallest candidate over the sorted edges [b, e) of a row of distance cur,
// by a group of G lanes; every lane returns the group's minimum.  `low` is a
// lower bound of the distances that can still lower the row, so an edge is
// gathered only where low + w is below the best value so far, and the scan
// ends with the first trip that reaches a key where it is not.  Most rows end
// after a trip of two edges a lane; those that go on (unreached rows, above
// all) take longer trips, since the latency of a trip is what they wait for.
template <int G, typename OffT>
__device__ __forceinline__ int32_t sorted_row_min(const SortedView &sv, const int32_t *dist,
                                                  OffT b, OffT e, int lane, int32_t cur,
                                                  int32_t low, uint32_t &pairs,
                                                  uint32_t &gathered) {
    int32_t best = cur, m = HC_INF_DIST;
    if (!sorted_trip<G, 2>(sv, dist, b, e, lane, low, best, m, pairs, gathered)) return m;
    // (8-byte offsets take the registers of the longer trip)
    constexpr int R = sizeof(OffT) == 8 ? 2 : 4;
    for (OffT i = b + OffT(2 * G); i < e; i += OffT(R * G))
        if (!sorted_trip<G, R>(sv, dist, i, e, lane, low, best, m, pairs, gathered)) break;
    return m;
}

// Pushes the sorted edges [b, e) of a row of distance du that reach thresh or
// more (the lighter ones were relaxed by the bucket's push epochs).
template <int G, typename OffT>
__device__ __forceinline__ void scatter_row(const SortedView &sv, int32_t *dist, OffT b, OffT e,
                                            int lane, int32_t du, int32_t thresh,
                                            uint32_t &pairs, uint32_t &gathered) {
    for (OffT i = b + OffT(lane); i < e; i += OffT(G)) {
        const int2 x = sv.e[i];
        pairs++;
        const int32_t nd = relax(du, x.y);
        if (nd < thresh || nd >= HC_INF_DIST) continue;
        gathered++;
        if (nd < dist[x.x]) atomicMin(&dist[x.x], nd);
    }
}

// The bound of a row's scan, and whether the row is swept at all.
template <int JOB>
__device__ __forceinline__ bool row_wanted(const RowBounds &c, int32_t cur) {
    if (JOB == kRowPull || JOB == kRowBucket) return cur > c.low;
    if (JOB == kRowSettle) return cur >= c.base;
    return cur >= c.low && cur < c.thresh;
}

// A row of a wavefront's block, one per lane.
template <typename OffT>
struct RowHead {
    int32_t u, cur;
    OffT b, e;
    bool ok;
};

// Outcome of a row: its new value is min(cur, m); `hit` puts it into the next
// frontier.
template <int JOB>
__device__ __forceinline__ bool row_done(const RowBounds &ct, int32_t cur, int32_t top, int32_t m,
                                         unsigned long long deg, RowSums &s) {
    bool hit = m < top;
    if (JOB != kRowSettle) {
        if (hit) s.lowest = min(s.lowest, m);
    } else {
        const int32_t d = min(cur, m);
        hit = d < ct.thresh;
        if (!hit && d < HC_INF_DIST) {
            s.left++;
            s.lowest = min(s.lowest, d);
        }
    }
    if (hit) {
        s.cnt++;
        s.edges += deg;
    }
    return hit;
}

// The same for a chunk of a shared row (one lane).
template <int JOB, typename OffT>
__device__ __forceinline__ void shared_done(const RowBounds &ct, const GraphView<OffT> &g,
                                            int32_t *dist, uint32_t *wbm, int32_t u, int32_t cur,
                                            int32_t top, int32_t m, RowSums &s) {
    int32_t d = cur;
    bool hit = false;
    if (m < top) {
        const int32_t old = atomicMin(&dist[u], m);
        hit = m < old;
        d = min(old, m);
    }
    if (JOB != kRowSettle) {
        if (hit) s.lowest = min(s.lowest, m);
    } else {
        hit = d < ct.thresh;
        if (!hit && d < HC_INF_DIST) {
            s.left++;
            s.lowest = min(s.lowest, d);
        }
    }
    if (hit) {
        const uint32_t bit = 1u << (u & 31);
        if (!(atomicOr(&wbm[u >> 5], bit) & bit)) {
            s.cnt++;
            s.edges += (unsigned long long)(g.rend(u) - g.rbeg(u));
        }
    }
}

template <int JOB>
__device__ __forceinline__ int32_t row_top(const RowBounds &ct, int32_t cur) {
    return JOB == kRowBucket ? min(cur, ct.thresh) : cur;
}

// The wanted rows of a wavefront's block (one row head per lane), those of
// lanes j0, j0 + jstep, ... (several wavefronts may share a block; a row's
// wavefront must not depend on distances, which they read at different
// times), G lanes per row.  A row's distance and bounds are read by one lane,
// coalesced over the block, so a block without wanted rows costs its heads
// only; the wanted ones are packed together.
// SHARED: heads are chunks of hub rows, which several wavefronts lower: with
// atomicMin, the row's bit counted by the chunk that sets it, and a chunk of a
// settling sweep that finds the row below thresh sets the bit whoever lowered
// it; `left` then counts a hub by each chunk's view, which matters only when
// no row at all is below thresh.
template <int JOB, int G, bool SHARED, typename OffT>
__device__ __forceinline__ void sorted_block(const RowHead<OffT> &h, int j0, int jstep,
                                             const RowBounds &ct, const GraphView<OffT> &g,
                                             const SortedView &sv, int32_t *dist, uint32_t *wbm,
                                             RowSums &s) {
    const int lane = lane_id();
    const bool want = h.ok && lane % jstep == j0 && row_wanted<JOB>(ct, h.cur);
    bool hit = false;  // of this lane's row
    if (G == 1) {
        if (want) {
            if (JOB == kRowScatter) {
                scatter_row<1>(sv, dist, h.b, h.e, 0, h.cur, ct.thresh, s.pairs, s.gathered);
            } else {
                const int32_t top = row_top<JOB>(ct, h.cur);
                const int32_t m =
                    sorted_row_min<1>(sv, dist, h.b, h.e, 0, top, ct.low, s.pairs, s.gathered);
                if (m < top) dist[h.u] = m;
                hit = row_done<JOB>(ct, h.cur, top, m, (unsigned long long)(h.e - h.b), s);
            }
        }
    } else {
        constexpr int PER = kWave / G;
        const uint64_t mask = __ballot(want);
        const int n = __popcll(mask);
        // Lane r learns the lane of the r-th wanted row (the others fill the
        // places after them).
        const int rank = __popcll(mask & lanemask_lt());
        const int src =
            __builtin_amdgcn_ds_permute((want ? rank : n + lane - rank) << 2, lane);
        for (int j = 0; j * PER < n; j++) {
            const int gi = j * PER + lane / G;
            const bool have = gi < n;
            const int sl = __shfl(src, gi & (kWave - 1));
            const int32_t cur = __shfl(h.cur, sl);
            const int32_t u = __shfl(h.u, sl);
            const OffT b = __shfl(h.b, sl), e = __shfl(h.e, sl);
            bool ghit = false;
            if (have) {
                if (JOB == kRowScatter) {
                    scatter_row<G>(sv, dist, b, e, lane % G, cur, ct.thresh, s.pairs, s.gathered);
                } else {
                    const int32_t top = row_top<JOB>(ct, cur);
                    const int32_t m = sorted_row_min<G>(sv, dist, b, e, lane % G, top, ct.low,
                                                        s.pairs, s.gathered);
                    if (SHARED) {
                        if (lane == 0) shared_done<JOB>(ct, g, dist, wbm, u, cur, top, m, s);
                    } else if (lane % G == 0) {
                        if (m < top) dist[u] = m;
                        ghit = row_done<JOB>(ct, cur, top, m, (unsigned long long)(e - b), s);
                    }
                }
            }
            if (JOB != kRowScatter && !SHARED) {
                // The groups' outcomes back to their rows' lanes.
                for (uint64_t gm = __ballot(ghit); gm; gm &= gm - 1) {
                    const int l = __ffsll((unsigned long long)gm) - 1;
                    hit = hit || lane == __builtin_amdgcn_readlane(sl, l);
                }
            }
        }
    }
    if (JOB != kRowScatter && !SHARED) wave_or_bits(wbm, h.u, hit);
}

// Wavefronts that share a block of 64 heads: 16 for hub chunks
// and heavy rows (64 lanes a row), and while the plan has fewer blocks than
// the grid wavefronts, four for the lighter ones.
constexpr int kHeavySplit = 16;

// One sweep over the plan (grid-stride, wavefront units), the next unit's
// heads read ahead of this unit's rows.
template <int JOB, typename OffT>
__device__ __forceinline__ void sorted_sweep(const PlanDev &p, const RowBounds &ct,
                                             const GraphView<OffT> &g, const SortedView &sv,
                                             int32_t *dist, uint32_t *wbm, RowSums &s) {
    const int b0 = (p.cnt[0] + 63) / 64, b2 = (p.cnt[2] + 63) / 64;
    const int b3 = (p.cnt[3] + 63) / 64, b4 = (p.cnt[4] + 63) / 64, b5 = (p.cnt[5] + 63) / 64;
    const int stride = gridDim.x * kWavesPerBlock;
    const int split = b3 + b4 < stride ? 4 : 1;
    const int t0 = b0 * kHeavySplit, t2 = t0 + b2 * kHeavySplit;
    const int t3 = t2 + b3 * 4 * split, t4 = t3 + b4 * split, total = t4 + b5;
    const int lane = lane_id();
    // The lane's row of a unit (class indexes are constants: an indexed plan
    // would be copied to scratch).
    auto head = [&](int unit) {
        RowHead<OffT> h{0, 0, OffT(0), OffT(0), false};
        int i = 0, beg = 0;
        const int32_t *list = nullptr;
        if (unit < t0) {
            i = unit / kHeavySplit * 64 + lane;
            if (i < p.cnt[0]) {
                const HubChunk c = p.chunks[i];
                h.u = c.u;
                h.b = OffT(c.b);
                h.e = OffT(c.e);
                h.cur = dist[c.u];
                // The chunk's first key rules out the rest of it.
                h.ok = JOB == kRowScatter ||
                       ct.low + sv.floor(sv.e[c.b].y) < row_top<JOB>(ct, h.cur) ||
                       (JOB == kRowSettle && h.cur >= ct.base);
            }
            return h;
        } else if (unit < t2) {
            i = (unit - t0) / kHeavySplit * 64 + lane;
            h.ok = i < p.cnt[2];
            beg = p.beg[2];
            list = p.list[2];
        } else if (unit < t3) {
            i = (unit - t2) / (4 * split) * 64 + lane;
            h.ok = i < p.cnt[3];
            beg = p.beg[3];
            list = p.list[3];
        } else if (unit < t4) {
            i = (unit - t3) / split * 64 + lane;
            h.ok = i < p.cnt[4];
            beg = p.beg[4];
            list = p.list[4];
        } else if (unit < total) {
            i = (unit - t4) * 64 + lane;
            h.ok = i < p.cnt[5];
            beg = p.beg[5];
            list = p.list[5];
        }
        if (h.ok) {
            h.u = list ? list[i] : beg + i;
            h.cur = dist[h.u];
            h.b = g.rbeg(h.u);
            h.e = g.rend(h.u);
        }
        return h;
    };
    int unit = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    RowHead<OffT> h = head(unit);
    while (unit < total) {
        const RowHead<OffT> nx = head(unit + stride);
        if (unit < t0)
            sorted_block<JOB, 64, true>(h, unit % kHeavySplit, kHeavySplit, ct, g, sv, dist, wbm,
                                        s);
        else if (unit < t2)
            sorted_block<JOB, 64, false>(h, (unit - t0) % kHeavySplit, kHeavySplit, ct, g, sv,
                                         dist, wbm, s);
        else if (unit < t3)
            sorted_block<JOB, 16, false>(h, (unit - t2) % (4 * split), 4 * split, ct, g, sv, dist,
                                         wbm, s);
        else if (unit < t4)
            sorted_block<JOB, 4, false>(h, (unit - t3) % split, split, ct, g, sv, dist, wbm, s);
        else
            sorted_block<JOB, 1, false>(h, 0, 1, ct, g, sv, dist, wbm, s);
        unit += stride;
        h = nx;
    }
}

// Promotion from the far bitmap: the far vertices in the new bucket [base, thresh)
// become the frontier (bits of `wbm`, compacted into its queues by the launch
// after), and those below it leave the bitmap, since they were lowered into an
// earlier bucket meanwhile and relaxed there.  A thread owns one word of both
// bitmaps.
template <typename OffT>
__device__ __forceinline__ void promote_far(const RowBounds &ct, const GraphView<OffT> &g,
                                            const int32_t *dist, uint32_t *far, int32_t words,
                                            uint32_t *wbm, RowSums &s) {
    for (int w = blockIdx.x * kBlock + threadIdx.x; w < words; w += gridDim.x * kBlock) {
        const uint32_t word = far[w];
        uint32_t gone = 0, now = 0;
        for (uint32_t x = word; x; x &= x - 1) {
            const int b = __ffs(x) - 1;
            const int32_t v = w * 32 + b;
            const int32_t d = dist[v];
            if (d >= ct.thresh) {
                s.left++;
                s.lowest = min(s.lowest, d);
                continue;
            }
            gone |= 1u << b;
            if (d < ct.base) continue;
            now |= 1u << b;
            s.cnt++;
            s.edges += (unsigned long long)(g.rend(v) - g.rbeg(v));
        }
        if (gone) far[w] = word & ~gone;
        if (now) wbm[w] = now;  // cleared by the launch before; no other writer
    }
}

// Promotion by a scan: the vertices in [base, thresh) become the frontier, and
// with `far` (or nullptr) those above it its bitmap.  A wavefront owns two words
// of the bitmaps.
template <typename OffT>
__device__ __forceinline__ void promote_scan(const RowBounds &ct, const GraphView<OffT> &g,
                                             const int32_t *dist, uint32_t *far, uint32_t *wbm,
                                             RowSums &s) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i0 = (int64_t)blockIdx.x * kBlock; i0 < g.n; i0 += stride) {
        const int64_t i = i0 + threadIdx.x;
        const bool in = i < g.n;
        const int32_t u = (int32_t)(in ? i : 0);
        const int32_t d = in ? dist[u] : HC_INF_DIST;
        const bool hit = in && d >= ct.base && d < ct.thresh;
        const bool later = d >= ct.thresh && d < HC_INF_DIST;
        const uint64_t m = __ballot(hit);
        if (hit) {
            s.cnt++;
            s.edges += (unsigned long long)(g.rend(u) - g.rbeg(u));
        } else if (later) {
            s.left++;
            s.lowest = min(s.lowest, d);
        }
        if (far) {
            const uint64_t f = __ballot(later);
            if (in && lane_id() == 0) far[u >> 5] = uint32_t(f);
            if (in && lane_id() == 32) far[u >> 5] = uint32_t(f >> 32);
        }
        // (the epoch before cleared the bitmap)
        if (lane_id() == 0 && uint32_t(m)) wbm[u >> 5] = uint32_t(m);
        if (lane_id() == 32 && uint32_t(m >> 32)) wbm[u >> 5] = uint32_t(m >> 32);
    }
}

// ---------------------------------------------------------------------------
// Kernels of the device-driven loop
// ---------------------------------------------------------------------------

// `nstage` hub distances are staged in dynamic LDS for pull epochs; push
// epochs stage up to `push_cap` output entries there.  D16: pull
// gathers read the 16-bit mirror `d16` instead.
template <typename OffT, bool D16, bool CB>
__global__ __launch_bounds__(kBlock) void sssp_step_kernel(
    PlanDev p, GraphView<OffT> g, int32_t *__restrict__ dist, uint16_t *d16, FrontierBufs fb,
    StepCtl *ctl, int32_t nstage, int32_t push_cap, int defer_dedup, PlanDev pcb,
    GraphView<OffT> cbv, int cbk) {
    extern __shared__ int32_t s_stage[];
    if (ctl->done) return;
    const int mode = ctl->mode;
    const int k = ctl->epoch;
    const int cur = k & 1, nxt = cur ^ 1;  // queue parities
    // Bitmaps: changed in epoch k-1 (read), changed in epoch k (written),
    // and the one to clear for epoch k+1.
    const uint32_t *rbm = fb.bm[k % 3];
    uint32_t *wbm = fb.bm[(k + 1) % 3];
    uint32_t *cbm = fb.bm[(k + 2) % 3];
    for (int w = blockIdx.x * kBlock + threadIdx.x; w < fb.words; w += gridDim.x * kBlock)
        cbm[w] = 0;
    uint32_t cnt = 0, gathered = 0;
    unsigned long long eacc = 0;
    if (mode == kPull && CB) {
        // Column-blocked sweep (the host picks it only when filtering is
        // not forced; its sweeps gather every neighbour):
        // the heavy rows of pcb block by block, then the light rows of plan
        // p once over the plain CSR (heavy rows first, as in the plain
        // sweep's class order, so light rows read their neighbours' values
        // of this epoch).
        if (D16) {
            const Dist16Reader rd{d16, dist};
            sssp_pull_sweep_cb(pcb, g, cbv, cbk, rd, dist, d16, wbm, cnt, eacc, gathered);
            sssp_pull_sweep<true, false>(p, g, rd, unstaged(rbm), dist, d16, wbm, cnt, eacc,
                                         gathered);
        } else {
            const Staged<int32_t> rd = stage(dist, nstage, s_stage);
            sssp_pull_sweep_cb(pcb, g, cbv, cbk, rd, dist, nullptr, wbm, cnt, eacc, gathered);
            sssp_pull_sweep<true, false>(p, g, rd, unstaged(rbm), dist, nullptr, wbm, cnt, eacc,
                                         gathered);
        }
    } else if (mode == kPull) {
        // One gather path per instantiation: both in one kernel would make
        // it hold the registers of both (and spill).
        if (D16) {
            const Dist16Reader rd{d16, dist};
            if (ctl->filter)
                sssp_pull_sweep<true, true>(p, g, rd, unstaged(rbm), dist, d16, wbm, cnt, eacc,
                                            gathered);
            else
                sssp_pull_sweep<true, false>(p, g, rd, unstaged(rbm), dist, d16, wbm, cnt, eacc,
                                             gathered);
        } else {
            const Staged<int32_t> rd = stage(dist, nstage, s_stage);
            if (ctl->filter)
                sssp_pull_sweep<true, true>(p, g, rd, unstaged(rbm), dist, nullptr, wbm, cnt,
                                            eacc, gathered);
            else
                sssp_pull_sweep<true, false>(p, g, rd, unstaged(rbm), dist, nullptr, wbm, cnt,
                                             eacc, gathered);
        }
    } else {
        // Output staged in the dynamic LDS (unused by push epochs).
        __shared__ uint32_t s_out;
        if (threadIdx.x == 0) s_out = 0;
        __syncthreads();
        const PushOut out{s_stage, &s_out, (uint32_t)push_cap, defer_dedup ? wbm : nullptr};
        int32_t lowest = HC_INF_DIST;
        uint32_t nfar = 0, pairs = 0;
        sssp_push_sweep(g, CsrEdges<OffT>{g.adj, g.wt}, dist, fb, ctl, out, cur, nxt, wbm, cnt,
                        eacc, lowest, nfar, pairs, gathered);
        const PushKept k = push_out_flush(out, g, fb, ctl, nxt);
        cnt += k.n;
        eacc += k.e;
    }
    write_partials(fb.part, cnt, eacc, gathered);
}

// `left` and `lowest` of a workgroup, cleared by thread 0 before a barrier.
struct RowSumsLds {
    uint32_t left;
    int32_t lowest;
    __device__ __forceinline__ void clear() {
        left = 0;
        lowest = HC_INF_DIST;
    }
};

__device__ __forceinline__ void write_row_sums(const Partials &part, const RowSums &s,
                                               RowSumsLds &lds) {
    if (s.left) atomicAdd(&lds.left, s.left);
    if (s.lowest < HC_INF_DIST) atomicMin(&lds.lowest, s.lowest);
    __syncthreads();
    write_partials<true>(part, s.cnt, s.edges,
                         (unsigned long long)s.pairs << 32 | s.gathered, lds.left, 0,
                         (unsigned long long)(HC_INF_DIST - lds.lowest));
}

// The step of the buckets on the plain CSR: push and promotion epochs.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void sssp_near_far_kernel(GraphView<OffT> g,
                                                               int32_t *__restrict__ dist,
                                                               FrontierBufs fb, StepCtl *ctl,
                                                               int32_t push_cap,
                                                               int defer_dedup) {
    extern __shared__ int32_t s_stage[];
    __shared__ uint32_t s_out;
    __shared__ RowSumsLds s_sums;
    if (ctl->done) return;
    const int k = ctl->epoch;
    const int cur = k & 1, nxt = cur ^ 1;
    uint32_t *wbm = fb.bm[(k + 1) % 3];
    uint32_t *cbm = fb.bm[(k + 2) % 3];
    for (int w = blockIdx.x * kBlock + threadIdx.x; w < fb.words; w += gridDim.x * kBlock)
        cbm[w] = 0;
    if (threadIdx.x == 0) {
        s_out = 0;
        s_sums.clear();
    }
    __syncthreads();
    RowSums s;
    if (ctl->mode == kPromote) {
        const RowBounds rb{ctl->low, ctl->base, ctl->thresh};
        promote_far(rb, g, dist, fb.far, fb.words, wbm, s);
    } else {
        const PushOut out{s_stage, &s_out, (uint32_t)push_cap, defer_dedup ? wbm : nullptr};
        sssp_push_sweep(g, CsrEdges<OffT, true>{g.adj, g.wt}, dist, fb, ctl, out, cur, nxt, wbm,
                        s.cnt, s.edges, s.lowest, s.left, s.pairs, s.gathered);
        const PushKept kept = push_out_flush(out, g, fb, ctl, nxt);
        s.cnt += kept.n;
        s.edges += kept.e;
    }
    write_row_sums(fb.part, s, s_sums);
}

// The step on the weight-sorted adjacency (the default): pull epochs or, with
// buckets, settling sweeps look only at the edges that can lower a row (see
// sorted.hip), push epochs of heavy buckets only at those that land in the
// bucket.
// Kronecker 23: a pull epoch gathers 4-35 M distances instead of 259 M and
// takes 160-340 us instead of 1600, a source 1.36 ms instead of 5.15; what is
// left is the lines of the row heads and starts and, in the push that meets
// most of the graph, the atomics (27 G/s at any size and locality on this
// GPU, where random loads reach 65 G/s from 33 MB and 262 G/s from L2).
// Uniform 23: 4.06 ms a source instead of 10.6.
template <typename OffT, bool BUCKETS>
__global__ __launch_bounds__(kBlock) void sssp_sorted_step_kernel(
    PlanDev p, GraphView<OffT> g, SortedView sv, int32_t *__restrict__ dist, FrontierBufs fb,
    StepCtl *ctl, int32_t push_cap, int defer_dedup) {
    extern __shared__ int32_t s_stage[];
    __shared__ uint32_t s_out;
    __shared__ RowSumsLds s_sums;
    if (ctl->done) return;
    const int mode = ctl->mode;
    const int k = ctl->epoch;
    const int cur = k & 1, nxt = cur ^ 1;
    uint32_t *wbm = fb.bm[(k + 1) % 3];
    uint32_t *cbm = fb.bm[(k + 2) % 3];
    for (int w = blockIdx.x * kBlock + threadIdx.x; w < fb.words; w += gridDim.x * kBlock)
        cbm[w] = 0;
    if (threadIdx.x == 0) {
        s_out = 0;
        s_sums.clear();
    }
    __syncthreads();
    RowSums s;
    const RowBounds rb{ctl->low, ctl->base, ctl->thresh};
    if (mode == kPush && !(BUCKETS && ctl->settle)) {
        const PushOut out{s_stage, &s_out, (uint32_t)push_cap, defer_dedup ? wbm : nullptr};
        sssp_push_sweep(g, SortedEdges<OffT, BUCKETS>{sv}, dist, fb, ctl, out, cur, nxt, wbm, s.cnt,
                        s.edges, s.lowest, s.left, s.pairs, s.gathered);
        const PushKept kept = push_out_flush(out, g, fb, ctl, nxt);
        s.cnt += kept.n;
        s.edges += kept.e;
    } else if (!BUCKETS) {
        sorted_sweep<kRowPull>(p, rb, g, sv, dist, wbm, s);
    } else if (mode == kPush) {
        sorted_sweep<kRowScatter>(p, rb, g, sv, dist, wbm, s);
    } else if (ctl->settle == 3) {
        sorted_sweep<kRowBucket>(p, rb, g, sv, dist, wbm, s);
    } else if (ctl->settle == 1) {
        sorted_sweep<kRowSettle>(p, rb, g, sv, dist, wbm, s);
    } else if (ctl->far_on && ctl->settle == 0) {
        promote_far(rb, g, dist, fb.far, fb.words, wbm, s);
    } else {
        promote_scan(rb, g, dist, ctl->settle ? fb.far : nullptr, wbm, s);
    }
    write_row_sums(fb.part, s, s_sums);
}

// Next bucket: the vertices in [base, base + delta) at least.
__device__ __forceinline__ void next_bucket(StepCtl *c, int32_t base) {
    if (c->bucket_e > 0) {
        c->prev2_e = c->prev_e;
        c->prev_e = c->bucket_e;
    }
    c->base = base;
    c->thresh = (int32_t)min((long long)base + c->delta, (long long)HC_INF_DIST);
    c->bucket_e = 0;
}

// Epoch controller (one thread, on the header copy c), from the step sums
// of the epoch that ran.
__device__ void sssp_decide(StepCtl *c, StepCtl *trace,
                            const unsigned long long (&sums)[kSumSlots]) {
    const unsigned long long out_n = sums[0], out_e = sums[1], gathered = sums[2];
    const unsigned long long left = sums[3], pairs = sums[4];
    // Sorted sweeps: offsets and distance of every row, and the pairs and
    // distances read.
    const unsigned long long rows =
        (unsigned long long)c->sweep_bytes - 12ull * (unsigned long long)c->m;
    const unsigned long long looked = 8ull * pairs + 4ull * gathered;
    const int32_t lowest = HC_INF_DIST - (int32_t)sums[kMaxSlot];
    const int k = c->epoch;
    const int ran = c->mode;
    const int settled = c->settle;
    if (ran == kPromote && c->far_on && settled == 0) {
        // far bitmap words, plus dist[v] and a bitmap entry per far vertex
        c->alg_bytes += 4ull * (unsigned long long)((c->n + 31) / 32) + 8ull * (out_n + left);
        c->promotions++;
        c->far_live = (long long)left;
        trace_epoch(c, trace, k, ran, out_n, out_e, 0);
    } else if (ran == kPromote) {
        // dist per vertex; of a settling sweep also the offsets, and pairs and
        // distances read; a bit per frontier vertex
        c->alg_bytes += (settled == 1 || settled == 3 ? rows : 4ull * (unsigned long long)c->n) +
                        looked + 8ull * out_n;
        c->promotions++;
        c->far_live = (long long)left;
        trace_epoch(c, trace, k, ran, out_n, out_e, pairs);
    } else if (ran == kPush) {
        // offsets + dist[u] per frontier vertex (per row when settling); id +
        // weight + dist[v] per edge, in a heavy bucket as far as read; dist
        // write + bitmap/queue entry per improved vertex.
        const bool all = !c->sorted || c->delta == 0;
        c->alg_bytes += (settled ? rows : 12ull * c->in_n) + (all ? 12ull * c->in_e : looked) +
                        8ull * out_n;
        trace_epoch(c, trace, k, ran, out_n, out_e, all ? (unsigned long long)c->in_e : pairs);
        c->push_epochs++;
        c->far_live += (long long)left;  // far settings (may repeat a vertex)
    } else if (c->sorted) {
        c->alg_bytes += rows + looked + 8ull * out_n;
        c->pull_epochs++;
        trace_epoch(c, trace, k, ran, out_n, out_e, pairs);
    } else {
        // Offsets, ids and own distances always; weight + distance per
        // gathered edge; one bit per tested neighbour when filtering.
        c->alg_bytes += (unsigned long long)c->sweep_bytes - 8ull * (unsigned long long)c->m +
                        8ull * gathered + (c->filter ? (unsigned long long)c->m / 8 : 0ull) +
                        8ull * out_n;
        c->pull_epochs++;
        trace_epoch(c, trace, k, ran, out_n, out_e, (unsigned long long)c->m);
    }
    if ((ran == kPush && !settled) || settled == 3) c->bucket_e += c->in_e;
    c->epoch = k + 1;
    c->in_n = (long long)out_n;
    c->in_e = (long long)out_e;
    // The changed set of this epoch is complete: the next pull may gather
    // only from it (knob 1: always; k >= 2: when it holds under n / k
    // vertices, so that most gathers are skipped).
    c->filter = c->filter_knob == 1 ||
                (c->filter_knob >= 2 && (long long)out_n * c->filter_knob < (long long)c->n);
    int next = ran;
    if (c->max_epochs > 0 && k + 1 >= c->max_epochs) {
        c->done = 1;
    } else if (c->delta > 0) {
        c->settle = 0;
        const long long light = kLightEdges + c->n / 8;
        if (out_n != 0) {
            // Heavy: past the limit, or about to be if it outgrows the bucket
            // before it as that one did the one before.
            if (c->sorted && (c->bucket_e + (long long)out_e > light ||
                              (ran == kPromote && (double)c->prev_e * (double)c->prev_e >
                                                      (double)light * (double)c->prev2_e)))
                c->far_on = 0;
            // The bucket goes on: by a sweep of the rows above its lowest
            // pending value while the frontier is heavy, else by a push.
            c->low = ran == kPromote && settled != 3 ? c->base : lowest;
            next = kPush;
            if (!c->far_on && c->direction != 2 && (long long)out_e > c->m / kBucketSweep) {
                c->settle = 3;
                next = kPromote;
            }
        } else if (c->far_on) {
            // The bucket is complete, or was empty: on to the next width, or
            // to the smallest far distance.
            c->done_e += c->bucket_e;
            if (c->far_live == 0) {
                c->done = 1;
            } else {
                next = kPromote;
                next_bucket(c, ran == kPromote ? lowest : c->thresh);
            }
        } else if ((ran == kPush && !settled) || settled == 3) {
            // The bucket is complete.  A sweep over the rows above it costs
            // a few edges of each, a push from its vertices most of theirs:
            // the sweep, once the bucket holds a fair share of the edges not
            // yet done (and always the push while most rows are unreached,
            // whose scans find no bound).
            const long long rest = c->m - c->done_e - c->bucket_e;
            c->done_e += c->bucket_e;
            c->low = c->base;
            if (c->direction != 2 && c->bucket_e * kSettleShare > rest) {
                c->settle = 1;
                next = kPromote;
                next_bucket(c, c->thresh);
            } else {
                c->settle = 2;
                next = kPush;
            }
        } else if (ran == kPush) {
            if (c->bucket_e < light / 4) {
                c->settle = 4;
                c->far_on = 1;
            }
            next = kPromote;
            next_bucket(c, c->thresh);
        } else if (left != 0) {
            // An empty bucket: on to the smallest distance above it.
            next = kPromote;
            next_bucket(c, lowest);
        } else {
            c->done = 1;
        }
    } else {
        c->low = lowest;
        if (out_n == 0) c->done = 1;
        else if (c->direction != 0) next = c->direction == 1 ? kPull : kPush;
        else next = (long long)out_e > c->m / c->alpha ? kPull : kPush;
    }
    c->need_compact = (!c->done && ran != kPush && next == kPush) ? 1 : 0;
    c->mode = next;
}

// Between epochs k and k + 1: the controller (every workgroup decides on its
// own copy; workgroup 0 records the epoch and stores header k + 1), then
// the frontier compaction when the loop turns to push and, with the 16-bit
// mirror, its rebuild before a pull epoch.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void sssp_between_kernel(GraphView<OffT> g, FrontierBufs fb,
                                                              StepCtl *cur, StepCtl *nxt,
                                                              StepCtl *trace, Partials next_set,
                                                              const int32_t *dist, uint16_t *d16) {
    __shared__ StepCtl s_c;  // header fields only
    unsigned long long sums[kSumSlots];
    if (!ctl_begin(&s_c, cur, fb.part, sums)) return;
    if (threadIdx.x == 0) sssp_decide(&s_c, blockIdx.x == 0 ? trace : nullptr, sums);
    __syncthreads();
    ctl_end(&s_c, cur, nxt, fb, next_set);
    compact_body(g, fb, &s_c, 1, dist, d16);
}

// Smallest initial distance seen by each workgroup, for sssp_init_kernel.
__global__ __launch_bounds__(kBlock) void sssp_init_low_kernel(const int32_t *__restrict__ init,
                                                               int32_t n, Partials part) {
    int32_t m = HC_INF_DIST;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
        m = min(m, init[i]);
    m = block_min(m);
    if (threadIdx.x == 0) part.acc[blockIdx.x] = (unsigned long long)(long long)m;
}

// Initialises distances, bitmaps and the control block for one run.
// init_dist == nullptr: single source `src`; otherwise copy init_dist and
// start in pull mode with an empty frontier (sssp_pull_gpu semantics).
template <typename OffT>
__global__ __launch_bounds__(kBlock) void sssp_init_kernel(
    GraphView<OffT> g, int32_t *__restrict__ dist,
    const int32_t *__restrict__ init_dist, FrontierBufs fb, StepCtl *ctl,
    int32_t src, int direction, int alpha, int max_epochs, long long m,
    long long sweep_bytes, int grid, int filter, int chunk, uint16_t *d16, int delta, int sorted,
    int low_parts) {
    const int stride = gridDim.x * kBlock;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < g.n; i += stride) {
        const int32_t d = init_dist ? init_dist[i] : (i == src ? 0 : HC_INF_DIST);
        dist[i] = d;
        if (d16) d16[i] = dist16(d);
    }
    for (int w = blockIdx.x * kBlock + threadIdx.x; w < fb.words; w += stride) {
        // Epoch 0 reads bitmap 0 as the set changed before it: the source.
        fb.bm[0][w] = (!init_dist && w == (src >> 5)) ? (1u << (src & 31)) : 0u;
        fb.bm[1][w] = 0;
        fb.bm[2][w] = 0;
        fb.far[w] = 0;
    }
    // Smallest initial distance (sssp_init_low_kernel's results lie in the
    // counter sets, one per workgroup of that launch).
    __shared__ int32_t s_low;
    if (blockIdx.x == 0) {
        if (threadIdx.x == 0) s_low = HC_INF_DIST;
        __syncthreads();
        for (int i = threadIdx.x; i < low_parts; i += kBlock)
            atomicMin(&s_low, (int32_t)(long long)fb.part.acc[i]);
        __syncthreads();
        for (int j = 0; j < kSumSets; j++) clear_partials(sum_set(fb.part, j));
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl->sorted = sorted;
        // Every candidate of epoch 0 comes from the source, or from an
        // initial distance; where one of those is negative (relax() reads
        // it as unsigned) no edge is left out.
        ctl->low = !init_dist ? 0 : (s_low < 0 ? -HC_INF_DIST - 1 : s_low);
        // With initial distances the changed set before epoch 0 is unknown:
        // that epoch gathers every neighbour.
        ctl->filter_knob = filter;
        ctl->filter = init_dist ? 0 : (filter == 1 || (filter >= 2 && filter < g.n));
        for (int p = 0; p < 2; p++)
            for (int j = 0; j < 5; j++) fb.cnt[p][j] = 0;
        ctl->done = 0;
        ctl->epoch = 0;
        ctl->steps = 0;
        ctl->stage = 0;
        ctl->max_epochs = max_epochs;
        ctl->direction = direction;
        ctl->alpha = alpha;
        ctl->need_compact = 0;
        ctl->chunk = chunk;
        ctl->mid = kPushMid;
        ctl->n = g.n;
        ctl->grid = grid;
        ctl->m = m;
        ctl->sweep_bytes = sweep_bytes;
        ctl->push_epochs = ctl->pull_epochs = 0;
        ctl->delta = delta;
        ctl->base = 0;
        ctl->thresh = delta > 0 ? delta : HC_INF_DIST;
        ctl->settle = 0;
        ctl->promotions = 0;
        ctl->bucket_e = 0;
        ctl->done_e = 0;
        ctl->prev_e = ctl->prev2_e = m;
        ctl->far_on = delta > 0;
        ctl->far_live = 0;
        ctl->reached = 0;
        ctl->alg_bytes = 0;
        ctl->t_start = wall_clock64();
        ctl->t_end = ctl->t_start;
        if (init_dist) {
            ctl->mode = kPull;
            ctl->in_n = g.n;
            ctl->in_e = m;
        } else {
            OffT b = g.rbeg(src), e = g.rend(src);
            int64_t d = int64_t(e - b);
            int cls = degree_class(d, kPushMid);
            if (cls == 3) {  // chunk descriptors: written by workgroup 0 below
                fb.cnt[0][3] = (uint32_t)((d + chunk - 1) / chunk);
                fb.cnt[0][4] = 1;
            } else {
                fb.q[0][cls][0] = src;
                fb.cnt[0][cls] = 1;
            }
            ctl->in_n = 1;
            ctl->in_e = d;
            ctl->mode = direction == 1 ? kPull
                        : (direction == 2 || delta > 0) ? kPush
                        : (d > m / alpha ? kPull : kPush);
        }
    }
    if (blockIdx.x == 0 && !init_dist) write_source_chunks(g, fb, src, chunk);
}

template <typename OffT>
__global__ void sssp_pull_thread_kernel(GraphView<OffT> g,
                                        int32_t *__restrict__ dist,
                                        int32_t start, int32_t end,
                                        int32_t *updated) {
    uint32_t upd = 0;
    const int32_t stride = gridDim.x * blockDim.x;
    for (int32_t u = start + blockIdx.x * blockDim.x + threadIdx.x; u < end;
         u += stride) {
        uint32_t gathered = 0;
        int32_t m = row_min<1, false>(g, unstaged(dist), unstaged<uint32_t>(nullptr), g.rbeg(u),
                                      g.rend(u), 0, gathered);
        if (m < dist[u]) {
            dist[u] = m;
            upd++;
        }
    }
    for (int s = 32; s > 0; s >>= 1) upd += __shfl_xor(upd, s, 64);
    if (lane_id() == 0 && upd) atomicAdd(updated, (int32_t)upd);
}

template <typename OffT>
__global__ void sssp_pull_wave_kernel(GraphView<OffT> g,
                                      int32_t *__restrict__ dist,
                                      int32_t start, int32_t end,
                                      int32_t *updated) {
    uint32_t upd = 0;
    const int32_t waves = gridDim.x * (blockDim.x / kWave);
    const int32_t wid = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    for (int32_t u = start + wid; u < end; u += waves) {
        uint32_t gathered = 0;
        int32_t m = group_min<64>(row_min<64, false>(g, unstaged(dist), unstaged<uint32_t>(nullptr),
                                                     g.rbeg(u), g.rend(u), lane_id(), gathered));
        if (lane_id() == 0 && m < dist[u]) {
            dist[u] = m;
            upd++;
        }
    }
    if (lane_id() == 0 && upd) atomicAdd(updated, (int32_t)upd);
}

template <typename OffT>
__global__ void sssp_pull_block_kernel(GraphView<OffT> g,
                                       int32_t *__restrict__ dist,
                                       int32_t start, int32_t end,
                                       int32_t *updated) {
    uint32_t upd = 0;
    for (int32_t u = start + blockIdx.x; u < end; u += gridDim.x) {
        const OffT b = g.rbeg(u), e = g.rend(u);
        int32_t m = HC_INF_DIST;
        for (OffT i = b + threadIdx.x; i < e; i += blockDim.x)
            m = min(m, relax(dist[g.adj[i]], g.wt[i]));
        m = block_min(m);
        if (threadIdx.x == 0 && m < dist[u]) {
            dist[u] = m;
            upd++;
        }
    }
    if (threadIdx.x == 0 && upd) atomicAdd(updated, (int32_t)upd);
}

template <typename OffT>
__global__ __launch_bounds__(kBlock) void sssp_pull_fused_kernel(
    PlanDev p, GraphView<OffT> g, int32_t *__restrict__ dist,
    int32_t *updated, int32_t nstage) {
    extern __shared__ int32_t s_stage[];
    uint32_t upd = 0;
    unsigned long long eacc = 0;
    uint32_t gathered = 0;
    sssp_pull_sweep<false, false>(p, g, stage(dist, nstage, s_stage), unstaged<uint32_t>(nullptr),
                                  dist, nullptr, nullptr, upd, eacc, gathered);
    unsigned long long s = block_sum_u64(upd);
    if (threadIdx.x == 0 && s) atomicAdd(updated, (int32_t)s);
}

// Epoch API sweep over the column blocks of a whole graph; `seen` (n bits,
// zeroed by the host) counts each lowered row once.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void sssp_pull_cb_kernel(
    PlanDev plight, PlanDev pcb, GraphView<OffT> g, GraphView<OffT> cbv, int cbk,
    int32_t *__restrict__ dist, int32_t *updated, uint32_t *seen) {
    uint32_t upd = 0, gathered = 0;
    unsigned long long eacc = 0;
    sssp_pull_sweep_cb(pcb, g, cbv, cbk, unstaged(dist), dist, nullptr, seen, upd, eacc,
                       gathered);
    sssp_pull_sweep<false, false>(plight, g, unstaged(dist), unstaged<uint32_t>(nullptr), dist,
                                  nullptr, nullptr, upd, eacc, gathered);
    unsigned long long s = block_sum_u64(upd);
    if (threadIdx.x == 0 && s) atomicAdd(updated, (int32_t)s);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------


// Share of all edges held by the 1% highest-degree rows (cached; the caller
// holds g->mu).  Skewed graphs (Kronecker: about half) and flat ones
// (uniform: about 1%) want different push/pull switch points: a push epoch
// on a flat graph relaxes edges whose targets are spread over the whole
// distance array, so its atomics cost far more per edge.
static double hub_share(hc_graph_s *g) {
    if (g->hub_share >= 0.0) return g->hub_share;
    const int32_t rows = g->rows;
    if (rows <= 0 || g->m <= 0) return g->hub_share = 0.0;
    const int32_t k = std::max<int32_t>(1, rows / 100);
    int64_t top = 0;
    if (g->sorted) {
        top = g->h_off[k] - g->h_off[0];
    } else {
        std::vector<int64_t> deg(rows);
        for (int32_t i = 0; i < rows; i++) deg[i] = g->h_off[i + 1] - g->h_off[i];
        std::nth_element(deg.begin(), deg.begin() + (k - 1), deg.end(), std::greater<int64_t>());
        for (int32_t i = 0; i < k; i++) top += deg[i];
    }
    return g->hub_share = double(top) / double(g->m);
}

bool flat_graph(hc_graph_s *g) { return hub_share(g) < 0.05; }

struct SsspWs {
    FrontierWs f;
    uint16_t *d16 = nullptr;  // 16-bit distance mirror, allocated on first use
};

void free_sssp_ws(hc_graph_s *g) {
    if (!g->ws_sssp) return;
    auto *ws = static_cast<SsspWs *>(g->ws_sssp);
    frontier_ws_free(&ws->f);
    if (ws->d16) hipFree(ws->d16);
    delete ws;
    g->ws_sssp = nullptr;
}

static int get_sssp_ws(hc_graph_s *g, SsspWs **out) {
    // The partial slots are sized for the launch grid; re-allocate when the
    // tuned grid changes.
    if (g->ws_sssp && static_cast<SsspWs *>(g->ws_sssp)->f.grid != grid_blocks()) free_sssp_ws(g);
    if (!g->ws_sssp) {
        auto *ws = new SsspWs();
        int rc = frontier_ws_alloc(g, &ws->f);
        if (rc != HC_OK) {
            delete ws;
            return rc;
        }
        g->ws_sssp = ws;
    }
    *out = static_cast<SsspWs *>(g->ws_sssp);
    return HC_OK;
}

// Bytes a bucketed pull sweep reads and writes per the algorithm: row
// offsets, neighbour id + weight + gathered distance per edge, own distance.
long long sssp_sweep_bytes(const hc_graph_s *g, const PlanHost *ph) {
    const PlanDev &p = ph->dev;
    long long rows = 0;
    for (int c = 1; c < kNumClasses; c++) rows += p.cnt[c];
    rows += p.num_hubs;
    const long long ob = g->off64 ? 8 : 4;
    return ob * (rows + 1) + 12ll * g->m + 4ll * rows;
}

template <typename OffT>
static int launch_pull_epoch(hc_graph_s *g, int mapping, int32_t start,
                             int32_t end, int32_t *dist, int32_t *updated,
                             int blocks, int threads, hipStream_t s) {
    GraphView<OffT> v = view<OffT>(g);
    switch (mapping) {
        case HC_MAP_THREAD:
            if (!threads) threads = 256;
            if (!blocks) blocks = std::max(1, std::min(grid_blocks(), (end - start + threads - 1) / threads));
            sssp_pull_thread_kernel<OffT><<<blocks, threads, 0, s>>>(v, dist, start, end, updated);
            break;
        case HC_MAP_WAVE:
            if (!threads) threads = 256;
            if (!blocks) blocks = grid_blocks();
            sssp_pull_wave_kernel<OffT><<<blocks, threads, 0, s>>>(v, dist, start, end, updated);
            break;
        case HC_MAP_BLOCK:
            if (!threads) threads = 256;
            if (!blocks) blocks = grid_blocks();
            sssp_pull_block_kernel<OffT><<<blocks, threads, 0, s>>>(v, dist, start, end, updated);
            break;
        default: {
            const PlanHost *ph = nullptr;
            // A whole-graph sweep gathers column block by column block.
            const ColBlocks *cb = nullptr;
            if (start == 0 && end == g->n) HC_TRY(get_col_blocks(g, col_shift_for(g, flat_graph(g)), s, &cb));
            if (cb) {
                const PlanHost *pl = nullptr;
                HC_TRY(get_plan(g, 0, g->n, cb_plan_config(cb->K), &ph));
                HC_TRY(get_plan(g, 0, g->n, cb_light_config(cb->K), &pl));
                const int units = ph->total_units * cb->K + pl->total_units;
                if (units == 0) return HC_OK;
                GraphView<OffT> cbv{static_cast<const OffT *>(cb->off), cb->adj, cb->wt, 0, g->n};
                HC_HIP(hipMemsetAsync(cb->seen, 0, sizeof(uint32_t) * ((g->n + 31) / 32), s));
                const int nb = std::max(1, std::min(units, grid_blocks()));
                sssp_pull_cb_kernel<OffT><<<nb, kBlock, 0, s>>>(pl->dev, ph->dev, v, cbv, cb->K,
                                                                dist, updated, cb->seen);
                break;
            }
            HC_TRY(get_plan(g, start, end, sssp_plan_config(), &ph));
            if (ph->total_units == 0) return HC_OK;
            int nb = std::max(1, std::min(ph->total_units, grid_blocks()));
            const int32_t ns = std::min<int32_t>(tuning().sssp_stage, g->n);
            sssp_pull_fused_kernel<OffT><<<nb, kBlock, ns * sizeof(int32_t), s>>>(
                ph->dev, v, dist, updated, ns);
        }
    }
    HC_HIP(hipGetLastError());
    return HC_OK;
}

static int check_launch(int mapping, int blocks, int threads) {
    HC_CHECK_ARG(mapping >= HC_MAP_THREAD && mapping <= HC_MAP_BUCKETED,
                 "unknown mapping %d", mapping);
    HC_CHECK_ARG(blocks >= 0 && threads >= 0, "negative launch shape");
    HC_CHECK_ARG(threads <= 1024, "threads must be <= 1024");
    if (mapping == HC_MAP_WAVE || mapping == HC_MAP_BLOCK)
        HC_CHECK_ARG(threads % kWave == 0,
                     "thread count must be a multiple of 64 for this mapping");
    return HC_OK;
}


template <typename OffT>
struct SsspLaunch {
    PlanDev plan;
    GraphView<OffT> g;
    int32_t *dist;
    uint16_t *d16;  // 16-bit distance mirror (sssp.dist16), or nullptr
    FrontierBufs fb;
    StepCtl *ctl;
    int grid;
    hipStream_t s;
    int32_t nstage;
    int32_t lds_entries;
    int32_t push_cap;
    int defer_dedup;
    KernelTimer *kt;
    PlanDev cbplan;          // column-blocked pull sweeps (cbk > 0)
    GraphView<OffT> cbv;
    int cbk;
    SortedView sv;           // weight-sorted adjacency (e: not nullptr)
    bool buckets;
    template <bool D16, bool CB>
    void step(FrontierBufs fb, StepCtl *cur) {
        timed_launch(kt, sssp_step_kernel<OffT, D16, CB>, dim3(grid), dim3(kBlock),
                     uint32_t(lds_entries * sizeof(int32_t)), s, plan, g, dist, d16, fb, cur,
                     nstage, push_cap, defer_dedup, cbplan, cbv, cbk);
    }
    template <bool BUCKETS>
    void sorted_step(FrontierBufs fb, StepCtl *cur) {
        timed_launch(kt, sssp_sorted_step_kernel<OffT, BUCKETS>, dim3(grid), dim3(kBlock),
                     uint32_t(lds_entries * sizeof(int32_t)), s, plan, g, sv, dist, fb, cur,
                     push_cap, defer_dedup);
    }
    // Epoch k: header slot k & 1, counter set k % 3.
    static int launch(void *arg, long long k) {
        auto *a = static_cast<SsspLaunch *>(arg);
        FrontierBufs fb = a->fb;
        fb.part = sum_set(a->fb.part, k);
        StepCtl *cur = a->ctl + (k & 1), *nxt = a->ctl + ((k + 1) & 1);
        if (a->sv.e) {
            if (a->buckets) a->template sorted_step<true>(fb, cur);
            else a->template sorted_step<false>(fb, cur);
        } else if (a->buckets) {
            timed_launch(a->kt, sssp_near_far_kernel<OffT>, dim3(a->grid), dim3(kBlock),
                         uint32_t(a->lds_entries * sizeof(int32_t)), a->s, a->g, a->dist, fb, cur,
                         a->push_cap, a->defer_dedup);
        } else if (a->d16) {
            if (a->cbk) a->template step<true, true>(fb, cur);
            else a->template step<true, false>(fb, cur);
        } else {
            if (a->cbk) a->template step<false, true>(fb, cur);
            else a->template step<false, false>(fb, cur);
        }
        sssp_between_kernel<OffT><<<compact_grid(a->grid), kBlock, 0, a->s>>>(
            a->g, fb, cur, nxt, a->ctl, sum_set(a->fb.part, k + 1), a->dist, a->d16);
        if (hipGetLastError() != hipSuccess) return fail(HC_ERR_HIP, "SSSP epoch launch failed");
        return HC_OK;
    }
};


// Bucket width of the single-source loop (knob sssp.delta).  Sorted adjacency: 4 x
// the sampled largest weight / mean degree on flat graphs (uniform 23, weights
// 1..255, degree 32: widths 24 / 32 / 48 / 64 / 96 4.41 / 4.06 / 4.41 / 4.56 / 4.70
// ms), off on skewed ones, whose pull sweeps win (Kronecker 23: 1.36 ms
// against 2.4 / 1.8 ms with widths 32 / 96).
// Plain CSR: 2 x, on flat graphs of at least kNearFarMinEdges edges.  Buckets
// save re-relaxations and cost epochs, so the line is where an epoch's work
// outweighs its launches (plain loop against buckets; uniform graphs, 65 K
// vertices, 2.1 M edges: 0.56 / 0.99 ms; 256 K, 7.9 M: 1.01 / 1.34; 4 M, 16.8 M:
// 2.24 / 2.39; 1 M, 33.6 M: 2.28 / 2.15; 16 M, 67 M: 8.79 / 5.86; 8 M, 268 M:
// 20.7 / 9.75; grids of 4.2 M, 16.8 M and 67 M edges: 26 / 55, 114 / 147, 579 /
// 344).
constexpr int64_t kNearFarMinEdges = int64_t(1) << 24;
static int sssp_delta(hc_graph_s *g, bool sorted) {
    const int d = tuning().sssp_delta;
    if (d >= 0) return d;
    if (!g->weighted || g->m == 0 || g->max_weight <= 0 || !flat_graph(g)) return 0;
    if (!sorted && g->m < kNearFarMinEdges) return 0;
    const double mean_deg = (double)g->m / std::max(1, g->rows);
    return (int)std::max(1.0, std::ceil((sorted ? 4.0 : 2.0) * g->max_weight / mean_deg));
}

template <typename OffT>
static int run_sssp_loop(hc_graph_s *g, int32_t src, const int32_t *init_dist,
                         int32_t *dist, int direction, int alpha,
                         int max_epochs, hc_run_stats_t *stats, hipStream_t s) {
    SsspWs *ws = nullptr;
    HC_TRY(get_sssp_ws(g, &ws));
    GraphView<OffT> v = view<OffT>(g);
    // The weight-sorted adjacency (buckets set by a knob need it on any graph),
    // unless a knob asks for one of the plain sweeps' variants or there is no
    // memory for the copy.
    const Tuning &t = tuning();
    SortedView sv{nullptr, 0};
    const bool want = t.sssp_sorted == 2 ||
                      (t.sssp_sorted == 1 && (g->m >= kSortedMinEdges || t.sssp_delta > 0));
    if (want && t.sssp_filter == 0 && t.sssp_dist16 != 1 && t.pull_col_shift <= 0)
        HC_TRY(get_sorted(g, s, &sv));
    const bool sorted = sv.e != nullptr;
    const PlanHost *ph = nullptr;
    HC_TRY(get_plan(g, 0, g->n, sorted ? sorted_plan_config() : sssp_plan_config(), &ph));
    // A pruned pull costs little more than its row heads: pull early
    // (Kronecker 23: alpha 4 / 8 / 16 / 32 1.72 / 1.39 / 1.36 / 1.35 ms).
    if (alpha <= 0) alpha = t.sssp_alpha > 0 ? t.sssp_alpha : (sorted ? 16 : flat_graph(g) ? 2 : 4);
    // Buckets (sssp.delta): no pulls on the CSR.
    const int delta = init_dist || direction == 1 ? 0 : sssp_delta(g, sorted);
    uint16_t *d16 = nullptr;
    if (!sorted && delta == 0 && (t.sssp_dist16 == 1 || (t.sssp_dist16 == 2 && flat_graph(g)))) {
        if (!ws->d16 && hipMalloc(&ws->d16, sizeof(uint16_t) * std::max(g->n, 1)) != hipSuccess)
            return fail(HC_ERR_OOM, "16-bit distance mirror allocation failed");
        d16 = ws->d16;
    }
    const long long sweep = sssp_sweep_bytes(g, ph);
    const int32_t nstage = std::min<int32_t>(tuning().sssp_stage, g->n);
    const int32_t push_cap = tuning().push_stage;
    const int32_t lds_entries = std::max<int32_t>(nstage, push_cap);
    // Pull epochs gather column block by column block (not with filtering,
    // which tests a changed bit per neighbour before its gather).
    const ColBlocks *cb = nullptr;
    const PlanHost *phb = nullptr;
    // A loop that pulls only its few heavy epochs gains nothing from the blocks of
    // a small graph, and the first query would build them (uniform, 2M vertices,
    // 8.4 M edges, weights 1..3: 1.01 ms a query either way, the first 2.37 ms
    // with and 2.07 without).
    const bool blocks = t.pull_col_shift > 0 || init_dist || direction == 1 ||
                        g->m >= kSortedMinEdges;
    if (!sorted && delta == 0 && direction != 2 && tuning().sssp_filter != 1 && blocks) {
        HC_TRY(get_col_blocks(g, col_shift_for(g, flat_graph(g)), s, &cb));
        if (cb) {
            // Plain sweep for the light rows only.
            HC_TRY(get_plan(g, 0, g->n, cb_light_config(cb->K), &ph));
            HC_TRY(get_plan(g, 0, g->n, cb_plan_config(cb->K), &phb));
        }
    }
    const void *step_fn =
        sorted ? (delta > 0 ? reinterpret_cast<const void *>(&sssp_sorted_step_kernel<OffT, true>)
                            : reinterpret_cast<const void *>(&sssp_sorted_step_kernel<OffT, false>))
        : delta > 0 ? reinterpret_cast<const void *>(&sssp_near_far_kernel<OffT>)
        : d16 ? (cb ? reinterpret_cast<const void *>(&sssp_step_kernel<OffT, true, true>)
                  : reinterpret_cast<const void *>(&sssp_step_kernel<OffT, true, false>))
            : (cb ? reinterpret_cast<const void *>(&sssp_step_kernel<OffT, false, true>)
                  : reinterpret_cast<const void *>(&sssp_step_kernel<OffT, false, false>));
    const int grid = resident_grid(step_fn,
                                   kBlock, lds_entries * sizeof(int32_t),
                                   std::min(ws->f.grid, grid_blocks(tuning().sssp_grid_per_cu)));
    const int init_grid = std::max(1, std::min(grid, (g->n + kBlock - 1) / kBlock));
    const int low_parts = init_dist && sorted ? std::min(init_grid, kSumWords * kSumSets) : 0;
    if (low_parts)
        sssp_init_low_kernel<<<low_parts, kBlock, 0, s>>>(init_dist, g->n, ws->f.fb.part);
    sssp_init_kernel<OffT><<<init_grid, kBlock, 0, s>>>(
        v, dist, init_dist, ws->f.fb, ws->f.ctl, src, direction, alpha,
        max_epochs, (long long)g->m, sweep, grid, tuning().sssp_filter, tuning().push_chunk, d16,
        delta, sorted ? 1 : 0, low_parts);
    HC_HIP(hipGetLastError());
    ws->f.kt.reset();
    // Push epochs deduplicate improved vertices when staging them (flat
    // graphs: few repeats) or on the spot (skewed graphs: hubs' neighbours
    // are lowered by many edges, and repeats would fill the staging).
    const int defer_dedup = tuning().sssp_push_dedup == 2 ? (flat_graph(g) ? 1 : 0)
                                                          : tuning().sssp_push_dedup;
    SsspLaunch<OffT> L{ph->dev, v, dist, d16, ws->f.fb, ws->f.ctl, grid, s, nstage, lds_entries,
                       push_cap, defer_dedup, &ws->f.kt, phb ? phb->dev : PlanDev{},
                       cb ? GraphView<OffT>{static_cast<const OffT *>(cb->off), cb->adj, cb->wt,
                                            0, g->n}
                          : GraphView<OffT>{},
                       cb ? cb->K : 0, sv, delta > 0};
    // Bellman-Ford needs at most n epochs (buckets add promotion epochs and
    // re-pushes: a generous bound); the cap bounds a faulty loop.
    const long long bound = delta > 0 ? 64LL * (g->n + 1) + 4096 : (long long)g->n;
    const long long cap = (max_epochs > 0 ? std::min<long long>(max_epochs, bound) : bound) + 2;
    long long launches = 0;
    StepCtl fc;
    HC_TRY(run_epoch_loop(&ws->f, s, cap, &SsspLaunch<OffT>::launch, &L, &launches, &fc));
    if (!fc.done && max_epochs <= 0)
        return fail(HC_ERR_HIP, "SSSP loop did not converge in %lld epochs", launches);
    if (stats) {
        std::memset(stats, 0, sizeof(*stats));
        // Device wall clock from the init kernel to the controller of the
        // last epoch (launches queued past it are not part of the loop).
        stats->ms = double(fc.t_end - fc.t_start) / device_state().clock_khz;
        stats->epochs = fc.epoch;
        stats->push_epochs = fc.push_epochs;
        stats->pull_epochs = fc.pull_epochs;
        stats->launches = (int32_t)(2 * launches);
        stats->reached = -1;
        stats->alg_bytes = (double)fc.alg_bytes;
        if (ws->f.kt.on) {
            stats->kernel_launches = (int32_t)std::min<long long>(fc.steps, ws->f.kt.pairs());
            stats->kernel_ms = ws->f.kt.sum_ms(stats->kernel_launches);
        }
    }
    return HC_OK;
}

}  // namespace hc

using namespace hc;

extern "C" {

int hc_sssp_pull_epoch(hc_graph_t g, int mapping, int32_t start_id,
                       int32_t end_id, int32_t *dist, int32_t *updated,
                       int blocks, int threads, hc_stream_t stream) {
    HC_CHECK_ARG(g && dist && updated, "NULL argument");
    HC_CHECK_ARG(g->weighted, "SSSP needs a weighted graph");
    HC_CHECK_ARG(g->row0 <= start_id && start_id <= end_id &&
                     end_id <= g->row0 + g->rows,
                 "range [%d,%d) outside the rows held [%d,%d)", start_id,
                 end_id, g->row0, g->row0 + g->rows);
    HC_TRY(check_launch(mapping, blocks, threads));
    HC_TRY(ensure_init());
    if (start_id == end_id) return HC_OK;
    GraphCall call(g);
    hipStream_t s = pick_stream(stream);
    return g->off64 ? launch_pull_epoch<uint64_t>(g, mapping, start_id, end_id, dist, updated, blocks, threads, s)
                    : launch_pull_epoch<uint32_t>(g, mapping, start_id, end_id, dist, updated, blocks, threads, s);
}

int hc_sssp(hc_graph_t g, int32_t source, int32_t *dist,
            const hc_sssp_opts_t *opts, hc_run_stats_t *stats,
            hc_stream_t stream) {
    HC_CHECK_ARG(g && dist, "NULL argument");
    HC_CHECK_ARG(g->weighted, "SSSP needs a weighted graph");
    HC_CHECK_ARG(g->row0 == 0 && g->rows == g->n,
                 "full runs need a whole-graph handle");
    HC_CHECK_ARG(source >= 0 && source < g->n, "source %d outside [0,%d)",
                 source, g->n);
    int direction = opts ? opts->direction : 0;
    int alpha = opts && opts->alpha > 0 ? opts->alpha : 0;  // 0: the loop's default
    int max_epochs = opts ? opts->max_epochs : 0;
    HC_CHECK_ARG(direction >= 0 && direction <= 2, "direction must be 0, 1 or 2");
    HC_TRY(ensure_init());
    GraphCall call(g);
    hipStream_t s = pick_stream(stream);
    return g->off64 ? run_sssp_loop<uint64_t>(g, source, nullptr, dist, direction, alpha, max_epochs, stats, s)
                    : run_sssp_loop<uint32_t>(g, source, nullptr, dist, direction, alpha, max_epochs, stats, s);
}

int hc_sssp_pull(hc_graph_t g, int mapping, const int32_t *init_dist,
                 int32_t *dist, int blocks, int threads,
                 hc_run_stats_t *stats, hc_stream_t stream) {
    HC_CHECK_ARG(g && init_dist && dist, "NULL argument");
    HC_CHECK_ARG(g->weighted, "SSSP needs a weighted graph");
    HC_CHECK_ARG(g->row0 == 0 && g->rows == g->n,
                 "full runs need a whole-graph handle");
    HC_TRY(check_launch(mapping, blocks, threads));
    HC_TRY(ensure_init());
    hipStream_t s = pick_stream(stream);
    if (mapping == HC_MAP_BUCKETED) {
        GraphCall call(g);
        return g->off64 ? run_sssp_loop<uint64_t>(g, 0, init_dist, dist, 1, 8, 0, stats, s)
                        : run_sssp_loop<uint32_t>(g, 0, init_dist, dist, 1, 8, 0, stats, s);
    }
    // Host-driven loop of sssp_pull_gpu (src/kernels/gpu/sssp.cuh:76-85):
    // zero the counter, run one epoch, read the counter back.
    int32_t *d_upd = nullptr;
    HC_HIP(hipMalloc(&d_upd, sizeof(int32_t)));
    int rc = HC_OK;
    hipEvent_t e0, e1;
    hipEventCreate(&e0);
    hipEventCreate(&e1);
    if (hipMemcpyAsync(dist, init_dist, sizeof(int32_t) * g->n,
                       hipMemcpyDeviceToDevice, s) != hipSuccess)
        rc = fail(HC_ERR_HIP, "copy of init_dist failed");
    int epochs = 0;
    hipEventRecord(e0, s);
    int32_t h_upd = 1;
    while (rc == HC_OK && h_upd != 0) {
        hipMemsetAsync(d_upd, 0, sizeof(int32_t), s);
        {
            GraphCall call(g);
            rc = g->off64 ? launch_pull_epoch<uint64_t>(g, mapping, 0, g->n, dist, d_upd, blocks, threads, s)
                          : launch_pull_epoch<uint32_t>(g, mapping, 0, g->n, dist, d_upd, blocks, threads, s);
        }
        if (rc != HC_OK) break;
        if (hipMemcpyAsync(&h_upd, d_upd, sizeof(int32_t), hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            rc = fail(HC_ERR_HIP, "epoch failed");
        epochs++;
    }
    hipEventRecord(e1, s);
    hipEventSynchronize(e1);
    float ms = 0;
    hipEventElapsedTime(&ms, e0, e1);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipFree(d_upd);
    if (rc == HC_OK && stats) {
        std::memset(stats, 0, sizeof(*stats));
        stats->ms = ms;
        stats->epochs = epochs;
        stats->pull_epochs = epochs;
        stats->launches = epochs;
    }
    return rc;
}

}  // extern "C"
