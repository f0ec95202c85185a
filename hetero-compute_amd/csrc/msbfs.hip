// Breadth-first depths from up to 64 sources at once, bit-parallel.
//
// The reference answers one BFS per driver call (bfs_gpu,
// src/kernels/gpu/bfs.cuh:21-95; bfs_do_cpu, src/kernels/cpu/bfs.cuh:48-114).
// Here the 64 searches share every sweep: each vertex keeps a 64-bit mask of
// the sources that have reached it (seen) and, per level, the mask of the
// sources whose frontier it is on.  Level L's frontier bit q of v is set
// exactly when v's depth from source q is L, so the depths are the unique
// BFS levels, identical to single-source runs.  A level costs one pass over
// the edges that matter with an 8-byte gather per edge, instead of one pass
// per source.
//
// Levels alternate between two directions, chosen from the frontier's edge
// count as bfs_do_cpu chooses between push and pull:
//  * push: the frontier list's vertices OR their frontier mask, less the
//    target's seen mask, into the target's next mask (an atomic only when
//    it adds a bit), and the first to set a target's mask appends it to the
//    next list;
//  * pull: every vertex not yet seen from all sources ORs its neighbours'
//    frontier masks (lanes stop once they hold every missing bit), over the
//    degree-bucketed plan, and records the bits it did not have.
// A commit pass over the next list then sets the depth entries of the new
// bits and folds them into seen.  Frontier masks and lists rotate over three
// buffers: level L reads buffer L-1, writes buffer L and clears buffer L-2
// by its list, so no pass clears a whole array.
//
// Depths are the int32 matrix of the batched SSSP interface, vertex-major
// (depth[v * 64 + q]), filled with HC_INF_DIST first.
#include <algorithm>
#include <cstring>
#include <vector>

#include "../../include/hc_batch.h"
#include "device_common.h"

namespace hc {

constexpr int kMsQ = 64;

// Per-level counters of one rotation slot: list length, its edge count
// (sum of degrees), edges examined, depth entries written.
struct MsCount {
    uint32_t len;
    uint32_t pad;
    unsigned long long deg, edges, bits;
};

struct MsBufs {
    uint64_t *seen;
    uint64_t *fr[3];
    int32_t *q[3];
    MsCount *cnt;  // [3]
    int32_t *depth;
    int32_t n;
    uint64_t full;  // bits of the sources in use
};

struct MsSeeds {
    int32_t v[kMsQ];
    uint64_t mask[kMsQ];
    int32_t k;
};

__device__ __forceinline__ uint64_t or_xor_shfl(uint64_t v, int s, int width) {
    return v | (uint64_t)__shfl_xor((unsigned long long)v, s, width);
}

template <int G>
__device__ __forceinline__ uint64_t group_or(uint64_t v) {
#pragma unroll
    for (int s = G / 2; s > 0; s >>= 1) v = or_xor_shfl(v, s, G);
    return v;
}

// OR over the 256-thread workgroup; valid in thread 0.
__device__ __forceinline__ uint64_t block_or(uint64_t v, uint64_t *s_part) {
    v = group_or<kWave>(v);
    __syncthreads();
    if (lane_id() == 0) s_part[threadIdx.x / kWave] = v;
    __syncthreads();
    uint64_t t = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < kWavesPerBlock; i++) t |= s_part[i];
    return t;
}

// Depth matrix to HC_INF_DIST, masks and seen to zero.
__global__ __launch_bounds__(kBlock) void ms_fill_kernel(MsBufs b) {
    const size_t stride = (size_t)gridDim.x * kBlock;
    const size_t cells = (size_t)b.n * kMsQ;
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < cells; i += stride)
        b.depth[i] = HC_INF_DIST;
    for (size_t v = blockIdx.x * (size_t)kBlock + threadIdx.x; v < (size_t)b.n; v += stride) {
        b.seen[v] = 0;
        b.fr[0][v] = 0;
        b.fr[1][v] = 0;
        b.fr[2][v] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x < 3) b.cnt[threadIdx.x] = MsCount{0, 0, 0, 0, 0};
}

// Level 0: the distinct source vertices with their masks.
template <typename OffT>
__global__ void ms_seed_kernel(MsBufs b, GraphView<OffT> g, MsSeeds s) {
    const int t = threadIdx.x;
    if (t < s.k) {
        const int32_t v = s.v[t];
        const uint64_t m = s.mask[t];
        b.seen[v] = m;
        b.fr[0][v] = m;
        b.q[0][t] = v;
        for (int q = 0; q < kMsQ; q++)
            if ((m >> q) & 1) b.depth[(size_t)v * kMsQ + q] = 0;
        atomicAdd(&b.cnt[0].deg, (unsigned long long)(g.rend(v) - g.rbeg(v)));
    }
    if (t == 0) b.cnt[0].len = (uint32_t)s.k;
}

// Clears the masks of level L-2 (buffer (L+1) % 3) by its list.
__device__ __forceinline__ void ms_clear_old(const MsBufs &b, int L) {
    const int o = (L + 1) % 3;
    const unsigned long long len = b.cnt[o].len;
    uint64_t *f = b.fr[o];
    const int32_t *q = b.q[o];
    for (unsigned long long i = blockIdx.x * (unsigned long long)kBlock + threadIdx.x; i < len;
         i += (unsigned long long)gridDim.x * kBlock)
        f[q[i]] = 0;
}

// A wavefront's part of the next list, collected in LDS and sent with one
// reservation per kMsStage / 2 entries: appends straight to the list take
// same-address atomics, which serialize at 12 ns each on this GPU.
constexpr int kMsStage = 512;

struct MsStage {
    int32_t *buf;  // kMsStage entries of LDS, this wavefront's
    int n;         // entries held (the same in every lane)
};

__device__ __forceinline__ void ms_stage_flush(MsStage &st, int32_t *nq, MsCount &c) {
    if (st.n == 0) return;
    // The entries were written by other lanes of this wavefront.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t base = 0;
    if (lane_id() == 0) base = atomicAdd(&c.len, (uint32_t)st.n);
    base = __shfl(base, 0);
    for (int i = lane_id(); i < st.n; i += kWave) nq[base + i] = st.buf[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    st.n = 0;
}

__device__ __forceinline__ void ms_stage_append(MsStage &st, bool pred, int32_t v) {
    const uint64_t m = __ballot(pred);
    if (pred) st.buf[st.n + __popcll(m & lanemask_lt())] = v;
    st.n += __popcll(m);
}

// Push level L over the list of level L-1.  The list is cut into windows of
// kMsWindow vertices, each taken by as many workgroups as its edges warrant;
// every one of them sums the window's chunk counts in LDS (kMsChunk edges a
// chunk, a group of kMsGroup lanes each) and takes its share of the chunks, so
// a short list of hubs fills the GPU as well as a long one of leaves.
// (Measured, Kronecker 22, 64 sources: with the list's vertices dealt whole, a
// wavefront per heavy one, levels of a few thousand hub-rich vertices took
// 3-14 ms on a handful of workgroups.)
constexpr int kMsWindow = 4096;
constexpr int kMsGroup = 16;
constexpr int kMsTrip = 4;                      // edges a lane has in flight
constexpr int kMsChunk = kMsGroup * kMsTrip;
constexpr int kMsPer = kMsWindow / kBlock;
// A list of no more edges than this, and of no more than kMsFewMean a vertex (a
// hub's would be one wavefront's: Kronecker 256K vertices, four sources, 398 ->
// 494 us), skips the windows, whose offsets, barriers and search make a longer
// chain than the edges do (grid of 256^2 vertices, one source, 510 levels: 16.9
// us a push with them, 10.4 without).
constexpr unsigned long long kMsFewMean = 16;
constexpr unsigned long long kMsFewEdges = 8192;

// Exclusive chunk offsets of a window's n vertices in s_pre, P of them per thread
// (as few as cover n: they are a chain of loads, and a deep graph's short lists
// wait for it); returns their sum.
template <int P, typename OffT>
__device__ __forceinline__ uint32_t ms_window_offsets(const GraphView<OffT> &g, const int32_t *wl,
                                                      int n, uint32_t *s_pre, uint32_t *s_wave) {
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    uint32_t mine[P], t = 0;
#pragma unroll
    for (int k = 0; k < P; k++) {
        const int i = threadIdx.x * P + k;
        uint32_t ch = 0;
        if (i < n) {
            const int32_t u = wl[i];
            ch = (uint32_t)((g.rend(u) - g.rbeg(u) + OffT(kMsChunk - 1)) / OffT(kMsChunk));
        }
        mine[k] = t;
        t += ch;
    }
    uint32_t incl = t;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
        const uint32_t o = __shfl_up(incl, s, kWave);
        if (lane >= s) incl += o;
    }
    __syncthreads();  // the window before is done with s_pre
    if (lane == kWave - 1) s_wave[wave] = incl;
    __syncthreads();
    uint32_t before = incl - t, total = 0;
    for (int w = 0; w < kWavesPerBlock; w++) {
        if (w < wave) before += s_wave[w];
        total += s_wave[w];
    }
#pragma unroll
    for (int k = 0; k < P; k++)
        if (threadIdx.x * P + k < (unsigned)kMsWindow) s_pre[threadIdx.x * P + k] = before + mine[k];
    __syncthreads();
    return total;
}

// Workgroups per window of a push from `len` vertices with `deg` edges.
__host__ __device__ inline int ms_push_share(unsigned long long len, unsigned long long deg,
                                             int grid) {
    const unsigned long long wins = (len + kMsWindow - 1) / kMsWindow;
    if (wins == 0) return 1;
    // About four chunks (at least one a vertex) for each group of lanes.
    const unsigned long long want = (deg / kMsChunk + len) / (4ull * kBlock / kMsGroup) + 1;
    const unsigned long long per = (want + wins - 1) / wins;
    const unsigned long long most = (unsigned long long)grid / wins;
    return (int)(per < most ? per : (most ? most : 1));
}

template <typename OffT>
__global__ __launch_bounds__(kBlock) void ms_push_kernel(MsBufs b, GraphView<OffT> g, int L) {
    __shared__ uint32_t s_pre[kMsWindow];
    __shared__ uint32_t s_wave[kWavesPerBlock];
    __shared__ int32_t s_stage[kWavesPerBlock][kMsStage];
    const int cu = (L + 2) % 3, nx = L % 3;
    const uint64_t *cur = b.fr[cu];
    uint64_t *nxt = b.fr[nx];
    const int32_t *list = b.q[cu];
    int32_t *nq = b.q[nx];
    MsCount &c = b.cnt[nx];
    ms_clear_old(b, L);
    // Counters of buffer nx were reset by the previous commit; the list
    // length read here is level L-1's, final since its commit.
    const unsigned long long len = b.cnt[cu].len;
    const int per = ms_push_share(len, b.cnt[cu].deg, gridDim.x);
    const bool few = b.cnt[cu].deg <= min(kMsFewEdges, kMsFewMean * len);
    const unsigned long long wins = few ? 0 : (len + kMsWindow - 1) / kMsWindow;
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    MsStage st{s_stage[wave], 0};
    unsigned long long deg_acc = 0, edges = 0;
    // The next masks of a trip's targets (-1: none) of a frontier vertex with
    // mask fu.
    auto take = [&](const int32_t (&v)[kMsTrip], uint64_t fu) {
                    uint64_t bits[kMsTrip], have[kMsTrip];
#pragma unroll
                    for (int r = 0; r < kMsTrip; r++) {
                        bits[r] = v[r] >= 0 ? fu & ~b.seen[v[r]] : 0;
                        have[r] = v[r] >= 0 ? nxt[v[r]] : 0;
                    }
                    bool fresh[kMsTrip];
#pragma unroll
                    for (int r = 0; r < kMsTrip; r++) {
                        edges += v[r] >= 0;
                        // An atomic only when it adds a bit the next mask lacks.
                        fresh[r] = (bits[r] & ~have[r]) != 0 &&
                                   atomicOr((unsigned long long *)&nxt[v[r]],
                                            (unsigned long long)bits[r]) == 0;
                    }
#pragma unroll
                    for (int r = 0; r < kMsTrip; r++) {
                        if (fresh[r]) deg_acc += (unsigned long long)(g.rend(v[r]) - g.rbeg(v[r]));
                        ms_stage_append(st, fresh[r], v[r]);
                    }
        if (st.n > kMsStage - kMsTrip * kWave) ms_stage_flush(st, nq, c);
    };
    if (few) {
        // A few edges: four lanes a vertex, and the wavefront together for what
        // a vertex has beyond kMsChunk.
        constexpr int G = 4, PER = kWave / G;
        const unsigned long long waves = (unsigned long long)gridDim.x * kWavesPerBlock;
        for (unsigned long long q0 =
                 (blockIdx.x * (unsigned long long)kWavesPerBlock + wave) * PER;
             q0 < len; q0 += waves * PER) {
            const bool ok = q0 + lane / G < len;
            const int32_t u = ok ? list[q0 + lane / G] : 0;
            const OffT ub = ok ? g.rbeg(u) : OffT(0), ue = ok ? g.rend(u) : OffT(0);
            const uint64_t fu = ok ? cur[u] : 0;
            const OffT mid = min(ue, ub + OffT(kMsChunk));
            for (OffT t = 0; t < OffT(kMsChunk); t += OffT(kMsTrip * G)) {
                if (__ballot(ub + t < mid) == 0) break;
                int32_t v[kMsTrip];
#pragma unroll
                for (int r = 0; r < kMsTrip; r++) {
                    const OffT k = ub + t + OffT(r * G + lane % G);
                    v[r] = k < mid ? ldnt(&g.adj[k]) : -1;
                }
                take(v, fu);
            }
            for (uint64_t hv = __ballot(lane % G == 0 && mid < ue); hv; hv &= hv - 1) {
                const int l = __ffsll((unsigned long long)hv) - 1;
                const OffT e = __shfl(ue, l);
                const uint64_t hfu = (uint64_t)__shfl((unsigned long long)fu, l);
                for (OffT i = __shfl(mid, l); i < e; i += OffT(kMsTrip * kWave)) {
                    int32_t v[kMsTrip];
#pragma unroll
                    for (int r = 0; r < kMsTrip; r++) {
                        const OffT k = i + OffT(r * kWave + lane);
                        v[r] = k < e ? ldnt(&g.adj[k]) : -1;
                    }
                    take(v, hfu);
                }
            }
        }
    }
    const int sub = blockIdx.x % per;
    for (unsigned long long win = blockIdx.x / per; win < wins; win += gridDim.x / per) {
        if (blockIdx.x / per >= gridDim.x / per) break;  // past the last full share
        const int n = (int)min((unsigned long long)kMsWindow, len - win * kMsWindow);
        const int32_t *wl = list + win * kMsWindow;
        uint32_t total;
        if (n <= kBlock) total = ms_window_offsets<1>(g, wl, n, s_pre, s_wave);
        else if (n <= 4 * kBlock) total = ms_window_offsets<4>(g, wl, n, s_pre, s_wave);
        else total = ms_window_offsets<kMsPer>(g, wl, n, s_pre, s_wave);
        // Chunks in rounds of the wavefront's groups (the same count in all
        // its lanes).
        constexpr int kGroups = kWave / kMsGroup;
        const uint32_t first = (uint32_t)(sub * kWavesPerBlock + wave) * kGroups;
        const uint32_t step = (uint32_t)per * kWavesPerBlock * kGroups;
        for (uint32_t q0 = first; q0 < total; q0 += step) {
            const uint32_t q = q0 + lane / kMsGroup;
            int32_t v[kMsTrip];
            uint64_t fu = 0;
            if (q < total) {
                int lo = 0, hi = n;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) / 2;
                    if (s_pre[mid] <= q) lo = mid; else hi = mid;
                }
                const int32_t u = wl[lo];
                const OffT e = g.rend(u);
                const OffT i0 = g.rbeg(u) + OffT(q - s_pre[lo]) * OffT(kMsChunk) +
                                OffT(lane % kMsGroup);
                fu = cur[u];
#pragma unroll
                for (int r = 0; r < kMsTrip; r++) {
                    const OffT k = i0 + OffT(r * kMsGroup);
                    v[r] = k < e ? ldnt(&g.adj[k]) : -1;
                }
            } else {
#pragma unroll
                for (int r = 0; r < kMsTrip; r++) v[r] = -1;
            }
            take(v, fu);
        }
    }
    ms_stage_flush(st, nq, c);
    const unsigned long long d = block_sum_u64(deg_acc);
    const unsigned long long ed = block_sum_u64(edges);
    if (threadIdx.x == 0) {
        if (d) atomicAdd(&c.deg, d);
        if (ed) atomicAdd(&c.edges, ed);
    }
}

// One row (or hub chunk) of the pull sweep by a group of G lanes: OR of the
// neighbours' frontier masks, four edges per lane per trip (ids, then the
// four gathers, in flight together), each lane stopping once it holds every
// bit the row is missing.
template <int G, typename OffT>
__device__ __forceinline__ uint64_t ms_row_or(const GraphView<OffT> &g, const uint64_t *cur,
                                              OffT b0, OffT e, int lane, uint64_t need,
                                              unsigned long long &edges) {
    uint64_t acc = 0;
    for (OffT i = b0 + OffT(lane); i < e; i += OffT(4 * G)) {
        int32_t v[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const OffT k = i + OffT(r * G);
            v[r] = k < e ? ldnt(&g.adj[k]) : -1;
        }
        uint64_t m[4];
#pragma unroll
        for (int r = 0; r < 4; r++) m[r] = v[r] >= 0 ? cur[v[r]] : 0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            acc |= m[r];
            edges += v[r] >= 0;
        }
        if ((acc & need) == need) break;
    }
    return acc;
}

// A row of a wavefront's block, one per lane.
template <typename OffT>
struct MsHead {
    int32_t v;
    uint64_t need;  // sources that have not reached it (0: nothing to do)
    OffT b, e;
};

// The wanted rows among a wavefront's heads (those of lanes j0, j0 + jstep,
// ...; which wavefront takes a row must not depend on masks that change), G
// lanes per row.  SHARED: the heads are chunks of hub rows, whose bits are
// added with atomicOr.
template <int G, bool SHARED, typename OffT>
__device__ __forceinline__ void ms_pull_block(const MsHead<OffT> &h, int j0, int jstep,
                                              const GraphView<OffT> &g, const uint64_t *cur,
                                              uint64_t *nxt, int32_t *nq, MsCount &c, MsStage &st,
                                              unsigned long long &deg_acc,
                                              unsigned long long &edges) {
    constexpr int PER = kWave / G;
    const int lane = lane_id();
    const bool want = h.need != 0 && lane % jstep == j0;
    const uint64_t mask = __ballot(want);
    const int n = __popcll(mask);
    // Lane r learns the lane of the r-th wanted row.
    const int rank = __popcll(mask & lanemask_lt());
    const int src = __builtin_amdgcn_ds_permute((want ? rank : n + lane - rank) << 2, lane);
    for (int j = 0; j * PER < n; j++) {
        const int gi = j * PER + lane / G;
        const bool have = gi < n;
        const int sl = __shfl(src, gi & (kWave - 1));
        const int32_t v = __shfl(h.v, sl);
        const uint64_t need = (uint64_t)__shfl((unsigned long long)h.need, sl);
        const OffT b = __shfl(h.b, sl), e = __shfl(h.e, sl);
        uint64_t got = 0;
        if (have) {
            got = ms_row_or<G, OffT>(g, cur, b, e, lane % G, need, edges);
            if (G > 1) got = group_or<G>(got);
            got &= need;
        }
        bool first = false;
        if (have && lane % G == 0 && got != 0) {
            if (SHARED) {
                first = atomicOr((unsigned long long *)&nxt[v], (unsigned long long)got) == 0;
                if (first) deg_acc += (unsigned long long)(g.rend(v) - g.rbeg(v));
            } else {
                nxt[v] = got;  // the only group on this row
                first = true;
                deg_acc += (unsigned long long)(e - b);
            }
        }
        ms_stage_append(st, first, v);
        if (st.n > kMsStage - kWave) ms_stage_flush(st, nq, c);
    }
}

// Wavefronts that share a block of 64 heads of hub chunks and heavy rows (64
// lanes a row), and of 16-lane rows.
constexpr int kMsSplit = 16;
constexpr int kMsSplit16 = 4;

// Pull level L over the plan (all rows of the graph; sorted_plan_config), in
// wavefront units: a block of 64 rows' masks and bounds is read at once, the
// next block's ahead of this one's edges, and only rows that miss a source
// get lanes.  (Measured, Kronecker 22, 64 sources, three pull levels: 4.8 ms
// in column blocks with an append per wavefront straight to the list, 2.5 ms
// with staged appends, 1.6 ms here without the column blocks, whose copy took
// 90 ms to build.)
template <typename OffT>
__global__ __launch_bounds__(kBlock) void ms_pull_kernel(MsBufs b, GraphView<OffT> g, PlanDev p,
                                                         int L) {
    __shared__ int32_t s_stage[kWavesPerBlock][kMsStage];
    MsStage st{s_stage[threadIdx.x / kWave], 0};
    const int cu = (L + 2) % 3, nx = L % 3;
    const uint64_t *cur = b.fr[cu];
    uint64_t *nxt = b.fr[nx];
    int32_t *nq = b.q[nx];
    MsCount &c = b.cnt[nx];
    ms_clear_old(b, L);
    unsigned long long deg_acc = 0, edges = 0;
    const int b0 = (p.cnt[0] + 63) / 64, b2 = (p.cnt[2] + 63) / 64;
    const int b3 = (p.cnt[3] + 63) / 64, b4 = (p.cnt[4] + 63) / 64, b5 = (p.cnt[5] + 63) / 64;
    const int stride = gridDim.x * kWavesPerBlock;
    const int t0 = b0 * kMsSplit, t2 = t0 + b2 * kMsSplit, t3 = t2 + b3 * kMsSplit16;
    const int t4 = t3 + b4, total = t4 + b5;
    const int lane = lane_id();
    auto head = [&](int unit) {
        MsHead<OffT> h{0, 0, OffT(0), OffT(0)};
        int i = 0, beg = 0, cnt = 0;
        const int32_t *list = nullptr;
        if (unit < t0) {
            i = unit / kMsSplit * 64 + lane;
            if (i < p.cnt[0]) {
                const HubChunk ch = p.chunks[i];
                h.v = ch.u;
                h.b = OffT(ch.b);
                h.e = OffT(ch.e);
                h.need = b.full & ~b.seen[ch.u];
            }
            return h;
        } else if (unit < t2) {
            i = (unit - t0) / kMsSplit * 64 + lane;
            cnt = p.cnt[2];
            beg = p.beg[2];
            list = p.list[2];
        } else if (unit < t3) {
            i = (unit - t2) / kMsSplit16 * 64 + lane;
            cnt = p.cnt[3];
            beg = p.beg[3];
            list = p.list[3];
        } else if (unit < t4) {
            i = (unit - t3) * 64 + lane;
            cnt = p.cnt[4];
            beg = p.beg[4];
            list = p.list[4];
        } else if (unit < total) {
            i = (unit - t4) * 64 + lane;
            cnt = p.cnt[5];
            beg = p.beg[5];
            list = p.list[5];
        }
        if (i < cnt) {
            h.v = list ? list[i] : beg + i;
            h.need = b.full & ~b.seen[h.v];
            h.b = g.rbeg(h.v);
            h.e = g.rend(h.v);
        }
        return h;
    };
    int unit = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    MsHead<OffT> h = head(unit);
    while (unit < total) {
        const MsHead<OffT> ahead = head(unit + stride);
        if (unit < t0)
            ms_pull_block<64, true>(h, unit % kMsSplit, kMsSplit, g, cur, nxt, nq, c, st, deg_acc,
                                    edges);
        else if (unit < t2)
            ms_pull_block<64, false>(h, (unit - t0) % kMsSplit, kMsSplit, g, cur, nxt, nq, c, st,
                                     deg_acc, edges);
        else if (unit < t3)
            ms_pull_block<16, false>(h, (unit - t2) % kMsSplit16, kMsSplit16, g, cur, nxt, nq, c,
                                     st, deg_acc, edges);
        else if (unit < t4)
            ms_pull_block<4, false>(h, 0, 1, g, cur, nxt, nq, c, st, deg_acc, edges);
        else
            ms_pull_block<1, false>(h, 0, 1, g, cur, nxt, nq, c, st, deg_acc, edges);
        unit += stride;
        h = ahead;
    }
    ms_stage_flush(st, nq, c);
    const unsigned long long d = block_sum_u64(deg_acc);
    const unsigned long long ed = block_sum_u64(edges);
    if (threadIdx.x == 0) {
        if (d) atomicAdd(&c.deg, d);
        if (ed) atomicAdd(&c.edges, ed);
    }
}

// Pull level L over the column blocks of the graph (see colblock.hip):
// units (block k, plan unit) in block-major order, so the grid gathers from
// one window of 2^shift frontier masks at a time.  Plan classes are by mean
// slice degree and have no hub chunks.  A row's bits may come from several
// blocks: they are added with atomicOr (only when the next mask lacks one),
// and the call that made the mask non-zero lists the row.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void ms_pull_cb_kernel(MsBufs b, GraphView<OffT> g,
                                                            GraphView<OffT> cb, int K,
                                                            PlanDev p, int L) {
    __shared__ uint64_t s_or[kWavesPerBlock];
    __shared__ int32_t s_stage[kWavesPerBlock][kMsStage];
    MsStage st{s_stage[threadIdx.x / kWave], 0};
    const int cu = (L + 2) % 3, nx = L % 3;
    const uint64_t *cur = b.fr[cu];
    uint64_t *nxt = b.fr[nx];
    int32_t *nq = b.q[nx];
    MsCount &c = b.cnt[nx];
    ms_clear_old(b, L);
    unsigned long long deg_acc = 0, edges = 0;
    const int U = p.unit_start[kNumClasses];
    const int total = U * K;
    for (int unit = blockIdx.x; unit < total; unit += gridDim.x) {
        const int blk = unit / U;
        const int pu = unit - blk * U;
        GraphView<OffT> gk = cb;
        gk.off = cb.off + (size_t)blk * ((size_t)g.n + 1);
        int cls = 0;
        while (pu >= p.unit_start[cls + 1]) cls++;
        const int k = pu - p.unit_start[cls];
        if (cls <= 1) {
            // A workgroup per row slice (no hub chunks in this plan).
            const int32_t v = p.list[1] ? p.list[1][k] : p.beg[1] + k;
            const uint64_t need = b.full & ~b.seen[v];
            uint64_t acc = 0;
            if (need)
                acc = ms_row_or<kBlock, OffT>(gk, cur, gk.rbeg(v), gk.rend(v), threadIdx.x, need,
                                              edges);
            const uint64_t got = block_or(acc, s_or) & need;
            bool first = false;
            if (threadIdx.x == 0 && (got & ~nxt[v])) {
                first = atomicOr((unsigned long long *)&nxt[v], (unsigned long long)got) == 0;
                if (first) deg_acc += (unsigned long long)(g.rend(v) - g.rbeg(v));
            }
            if (threadIdx.x < kWave) {
                ms_stage_append(st, first, v);
                if (st.n > kMsStage - kWave) ms_stage_flush(st, nq, c);
            }
            __syncthreads();
            continue;
        }
        const int G = cls == 2 ? 64 : cls == 3 ? 16 : cls == 4 ? 4 : 1;
        const int per = kBlock / G;
        const int idx = k * per + (int)threadIdx.x / G;
        const int li = (int)threadIdx.x % G;
        const bool ok = idx < p.cnt[cls];
        int32_t v = 0;
        uint64_t need = 0, acc = 0;
        if (ok) {
            v = p.list[cls] ? p.list[cls][idx] : p.beg[cls] + idx;
            need = b.full & ~b.seen[v];
            if (need) {
                const OffT rb = gk.rbeg(v), re = gk.rend(v);
                if (cls == 2)
                    acc = ms_row_or<64, OffT>(gk, cur, rb, re, li, need, edges);
                else if (cls == 3)
                    acc = ms_row_or<16, OffT>(gk, cur, rb, re, li, need, edges);
                else if (cls == 4)
                    acc = ms_row_or<4, OffT>(gk, cur, rb, re, li, need, edges);
                else
                    acc = ms_row_or<1, OffT>(gk, cur, rb, re, li, need, edges);
            }
        }
        if (cls == 2)
            acc = group_or<64>(acc);
        else if (cls == 3)
            acc = group_or<16>(acc);
        else if (cls == 4)
            acc = group_or<4>(acc);
        const uint64_t got = acc & need;
        bool first = false;
        if (ok && li == 0 && (got & ~nxt[v])) {
            first = atomicOr((unsigned long long *)&nxt[v], (unsigned long long)got) == 0;
            if (first) deg_acc += (unsigned long long)(g.rend(v) - g.rbeg(v));
        }
        ms_stage_append(st, first, v);
        if (st.n > kMsStage - kWave) ms_stage_flush(st, nq, c);
    }
    ms_stage_flush(st, nq, c);
    const unsigned long long d = block_sum_u64(deg_acc);
    const unsigned long long ed = block_sum_u64(edges);
    if (threadIdx.x == 0) {
        if (d) atomicAdd(&c.deg, d);
        if (ed) atomicAdd(&c.edges, ed);
    }
}

// Commit of level L: depth entries of the new bits, seen updated.  A
// wavefront takes up to 64 listed vertices, as many as give every wavefront
// some: their masks are read at once, a lane each, then their rows are written
// one after another, lane q source q's entry (with a vertex per wavefront the
// chain list, mask, row bounded a long level: 420 us for 2.3 M vertices of
// Kronecker 22; with 64 a short one of some hundred vertices took 8 us, and 4
// so).  Resets the counters of
// buffer (L+1) % 3, which level L+1 fills.
constexpr int kMsCommitMin = 4;
__global__ __launch_bounds__(kBlock) void ms_commit_kernel(MsBufs b, int L) {
    const int nx = L % 3;
    const uint64_t *nxt = b.fr[nx];
    const int32_t *q = b.q[nx];
    const unsigned long long len = b.cnt[nx].len;
    const int lane = lane_id();
    unsigned long long bits = 0;
    const unsigned long long waves = (unsigned long long)gridDim.x * kWavesPerBlock;
    const unsigned long long per =
        min((unsigned long long)kWave, max((unsigned long long)kMsCommitMin, len / 256));
    for (unsigned long long i0 = (blockIdx.x * (unsigned long long)kWavesPerBlock +
                                  threadIdx.x / kWave) * per;
         i0 < len; i0 += waves * per) {
        const int n = (int)min(per, len - i0);
        int32_t v = 0;
        uint64_t nb = 0;
        if (lane < n) {
            v = q[i0 + lane];
            nb = nxt[v];
            b.seen[v] |= nb;
            bits += (unsigned long long)__popcll(nb);
        }
        const uint32_t lo = (uint32_t)nb, hi = (uint32_t)(nb >> 32);
        for (int j = 0; j < n; j++) {
            const int32_t vj = __builtin_amdgcn_readlane(v, j);
            const uint32_t lj = __builtin_amdgcn_readlane(lo, j);
            const uint32_t hj = __builtin_amdgcn_readlane(hi, j);
            if (((lane < 32 ? lj : hj) >> (lane & 31)) & 1u) b.depth[(size_t)vj * kMsQ + lane] = L;
        }
    }
    const unsigned long long t = block_sum_u64(bits);
    if (threadIdx.x == 0 && t) atomicAdd(&b.cnt[nx].bits, t);
    if (blockIdx.x == 0 && threadIdx.x == 0) b.cnt[(L + 1) % 3] = MsCount{0, 0, 0, 0, 0};
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

struct MsBfsWs {
    void *dmem = nullptr;
    MsCount *h_cnt = nullptr;  // pinned mirror of the three counter slots
    MsBufs b{};
    ~MsBfsWs() {
        if (dmem) hipFree(dmem);
        if (h_cnt) hipHostFree(h_cnt);
    }
};

void free_msbfs_ws(hc_graph_s *g) {
    delete static_cast<MsBfsWs *>(g->ws_msbfs);
    g->ws_msbfs = nullptr;
}

static int get_msbfs_ws(hc_graph_s *g, MsBfsWs **out) {
    auto *ws = static_cast<MsBfsWs *>(g->ws_msbfs);
    if (!ws) {
        ws = new (std::nothrow) MsBfsWs();
        if (!ws) return fail(HC_ERR_OOM, "host allocation failed");
        const size_t n = (size_t)std::max(g->n, 1);
        auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
        const size_t sz_mask = al(sizeof(uint64_t) * n), sz_q = al(sizeof(int32_t) * n);
        const size_t sz_cnt = al(sizeof(MsCount) * 3);
        const size_t total = 4 * sz_mask + 3 * sz_q + sz_cnt;
        char *base = nullptr;
        if (hipMalloc(reinterpret_cast<void **>(&base), total) != hipSuccess) {
            delete ws;
            return fail(HC_ERR_OOM, "batched-BFS workspace of %zu bytes failed", total);
        }
        ws->dmem = base;
        if (hipHostMalloc(reinterpret_cast<void **>(&ws->h_cnt), sizeof(MsCount) * 3,
                          hipHostMallocDefault) != hipSuccess) {
            delete ws;
            return fail(HC_ERR_OOM, "pinned counter allocation failed");
        }
        MsBufs &b = ws->b;
        b.seen = reinterpret_cast<uint64_t *>(base);
        for (int k = 0; k < 3; k++) b.fr[k] = reinterpret_cast<uint64_t *>(base + (k + 1) * sz_mask);
        for (int k = 0; k < 3; k++)
            b.q[k] = reinterpret_cast<int32_t *>(base + 4 * sz_mask + k * sz_q);
        b.cnt = reinterpret_cast<MsCount *>(base + 4 * sz_mask + 3 * sz_q);
        b.n = g->n;
        g->ws_msbfs = ws;
    }
    *out = ws;
    return HC_OK;
}

template <typename OffT>
static int run_msbfs(hc_graph_s *g, const int32_t *sources, int num, int32_t *depth,
                     int max_levels, hc_run_stats_t *stats, hipStream_t s) {
    MsBfsWs *ws = nullptr;
    HC_TRY(get_msbfs_ws(g, &ws));
    const PlanHost *ph = nullptr;
    HC_TRY(get_plan(g, 0, g->n, sorted_plan_config(), &ph));
    const ColBlocks *cb = nullptr;
    const PlanHost *pcb = nullptr;
    const int shift = tuning().msbfs_col_shift;
    if (shift > 0) HC_TRY(get_col_blocks(g, shift, s, &cb));
    if (cb) {
        PlanConfig c = cb_plan_config(cb->K);
        c.min_degree = 1;
        HC_TRY(get_plan(g, 0, g->n, c, &pcb));
    }
    MsBufs b = ws->b;
    b.depth = depth;
    b.full = num >= kMsQ ? ~0ull : ((1ull << num) - 1);
    MsSeeds seeds{};
    for (int q = 0; q < num; q++) {
        int j = 0;
        while (j < seeds.k && seeds.v[j] != sources[q]) j++;
        if (j == seeds.k) {
            seeds.v[j] = sources[q];
            seeds.mask[j] = 0;
            seeds.k++;
        }
        seeds.mask[j] |= 1ull << q;
    }
    const GraphView<OffT> gv = view<OffT>(g);
    const int grid = grid_blocks();
    const int alpha = std::max(1, tuning().msbfs_alpha);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    HC_HIP(hipEventCreate(&e0));
    HC_HIP(hipEventCreate(&e1));
    HC_HIP(hipEventRecord(e0, s));
    ms_fill_kernel<<<grid, kBlock, 0, s>>>(b);
    ms_seed_kernel<OffT><<<1, kMsQ, 0, s>>>(b, gv, seeds);
    int rc = hipGetLastError() == hipSuccess ? HC_OK : fail(HC_ERR_HIP, "batched BFS start failed");
    unsigned long long len = (unsigned long long)seeds.k, deg = 0;
    for (int q = 0; q < seeds.k; q++) {
        const int32_t v = seeds.v[q];
        deg += (unsigned long long)(g->h_off[v + 1] - g->h_off[v]);
    }
    const unsigned long long m = (unsigned long long)std::max<int64_t>(g->m, 1);
    const int cap = max_levels > 0 ? max_levels : g->n + 1;
    int levels = 0, pushes = 0, pulls = 0;
    double bytes = 4.0 * kMsQ * (double)g->n + 32.0 * g->n;  // fill
    while (rc == HC_OK && len > 0 && levels < cap) {
        const int L = levels + 1;
        const bool push = deg * (unsigned long long)alpha < m;
        if (push) {
            ms_push_kernel<OffT><<<grid, kBlock, 0, s>>>(b, gv, L);
            pushes++;
        } else if (cb) {
            const GraphView<OffT> cbv{static_cast<const OffT *>(cb->off), cb->adj, nullptr, 0,
                                      g->n};
            ms_pull_cb_kernel<OffT><<<grid, kBlock, 0, s>>>(b, gv, cbv, cb->K, pcb->dev, L);
            pulls++;
        } else {
            ms_pull_kernel<OffT><<<grid, kBlock, 0, s>>>(b, gv, ph->dev, L);
            pulls++;
        }
        ms_commit_kernel<<<grid, kBlock, 0, s>>>(b, L);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(ws->h_cnt + L % 3, b.cnt + L % 3, sizeof(MsCount),
                           hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess) {
            rc = fail(HC_ERR_HIP, "batched BFS level %d failed", L);
            break;
        }
        const MsCount c = ws->h_cnt[L % 3];
        // Offsets and ids of the examined edges, the 8-byte mask gathered
        // per edge (seen on push, the frontier on pull) and per listed
        // vertex, and the depth entries written.
        bytes += 12.0 * (double)c.edges + 24.0 * (double)c.len + 4.0 * (double)c.bits +
                 (push ? 16.0 * (double)len : 8.0 * g->n);
        len = c.len;
        deg = c.deg;
        levels = L;
    }
    HC_HIP(hipEventRecord(e1, s));
    HC_HIP(hipEventSynchronize(e1));
    float ms = 0;
    HC_HIP(hipEventElapsedTime(&ms, e0, e1));
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    HC_TRY(rc);
    if (stats) {
        std::memset(stats, 0, sizeof(*stats));
        stats->ms = ms;
        stats->epochs = levels;
        stats->push_epochs = pushes;
        stats->pull_epochs = pulls;
        stats->launches = 2 + 2 * levels;
        stats->reached = num;
        stats->alg_bytes = bytes;
    }
    return HC_OK;
}

int run_msbfs_entry(hc_graph_s *g, const int32_t *sources, int num, int32_t *depth,
                    int max_levels, hc_run_stats_t *stats, hipStream_t s) {
    return g->off64 ? run_msbfs<uint64_t>(g, sources, num, depth, max_levels, stats, s)
                    : run_msbfs<uint32_t>(g, sources, num, depth, max_levels, stats, s);
}

}  // namespace hc
