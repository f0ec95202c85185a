// Weight-sorted adjacency for the SSSP sweeps, built on the GPU from the
// resident CSR.
//
// A relaxation only helps when dist[v] + w is below dist[u].  With the edges
// of each row in order of rising weight, and a lower bound `low` of every
// distance that changed since u was last relaxed, a scan of row u can stop at
// the first edge with low + w >= dist[u]: no later edge can lower u.  On a
// Kronecker graph of 2^19 vertices with weights 1..255 a pull sweep then
// looks at 4-17% of the edges (one and 16 edges per stop test), on a uniform
// one bucketed pushes and sweeps look at a third.
//
// Ids and weights are interleaved (one 8-byte load per edge) in the CSR's row
// layout, so the CSR's offsets serve both.  The order is by key
// min(w >> shift, 63), coarse for weights above 63, and the stop test uses the
// key's lower bound (SortedView::floor), so it is exact all the same: with
// weights up to 255 a scan goes on for at most three units of weight, about
// one edge of a mean row, and the sort takes a quarter of the counters.
//
// Build, over the degree classes the sweeps use (sorted_plan_config): rows of
// at most 64 edges by a bitonic sort in registers, rows of at most 2048 by a
// counting sort per wavefront (64 keys in LDS), heavier ones by chunks
// (histogram, scan, scatter).  Kronecker 23 (2.59e8 edges) 3.7 ms, uniform 23
// 5.5 ms, once per graph and its shares: a first query on either costs no more
// than it did on the plain CSR.
#include <algorithm>
#include <climits>

#include "frontier.h"

namespace hc {

constexpr int kSortRun = 8;  // plan chunks a workgroup takes together

SortedSlot::~SortedSlot() {
    if (adj.e) (void)hipFree(adj.e);
}

__device__ __forceinline__ int sort_key(int32_t w, int shift) {
    const int k = w >> shift;
    return k < kSortKeys ? k : kSortKeys - 1;
}

// Rows of degree <= G: one per group of G lanes, bitonic in registers by
// (weight, id).
template <int G, typename OffT>
__device__ __forceinline__ void sort_group(const GraphView<OffT> &g, int2 *e, bool ok, int32_t u) {
    const int lane = threadIdx.x % G;
    const OffT b = ok ? g.rbeg(u) : OffT(0);
    const OffT d = ok ? g.rend(u) - b : OffT(0);
    unsigned long long key = ~0ull;
    if (OffT(lane) < d)
        key = ((unsigned long long)(uint32_t)ldnt(&g.wt[b + lane]) << 32) |
              (uint32_t)ldnt(&g.adj[b + lane]);
#pragma unroll
    for (int size = 2; size <= G; size <<= 1) {
#pragma unroll
        for (int s = size >> 1; s > 0; s >>= 1) {
            const unsigned long long o = __shfl_xor(key, s, G);
            const bool up = (lane & size) == 0 || size == G;
            const bool low = (lane & s) == 0;
            key = (low == up) ? (key < o ? key : o) : (key < o ? o : key);
        }
    }
    if (OffT(lane) < d) e[b + lane] = int2{(int32_t)(uint32_t)key, (int32_t)(key >> 32)};
}

// Orders one wavefront's LDS accesses before and after it.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One row per wavefront by counting sort, a key per lane in the wavefront's
// own LDS words.
template <typename OffT>
__device__ __forceinline__ void sort_row(const GraphView<OffT> &g, int2 *e, int shift, int32_t u,
                                         uint32_t *cnt) {
    const int lane = lane_id();
    const OffT b = g.rbeg(u), end = g.rend(u);
    cnt[lane] = 0;
    wave_lds_sync();
    for (OffT i = b + OffT(lane); i < end; i += OffT(kWave))
        atomicAdd(&cnt[sort_key(g.wt[i], shift)], 1u);
    wave_lds_sync();
    // Exclusive scan.
    const uint32_t t = cnt[lane];
    uint32_t incl = t;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
        const uint32_t o = __shfl_up(incl, s, kWave);
        if (lane >= s) incl += o;
    }
    cnt[lane] = incl - t;
    wave_lds_sync();
    for (OffT i = b + OffT(lane); i < end; i += OffT(kWave)) {
        const int32_t w = g.wt[i];
        const uint32_t at = atomicAdd(&cnt[sort_key(w, shift)], 1u);
        e[b + OffT(at)] = int2{g.adj[i], w};
    }
    wave_lds_sync();
}

// Rows of plan classes 2-5, in wavefront units: one row of classes 2 and 3
// (above 64 edges), four rows of class 4 (four groups of 16 lanes when they
// all fit, else one after another), 16 rows of class 5.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void sort_rows_kernel(PlanDev p, GraphView<OffT> g, int2 *e,
                                                           int shift) {
    __shared__ uint32_t s_cnt[kWavesPerBlock][kSortKeys];
    const int lane = lane_id();
    const int n2 = p.cnt[2], n3 = p.cnt[3];
    const int n4 = (p.cnt[4] + 3) / 4, n5 = (p.cnt[5] + 15) / 16;
    const int total = n2 + n3 + n4 + n5;
    const int stride = gridDim.x * kWavesPerBlock;
    for (int unit = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; unit < total;
         unit += stride) {
        if (unit < n2) {
            sort_row(g, e, shift, p.list[2] ? p.list[2][unit] : p.beg[2] + unit,
                     s_cnt[threadIdx.x / kWave]);
        } else if (unit < n2 + n3) {
            const int i = unit - n2;
            sort_row(g, e, shift, p.list[3] ? p.list[3][i] : p.beg[3] + i,
                     s_cnt[threadIdx.x / kWave]);
        } else if (unit < n2 + n3 + n4) {
            const int i = (unit - n2 - n3) * 4 + lane / 16;
            const bool ok = i < p.cnt[4];
            const int32_t u = ok ? (p.list[4] ? p.list[4][i] : p.beg[4] + i) : 0;
            if (__ballot(ok && g.rend(u) - g.rbeg(u) > OffT(16)) == 0) {
                sort_group<16>(g, e, ok, u);
            } else {
#pragma unroll 1
                for (int q = 0; q < kWave; q += 16) {
                    const int32_t uq = __builtin_amdgcn_readlane(u, q);
                    sort_group<64>(g, e, __builtin_amdgcn_readlane(ok ? 1 : 0, q) != 0, uq);
                }
            }
        } else {
            const int i = (unit - n2 - n3 - n4) * 16 + lane / 4;
            const bool ok = i < p.cnt[5];
            sort_group<4>(g, e, ok, ok ? (p.list[5] ? p.list[5][i] : p.beg[5] + i) : 0);
        }
    }
}

__global__ void sort_zero_kernel(uint32_t *x, size_t count) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += stride) x[i] = 0;
}

// Calls f(hub, row, first edge, last edge) for the runs of plan chunks of one
// hub among kSortRun consecutive chunks (the chunks of a row are consecutive
// and cover it in order).
template <typename F>
__device__ __forceinline__ void hub_runs(const PlanDev &p, F f) {
    const int groups = (p.cnt[0] + kSortRun - 1) / kSortRun;
    for (int r = blockIdx.x; r < groups; r += gridDim.x) {
        const int end = min(p.cnt[0], (r + 1) * kSortRun);
        for (int c = r * kSortRun; c < end;) {
            const HubChunk h = p.chunks[c];
            int64_t last = h.e;
            for (c++; c < end && p.chunks[c].hub == h.hub; c++) last = p.chunks[c].e;
            f(h.hub, h.u, h.b, last);
        }
    }
}

// hist[hub][key] += the run's edges of that key.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void sort_hub_count_kernel(PlanDev p, GraphView<OffT> g,
                                                                int shift, uint32_t *hist) {
    __shared__ uint32_t cnt[kSortKeys];
    hub_runs(p, [&](int hub, int32_t, int64_t b, int64_t e) {
        for (int k = threadIdx.x; k < kSortKeys; k += kBlock) cnt[k] = 0;
        __syncthreads();
        for (int64_t i = b + threadIdx.x; i < e; i += kBlock)
            atomicAdd(&cnt[sort_key(g.wt[i], shift)], 1u);
        __syncthreads();
        for (int k = threadIdx.x; k < kSortKeys; k += kBlock)
            if (cnt[k]) atomicAdd(&hist[(size_t)hub * kSortKeys + k], cnt[k]);
        __syncthreads();
    });
}

// Exclusive scan of each hub's keys (a workgroup of kSortKeys threads each).
__global__ __launch_bounds__(kSortKeys) void sort_hub_scan_kernel(int hubs, uint32_t *hist) {
    __shared__ uint32_t s[kSortKeys];
    for (int h = blockIdx.x; h < hubs; h += gridDim.x) {
        const uint32_t v = hist[(size_t)h * kSortKeys + threadIdx.x];
        s[threadIdx.x] = v;
        __syncthreads();
        for (int d = 1; d < kSortKeys; d <<= 1) {
            const uint32_t o = (int)threadIdx.x >= d ? s[threadIdx.x - d] : 0u;
            __syncthreads();
            s[threadIdx.x] += o;
            __syncthreads();
        }
        hist[(size_t)h * kSortKeys + threadIdx.x] = s[threadIdx.x] - v;
        __syncthreads();
    }
}

// Each run reserves its place in every key from the hub's cursors and writes
// its edges there.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void sort_hub_scatter_kernel(PlanDev p, GraphView<OffT> g,
                                                                  int2 *out, int shift,
                                                                  uint32_t *cursor) {
    __shared__ uint32_t cnt[kSortKeys];
    hub_runs(p, [&](int hub, int32_t u, int64_t b, int64_t e) {
        const int64_t row = (int64_t)g.rbeg(u);
        for (int k = threadIdx.x; k < kSortKeys; k += kBlock) cnt[k] = 0;
        __syncthreads();
        for (int64_t i = b + threadIdx.x; i < e; i += kBlock)
            atomicAdd(&cnt[sort_key(g.wt[i], shift)], 1u);
        __syncthreads();
        for (int k = threadIdx.x; k < kSortKeys; k += kBlock)
            cnt[k] = cnt[k] ? atomicAdd(&cursor[(size_t)hub * kSortKeys + k], cnt[k]) : 0u;
        __syncthreads();
        for (int64_t i = b + threadIdx.x; i < e; i += kBlock) {
            const int32_t w = g.wt[i];
            const uint32_t at = atomicAdd(&cnt[sort_key(w, shift)], 1u);
            out[row + at] = int2{g.adj[i], w};
        }
        __syncthreads();
    });
}

template <typename OffT>
static int build_sorted(hc_graph_s *g, hipStream_t s, SortedAdj *out) {
    const PlanHost *ph = nullptr;
    HC_TRY(get_plan(g, 0, g->n, sorted_plan_config(), &ph));
    const PlanDev &p = ph->dev;
    int shift = 0;
    while ((g->max_weight >> shift) >= kSortKeys) shift++;
    // The pairs, then the hubs' key counts (used by the build only).
    const size_t hwords = (size_t)p.num_hubs * kSortKeys;
    int2 *e = nullptr;
    if (hipMalloc(reinterpret_cast<void **>(&e),
                  sizeof(int2) * (size_t)g->m + sizeof(uint32_t) * hwords) != hipSuccess) {
        (void)hipGetLastError();
        return HC_OK;  // the sweeps run on the plain CSR
    }
    uint32_t *hist = reinterpret_cast<uint32_t *>(e + g->m);
    const GraphView<OffT> v = view<OffT>(g);
    const int grid = grid_blocks();
    if (hwords) {
        sort_zero_kernel<<<std::min<size_t>(grid, (hwords + 255) / 256), 256, 0, s>>>(hist, hwords);
        const int hg = std::min(grid, (p.cnt[0] + kSortRun - 1) / kSortRun);
        sort_hub_count_kernel<OffT><<<hg, kBlock, 0, s>>>(p, v, shift, hist);
        sort_hub_scan_kernel<<<std::min(grid, p.num_hubs), kSortKeys, 0, s>>>(p.num_hubs, hist);
        sort_hub_scatter_kernel<OffT><<<hg, kBlock, 0, s>>>(p, v, e, shift, hist);
    }
    if (ph->total_units > p.unit_start[2]) sort_rows_kernel<OffT><<<grid, kBlock, 0, s>>>(p, v, e, shift);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
        (void)hipFree(e);
        return fail(HC_ERR_HIP, "weight-sorted adjacency build failed");
    }
    out->e = e;
    out->shift = shift;
    return HC_OK;
}

int get_sorted(hc_graph_s *g, hipStream_t s, SortedView *out) {
    *out = SortedView{nullptr, 0};
    if (!g->weighted || g->m <= 0 || g->row0 != 0 || g->rows != g->n || g->max_degree > INT32_MAX)
        return HC_OK;
    SortedSlot &slot = *g->sortslot;
    std::lock_guard<std::mutex> lk(slot.mu);
    if (!slot.adj.e)
        HC_TRY(g->off64 ? build_sorted<uint64_t>(g, s, &slot.adj)
                        : build_sorted<uint32_t>(g, s, &slot.adj));
    *out = SortedView{slot.adj.e, slot.adj.shift};
    return HC_OK;
}

}  // namespace hc
