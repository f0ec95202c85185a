// A whole direction-optimizing BFS of one graph by one workgroup, its bitmaps in
// LDS (or in a global slot): the body of the many-graph launch (many.hip) and of
// the single-graph runs on small graphs (bfs.hip).
#pragma once

#include "frontier.h"

// A graph of a batch (of one, for a single-graph run).
struct Desc {
    int64_t node_base;  // first vertex of the graph in the batch
    int64_t off_base;   // first offset (node_base + graph index)
    int64_t edge_base;  // first adjacency entry
    int32_t n;
    int32_t pad;
    int64_t m;
};

namespace hc {

struct ManyStats {
    unsigned long long pushes, pulls, scanned;
};

// Bitmap word read: LDS bitmaps are read directly; global ones bypass the
// per-CU cache, since other waves of the workgroup update them with
// device-memory atomics.
template <bool Global>
__device__ __forceinline__ uint32_t bm_word(const uint32_t *b, int32_t w) {
    if (Global) return __hip_atomic_load(&b[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return b[w];
}

template <bool Global>
__device__ __forceinline__ bool bm_get(const uint32_t *b, int32_t v) {
    return (bm_word<Global>(b, v >> 5) >> (v & 31)) & 1u;
}

// Claims v in the visited bitmap; true for exactly one caller.
template <bool Global>
__device__ __forceinline__ bool bm_claim(uint32_t *b, int32_t v) {
    const uint32_t bit = 1u << (v & 31);
    if (bm_word<Global>(b, v >> 5) & bit) return false;
    return !(atomicOr(&b[v >> 5], bit) & bit);
}

// Block-wide sum of a per-thread 64-bit value (result valid in all threads).
template <int BLOCK>
__device__ __forceinline__ long long many_block_sum(long long v, long long *s_red) {
#pragma unroll
    for (int s = kWave / 2; s > 0; s >>= 1) v += __shfl_xor(v, s, kWave);
    __syncthreads();
    if (lane_id() == 0) s_red[threadIdx.x / kWave] = v;
    __syncthreads();
    long long t = 0;
#pragma unroll
    for (int i = 0; i < BLOCK / kWave; i++) t += s_red[i];
    return t;
}

// Top-down expansion of u's edges [b, e), G lanes (this one is `lane`), four
// edges a lane in flight.
template <int G, bool Global>
__device__ __forceinline__ void expand(const uint32_t *__restrict__ off,
                                       const int32_t *__restrict__ adj,
                                       int32_t *__restrict__ depth, int32_t *__restrict__ parents,
                                       uint32_t *vis, uint32_t *next, int level, int32_t u,
                                       uint32_t b, uint32_t e, int lane, long long &cnt,
                                       long long &sc) {
    for (uint32_t i = b + lane; i < e; i += 4 * G) {
        int32_t v[4];
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = i + r * G < e ? adj[i + r * G] : -1;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (v[r] < 0 || !bm_claim<Global>(vis, v[r])) continue;
            atomicOr(&next[v[r] >> 5], 1u << (v[r] & 31));
            depth[v[r]] = level;
            if (parents) parents[v[r]] = u;
            cnt++;
            sc += off[v[r] + 1] - off[v[r]];
        }
    }
}

// One direction-optimizing BFS of graph d from src by the whole workgroup;
// bm holds three bitmaps of `words` words (LDS, or a global slot when
// Global).  Frontier vertices of degree above light_deg are expanded by
// whole wavefronts, up to heavy_cap of them per level.
// TRACE: the levels are recorded in `trace` as the epoch loop records its
// epochs, and its totals set (single-graph runs).
template <int BLOCK, bool Global, bool TRACE = false>
__device__ __forceinline__ void bfs_one_graph(const Desc &d, int32_t src,
                              const uint32_t *__restrict__ off,
                              const int32_t *__restrict__ adj, int32_t *__restrict__ depth,
                              int32_t *__restrict__ parents, uint32_t *bm, int words,
                              int alpha, int beta, int light_deg, int heavy_cap,
                              int32_t *heavy, int *s_nheavy, long long *s_red, ManyStats &st,
                              StepCtl *trace = nullptr) {
    const int tid = threadIdx.x;
    long long t_start = 0;
    if (TRACE) t_start = wall_clock64();
    unsigned long long bytes = 0, reached = 1;
    const int n = d.n;
    uint32_t *vis = bm;
    uint32_t *front = bm + words;
    uint32_t *next = bm + 2 * words;
    for (int i = tid; i < 3 * words; i += BLOCK) bm[i] = 0;
    for (int u = tid; u < n; u += BLOCK) {
        depth[u] = -1;
        if (parents) parents[u] = -1;
    }
    __syncthreads();
    if (tid == 0) {
        vis[src >> 5] |= 1u << (src & 31);
        front[src >> 5] |= 1u << (src & 31);
        depth[src] = 0;
        if (parents) parents[src] = src;
    }
    __syncthreads();
    long long edges_to_check = d.m;
    long long scout = (long long)(off[src + 1] - off[src]);
    long long num_nodes = 1, prev_nodes = 0;
    bool pull = false;
    // Initial decision (bfs_do_cpu: num_edges = deg(src)).
    if (scout > edges_to_check / alpha) {
        pull = true;
    } else {
        edges_to_check -= scout;
    }
    long long fsize = 1;
    int level = 0;
    while (fsize > 0) {
        level++;
        long long cnt = 0, sc = 0, scanned = 0;
        if (!pull) {
            // Top-down: threads take frontier words; light vertices are
            // expanded by their thread, heavy ones queued for whole waves.
            if (tid == 0) *s_nheavy = 0;
            __syncthreads();
            for (int w = tid; w < words; w += BLOCK) {
                uint32_t bits = bm_word<Global>(front, w);
                while (bits) {
                    const int32_t u = w * 32 + __ffs(bits) - 1;
                    bits &= bits - 1;
                    const uint32_t b = off[u], e = off[u + 1];
                    if (e - b > (uint32_t)light_deg) {
                        const int slot = atomicAdd(s_nheavy, 1);
                        if (slot < heavy_cap) {
                            heavy[slot] = u;
                            continue;
                        }
                    }
                    scanned += e - b;
                    expand<1, Global>(off, adj, depth, parents, vis, next, level, u, b, e, 0, cnt,
                                      sc);
                }
            }
            __syncthreads();
            const int nh = min(*s_nheavy, heavy_cap);
            const int wave = tid / kWave, nwaves = BLOCK / kWave, lane = lane_id();
            for (int h = wave; h < nh; h += nwaves) {
                const int32_t u = heavy[h];
                const uint32_t b = off[u], e = off[u + 1];
                if (lane == 0) scanned += e - b;
                expand<kWave, Global>(off, adj, depth, parents, vis, next, level, u, b, e, lane,
                                      cnt, sc);
            }
            st.pushes += (tid == 0);
        } else {
            // Bottom-up: every unvisited vertex takes its first neighbour
            // (CSR order) in the frontier.
            // kRows vertices a thread at once: their bounds, then their first
            // neighbours, are in flight together (one workgroup runs the
            // graph, so the level waits on these chains: 512 graphs, 507 ->
            // 388 us with this and four edges in flight below).
            constexpr int kRows = 8;
            for (int u0 = tid; u0 < n; u0 += kRows * BLOCK) {
                uint32_t rb[kRows], re[kRows];
                int32_t f[kRows];
#pragma unroll
                for (int k = 0; k < kRows; k++) {
                    const int u = u0 + k * BLOCK;
                    const bool open = u < n && !bm_get<Global>(vis, u);
                    rb[k] = open ? off[u] : 0u;
                    re[k] = open ? off[u + 1] : 0u;
                }
#pragma unroll
                for (int k = 0; k < kRows; k++) f[k] = rb[k] < re[k] ? adj[rb[k]] : -1;
#pragma unroll
                for (int k = 0; k < kRows; k++) {
                    if (f[k] < 0) continue;
                    const int u = u0 + k * BLOCK;
                    int32_t par = -1;
                    scanned++;
                    if (bm_get<Global>(front, f[k])) par = f[k];
                    for (uint32_t i = rb[k] + 1; par < 0 && i < re[k]; i += 4) {
                        int32_t v[4];
#pragma unroll
                        for (int r = 0; r < 4; r++) v[r] = i + r < re[k] ? adj[i + r] : -1;
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            if (par >= 0 || v[r] < 0) continue;
                            scanned++;
                            if (bm_get<Global>(front, v[r])) par = v[r];
                        }
                    }
                    if (par >= 0) {
                        atomicOr(&vis[u >> 5], 1u << (u & 31));
                        atomicOr(&next[u >> 5], 1u << (u & 31));
                        depth[u] = level;
                        if (parents) parents[u] = par;
                        cnt++;
                        sc += re[k] - rb[k];
                    }
                }
            }
            st.pulls += (tid == 0);
        }
        const long long q = many_block_sum<BLOCK>(cnt, s_red);
        const long long scq = many_block_sum<BLOCK>(sc, s_red);
        st.scanned += (unsigned long long)scanned;
        if (TRACE) {
            const long long ex = many_block_sum<BLOCK>(scanned, s_red);
            // (the epoch loop's byte counts, with 4-byte offsets)
            bytes += pull ? 4ull * n + 4ull * ex + ex / 8 + 12ull * q + 4ull * words
                          : 12ull * fsize + 8ull * ex + 16ull * q;
            reached += q;
            if (tid == 0 && level <= kTraceLen) {
                trace->tr_t[level - 1] = wall_clock64();
                trace->tr_mode[level - 1] = (int8_t)(pull ? kPull : kPush);
                trace->tr_n[level - 1] = (uint32_t)q;
                trace->tr_e[level - 1] = (unsigned long long)scq;
                trace->tr_scan[level - 1] = (unsigned long long)ex;
            }
        }
        // Next level's frontier; clear the old one for reuse.
        uint32_t *t = front;
        front = next;
        next = t;
        for (int i = tid; i < words; i += BLOCK) next[i] = 0;
        fsize = q;
        // bfs_do_cpu's switching rule, evaluated identically by all threads.
        if (!pull) {
            scout = scq;
            if (q > 0) {
                if (scout > edges_to_check / alpha) {
                    pull = true;
                    num_nodes = q;
                } else {
                    edges_to_check -= scout;
                }
            }
        } else {
            prev_nodes = num_nodes;
            num_nodes = q;
            if (!(q > prev_nodes || q > n / beta)) {
                scout = 1;
                if (q > 0) {
                    if (scout > edges_to_check / alpha) {
                        num_nodes = q;
                    } else {
                        pull = false;
                        edges_to_check -= scout;
                    }
                }
            }
        }
        __syncthreads();
    }
    if (TRACE && tid == 0) {
        trace->t_start = t_start;
        trace->t_end = wall_clock64();
        trace->epoch = level;
        trace->push_epochs = (int32_t)st.pushes;
        trace->pull_epochs = (int32_t)st.pulls;
        trace->reached = reached;
        trace->alg_bytes = bytes;
        trace->done = 1;
        trace[0].steps = 1;
        trace[1].steps = 0;
    }
}

}  // namespace hc
