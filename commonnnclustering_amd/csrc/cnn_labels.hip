// Phases S and U: common-neighbour similarity, union-find labelling, sort_by_size.
//
// Replaces FitterExtBFS._fit (_fit.pyx:408-491) with its connected-components
// equivalent: core(i) = consider(i) && |N(i)| > m_core (_types.pyx:1561-1564);
// edge(i, j) = core(i) && core(j) && j in N(i) && |N(i) & N(j)| >= c_sim
// (SimilarityCheckerExtScreensorted._check, _types.pyx:2654-2706, early exit at
// c_sim).  The BFS opens clusters in ascending init-point order and never
// reaches an earlier cluster through a valid edge, so its labels are the
// components of (core points, edges) numbered by smallest point index; a
// union-find whose links always point from the larger to the smaller root
// yields the same partition regardless of scheduling.
//
// Work plan on the GPU (all on the context stream):
//   k_init      core flags, parent[i] = i, cleared component arrays
//   k_hook_tile each core row tests its two nearest smaller-index core
//               neighbours of its own tile and hooks its parent to one that
//               passes (a forest, no atomics); k_hook_queue tests the rows with
//               fewer in the tiles below (k_hook: per row, without tile words)
//   k_compress_roots, k_hook_roots_list  (lists only) flatten; roots re-point
//               at a smaller neighbouring root on a pass
//   k_root_count, k_snapshot  rank[i] = (component size << 32 | root) of core
//               points, and the tiles' largest and common ranks
//   k_round_tile every edge between different snapshot components is tested by
//               the endpoint of lower rank, unless the endpoints were joined
//               meanwhile; rows that own no edge are skipped by a per-tile bound
//               (k_round_b: per row, without tile words)
//   k_comp_stats flatten, component statistics; label assignment / sort_by_size
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <memory>

#include "cnn_internal.hpp"

namespace cnn {

// ------------------------------------------------------------------ union-find

__device__ __forceinline__ int uf_find(int *parent, int x) {
    int p = atomic_load_relaxed(&parent[x]);
    while (p != x) {
        int gp = atomic_load_relaxed(&parent[p]);
        if (gp == p) return p;
        __hip_atomic_store(&parent[x], gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // path halving
        x = gp;
        p = atomic_load_relaxed(&parent[x]);
    }
    return x;
}

// Link the larger root below the smaller one (parent[x] <= x always holds).
__device__ __forceinline__ void uf_union(int *parent, int a, int b) {
    for (;;) {
        a = uf_find(parent, a);
        b = uf_find(parent, b);
        if (a == b) return;
        if (a < b) { int t = a; a = b; b = t; }
        int old = atomicCAS(&parent[a], a, b);
        if (old == a) return;
    }
}

// ------------------------------------------------------------------ similarity

constexpr int kStatSlots = 1024;  // striped counters: no same-address atomic hot spot

struct LabelArgs {
    const int64_t *row_ptr;
    const int32_t *col;
    int64_t n;
    int c_sim;
    int m_core;
    uint8_t *core;
    int *parent;
    unsigned long long *stats;  // per slot: tests, passed, rows scanned, sampled components
    const uint64_t *rank;       // snapshot rank of core points: (component size << 32) | root; 0 otherwise
    const uint64_t *cand_max;   // per row tile: max rank over its candidate tiles (nullable)
    // per tile: the rank every point of the tile has (0: no core point; all
    // ones: ranks differ), so list entries in such tiles need no rank gather
    const uint64_t *tile_rank;
    const int32_t *selfpos;     // per row: position of its own index in its list (nullable)
    const int32_t *tile_csim;   // packed batches: c_sim / m_core per row tile (nullable)
    const int32_t *tile_mcore;
    // the lists as row words: per candidate tile pair of a spatial graph
    // (mask / pair_nz over tp_ptr / tp_col), or per row (wptr / wtile / wword)
    const uint64_t *mask;
    const uint8_t *pair_nz;
    const int64_t *tp_ptr;
    const int32_t *tp_col;
    const int64_t *wptr;
    const int32_t *wtile;
    const uint64_t *wword;
    const int32_t *diag;  // per row tile: its own pair's place in its list (nullable)
    // per-row degrees (nullable: row_ptr differences); word-only passes need no row_ptr
    const int32_t *deg;
    // several cutoff pairs in one launch, one per blockIdx.y (nullable: one
    // pair, c_sim / m_core): launch y takes csim_y[y] / mcore_y[y] and its own
    // slices of the per-point (stride n), per-tile (stride tiles) and
    // statistics arrays (see slice)
    const int32_t *csim_y;
    const int32_t *mcore_y;
    int64_t tiles;
    // tile pairs k_round_tile hands to k_round_queue: {row tile, position in its list}
    int2 *rq;
    unsigned long long *rq_len;
    int64_t rq_cap;
    // the row tiles in the order the per-tile kernels take them: heavy ones
    // first (nullable: ascending)
    const int32_t *tile_order;
};

// The cutoff pair of this launch's blockIdx.y and its slices of the
// per-pair arrays; unchanged for a single pair.
__device__ __forceinline__ LabelArgs slice(LabelArgs a) {
    if (!a.csim_y) return a;
    const int64_t y = blockIdx.y;
    a.core += y * a.n;
    a.parent += y * a.n;
    a.rank += y * a.n;
    a.stats += y * 4 * kStatSlots;
    if (a.rq) {
        a.rq += y * a.rq_cap;
        a.rq_len += y;
    }
    if (a.cand_max) a.cand_max += y * a.tiles;
    if (a.tile_rank) a.tile_rank += y * a.tiles;
    a.c_sim = a.csim_y[y];
    a.m_core = a.mcore_y[y];
    return a;
}

__device__ __forceinline__ int64_t deg_of(const LabelArgs &a, int64_t w) {
    return a.deg ? (int64_t)a.deg[w] : a.row_ptr[w + 1] - a.row_ptr[w];
}

// Row w's words: its row of the candidate tile pairs of its row tile (spatial
// graph masks), or its own word list.
__device__ __forceinline__ WordRow word_row(const LabelArgs &a, int64_t w) {
    WordRow r;
    if (a.mask) {
        const int64_t R = w >> 6;
        const int64_t kb = a.tp_ptr[R];
        r.tile = a.tp_col + kb;
        r.word = a.mask + kb * 64 + (w & 63);
        r.nz = a.pair_nz + kb;
        r.len = a.tp_ptr[R + 1] - kb;
        r.stride = 64;
    } else {
        const int64_t b = a.wptr[w];
        r.tile = a.wtile + b;
        r.word = a.wword + b;
        r.nz = nullptr;
        r.len = a.wptr[w + 1] - b;
        r.stride = 1;
    }
    return r;
}

__device__ __forceinline__ int csim_of(const LabelArgs &a, int64_t w) {
    return a.tile_csim ? a.tile_csim[w >> 6] : a.c_sim;
}

__device__ __forceinline__ void add_stats(const LabelArgs &a, unsigned tests, unsigned passed, unsigned rows = 0,
                                          unsigned roots = 0) {
    if ((threadIdx.x & 63) == 0 && (tests || rows || roots)) {
        const unsigned slot = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (kStatSlots - 1);
        if (tests) {
            atomicAdd(&a.stats[4 * slot], (unsigned long long)tests);
            atomicAdd(&a.stats[4 * slot + 1], (unsigned long long)passed);
        }
        if (rows) atomicAdd(&a.stats[4 * slot + 2], (unsigned long long)rows);
        if (roots) atomicAdd(&a.stats[4 * slot + 3], (unsigned long long)roots);
    }
}

// Per-component arrays cleared by k_init (each nullable; one slice per cutoff pair).
struct ComponentArrays {
    int32_t *cnt;     // sampled component sizes: 0
    int32_t *cmin;    // smallest caller index: INT_MAX
    int32_t *csize;   // final component sizes: 0
    int32_t *newlab;  // sort_by_size labels: 0
};

__global__ void k_init(LabelArgs a, const uint8_t *__restrict__ consider, const int32_t *__restrict__ perm,
                       ComponentArrays ca, ClearList clear) {
    if (blockIdx.y == 0) {
        const int64_t step = (int64_t)gridDim.x * blockDim.x;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < clear.count[q]; t += step)
                clear.p[q][t] = 0ull;
    }
    a = slice(a);
    int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= a.n) return;
    const int64_t deg = deg_of(a, w);
    const int m_core = a.tile_mcore ? a.tile_mcore[w >> 6] : a.m_core;
    const int32_t o = perm ? perm[w] : (int32_t)w;  // -1: padding row of a packed batch
    bool ok = deg > (int64_t)m_core && o >= 0;
    if (consider && ok) ok = consider[o] != 0;
    a.core[w] = ok ? 1 : 0;
    a.parent[w] = (int)w;
    const int64_t at = (int64_t)blockIdx.y * a.n + w;
    ca.cnt[at] = 0;
    ca.cmin[at] = INT_MAX;
    ca.csize[at] = 0;
    if (ca.newlab) ca.newlab[at] = 0;
}

// Test edge (w, j) unless the endpoints are already joined; link on a pass.
// Returns true when w and j are in one component afterwards.
__device__ __forceinline__ bool test_and_link(const LabelArgs &a, int w, int j, int64_t bw, int64_t ew, int c,
                                              unsigned &tests, unsigned &passed) {
    const int rw = uf_find(a.parent, w);
    const int rj = uf_find(a.parent, j);
    if (rw == rj) return true;
    const int64_t bj = a.row_ptr[j], ej = a.row_ptr[j + 1];
    const bool pass = wave_sim(a.col + bw, ew - bw, a.col + bj, ej - bj, c);
    ++tests;
    if (pass) {
        ++passed;
        if (__lane_id() == 0) uf_union(a.parent, w, j);
    }
    return pass;
}

// The same on row words (bitset similarity); A is w's word row, dw its degree.
__device__ __forceinline__ bool test_and_link_words(const LabelArgs &a, int w, int j, const WordRow &A, int64_t dw,
                                                    int c, unsigned &tests, unsigned &passed) {
    const int rw = uf_find(a.parent, w);
    const int rj = uf_find(a.parent, j);
    if (rw == rj) return true;
    const int64_t dj = deg_of(a, j);
    const bool pass = dw >= c && dj >= c && wave_sim_words(A, word_row(a, j), c);
    ++tests;
    if (pass) {
        ++passed;
        if (__lane_id() == 0) uf_union(a.parent, w, j);
    }
    return pass;
}

__device__ __forceinline__ uint64_t lane_bit_mask(int lane) { return 1ull << lane; }

// Sampling round (hooking): each core row tests its nearest smaller-index core
// neighbours in list order (the previous points of the working order, which
// are spatially closest) and points its parent at the first one that passes.
// Every row writes only its own parent entry and parents have smaller
// indices, so the hooks form a forest whose trees are the components of the
// passing edges tested here -- no atomics, no contention.
// Hooking of one core row on row words: its smaller-index neighbours in
// descending order, at most max_tests tests; below_own: those of its own tile
// were tested already (k_hook_tile), only the tiles below it are searched.
__device__ __forceinline__ void hook_row_words(const LabelArgs &a, int64_t w, int max_tests, bool below_own) {
    const int lane = threadIdx.x & 63;
    const int64_t dw = deg_of(a, w);
    // the row's words from its own tile down, 64 tiles a step (lane l holds
    // the l-th tile below the window's top), bits from the highest down:
    // smaller indices, nearest first
    const WordRow A = word_row(a, w);
    const int Rw = (int)(w >> 6);
    int64_t top = 0;  // tiles up to and including the row's own tile (below_own: below it)
    if (a.mask && a.diag && a.diag[Rw] >= 0) {
        top = a.diag[Rw] + (below_own ? 0 : 1);  // recorded when the lists were built
    } else {
        const int last = below_own ? Rw - 1 : Rw;
        for (int64_t t0 = 0; t0 < A.len; t0 += 64) {
            const int64_t t = t0 + lane;
            const uint64_t le = __ballot(t < A.len && A.tile[t] <= last);
            top += __popcll(le);
            if (__popcll(le) < 64) break;
        }
    }
    const int c = csim_of(a, w);
    unsigned tests = 0, passed = 0;
    int attempts = 0;
    bool done = false;
    for (int64_t t1 = top; t1 > 0 && attempts < max_tests && !done; t1 -= 64) {
        const int64_t t = t1 - 1 - lane;
        uint64_t v = 0ull;
        int C = 0;
        if (t >= 0) {
            C = A.tile[t];
            v = word_at(A, t);
            if (C == Rw) v &= lane_bit_mask((int)(w & 63)) - 1ull;  // smaller indices only
        }
        uint64_t tiles = __ballot(v != 0ull);
        while (tiles && attempts < max_tests && !done) {
            const int src = __ffsll((unsigned long long)tiles) - 1;
            tiles &= tiles - 1;
            const uint32_t vlo = __builtin_amdgcn_readlane((uint32_t)v, src);
            const uint32_t vhi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), src);
            const int Cs = __builtin_amdgcn_readlane(C, src);
            const bool bit = ((lane < 32 ? vlo >> lane : vhi >> (lane - 32)) & 1u) != 0u;
            uint64_t bits = __ballot(bit && a.core[Cs * 64 + lane]);
            while (bits && attempts < max_tests) {
                const int hb = 63 - __clzll((long long)bits);
                bits &= ~lane_bit_mask(hb);
                const int jj = Cs * 64 + hb;
                ++attempts;
                ++tests;
                const int64_t dj = deg_of(a, jj);
                if (dw >= c && dj >= c && wave_sim_words(A, word_row(a, jj), c)) {
                    ++passed;
                    if (lane == 0) a.parent[w] = jj;
                    done = true;
                    break;
                }
            }
        }
    }
    add_stats(a, tests, passed);
}

template <bool WORDS>
__global__ __launch_bounds__(256) void k_hook(LabelArgs a, int max_tests) {
    a = slice(a);
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= a.n || !a.core[w]) return;
    const int64_t b = a.row_ptr[w], e = a.row_ptr[w + 1];
    if constexpr (WORDS) {
        hook_row_words(a, w, max_tests, false);
        return;
    }
    // first entry >= w: the row's own entry, recorded when the lists were
    // emitted, or a 64-way search (each step probes 64 evenly spaced entries at
    // once and keeps the gap that holds the boundary)
    int64_t lo = a.selfpos ? min(b + (int64_t)a.selfpos[w], e) : b, hi = a.selfpos ? lo : e;
    while (lo < hi) {
        const int64_t step = (hi - lo + 63) >> 6;
        const int64_t pos = lo + lane * step;
        const bool below = pos < hi && a.col[pos] < (int32_t)w;
        const int cnt = __popcll(__ballot(below));  // probes 0 .. cnt-1 lie below w
        const int64_t nlo = cnt > 0 ? lo + (int64_t)(cnt - 1) * step + 1 : lo;
        const int64_t nhi = min(hi, lo + (int64_t)cnt * step);
        lo = nlo;
        hi = nhi;
    }
    unsigned tests = 0, passed = 0;
    int attempts = 0;
    // entries [b, lo) are the smaller indices, nearest first when walked backwards
    for (int64_t t1 = lo; t1 > b && attempts < max_tests; t1 -= 64) {
        const int64_t t = t1 - 1 - lane;
        const int j = t >= b ? a.col[t] : -1;
        uint64_t bits = __ballot(t >= b && a.core[j]);
        bool done = false;
        while (bits && attempts < max_tests) {
            const int src = __ffsll((unsigned long long)bits) - 1;
            bits &= bits - 1;
            const int jj = __shfl(j, src, 64);
            if (jj >= (int)w) continue;  // parents point to smaller indices only: the hooks stay a forest
            const int64_t bj = a.row_ptr[jj], ej = a.row_ptr[jj + 1];
            ++attempts;
            ++tests;
            if (wave_sim(a.col + b, e - b, a.col + bj, ej - bj, csim_of(a, w))) {
                ++passed;
                if (lane == 0) a.parent[w] = jj;
                done = true;
                break;
            }
        }
        if (done) break;
    }
    add_stats(a, tests, passed);
}

// Hooking within row tiles on tile-pair words: one wave per row tile, lane r =
// row w = 64R + r.  A core row tests its two nearest smaller-index core
// neighbours of its own tile.  Rows of one tile share the tile's candidate
// list, and pair k's 64 row words are contiguous (lane r reads row r's word),
// so one pass over the tile's non-empty pairs counts |N(w) & N(j)| of both
// candidates for all 64 rows at once (row j's word comes from lane j).  The
// own pair is read first: it names the candidates.  The pass stops once every
// row has a candidate with c_sim common neighbours.  A row hooks to the first
// row of its chain of hooked rows within the tile: only own entries are
// written, to smaller indices (a forest).  Core rows that had fewer than two
// candidates and no pass go to a queue (2 w + tests made) for k_hook_queue;
// one counter update per workgroup (a single address: per-wave updates took
// about 100 us for 21,000 tiles).
__global__ __launch_bounds__(256) void k_hook_tile(LabelArgs a, int64_t n_tiles, uint32_t *__restrict__ queue,
                                                   unsigned int *__restrict__ queue_len) {
    a = slice(a);
    queue += (int64_t)blockIdx.y * a.n;
    queue_len += blockIdx.y;
    __shared__ unsigned s_len[4], s_base;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t gR = (int64_t)blockIdx.x * 4 + wave;
    const bool valid = gR < n_tiles;
    const int64_t R = !valid ? 0 : a.tile_order ? (int64_t)a.tile_order[gR] : gR;
    const int64_t w = R * 64 + lane;
    const bool core_w = valid && w < a.n && a.core[w] != 0;
    const uint64_t cores = __ballot(core_w);
    bool hooked = false;
    int n_cand = 0;
    unsigned tests = 0, passed = 0;
    if (cores & (cores - 1)) {  // at least two core rows
        const int c = csim_of(a, R * 64);
        const int64_t kb = a.tp_ptr[R], ke = a.tp_ptr[R + 1];
        // the tile's own pair: recorded when the lists were built, or found by
        // a ballot per 64 of its ascending column tiles
        int64_t kd = -1;
        if (a.diag && a.diag[R] >= 0) kd = kb + a.diag[R];
        for (int64_t k0 = kb; k0 < ke && kd < 0; k0 += 64) {
            const int64_t kk = k0 + lane;
            const uint64_t hit = __ballot(kk < ke && a.tp_col[kk] == (int)R);
            if (hit) kd = k0 + __ffsll((unsigned long long)hit) - 1;
        }
        uint64_t own = 0ull;
        if (kd >= 0 && a.pair_nz[kd] != 0) own = a.mask[kd * 64 + lane];
        const uint64_t cand = core_w ? own & cores & ((1ull << lane) - 1ull) : 0ull;
        const int j1 = cand ? 63 - __clzll((long long)cand) : lane;
        const uint64_t rest = cand & ~(1ull << j1);
        const int j2 = rest ? 63 - __clzll((long long)rest) : j1;
        n_cand = cand ? (rest ? 2 : 1) : 0;
        int cnt1 = __popcll(own & __shfl(own, j1, 64)), cnt2 = __popcll(own & __shfl(own, j2, 64));
        bool done = __ballot(n_cand && cnt1 < c && cnt2 < c) == 0ull;
        for (int64_t k0 = kb; k0 < ke && !done; k0 += 64) {
            // the window's other non-empty pairs, then their words 8 at a time (loads in flight together)
            const int64_t kk = k0 + lane;
            const bool nzl = kk < ke && kk != kd && a.pair_nz[kk] != 0;
            uint64_t nzm = __ballot(nzl);
            while (nzm && !done) {
                int idx[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    idx[u] = nzm ? __ffsll((unsigned long long)nzm) - 1 : -1;
                    nzm &= nzm - 1;
                }
                uint64_t v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = idx[u] >= 0 ? a.mask[(k0 + idx[u]) * 64 + lane] : 0ull;
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    cnt1 += __popcll(v[u] & __shfl(v[u], j1, 64));
                    cnt2 += __popcll(v[u] & __shfl(v[u], j2, 64));
                }
                if (__ballot(n_cand && cnt1 < c && cnt2 < c) == 0ull) done = true;
            }
        }
        hooked = n_cand && (cnt1 >= c || cnt2 >= c);
        int p = hooked ? (cnt1 >= c ? j1 : j2) : lane;
#pragma unroll
        for (int step = 0; step < 6; ++step) p = __shfl(p, p, 64);  // to the head of the chain
        if (hooked) a.parent[w] = (int)(R * 64 + p);
        tests = (unsigned)(__popcll(__ballot(n_cand > 0)) + __popcll(__ballot(n_cand > 1)));
        passed = (unsigned)__popcll(__ballot(hooked));
    }
    // core rows left to the per-row hooking
    const bool left = core_w && !hooked && n_cand < 2;
    const uint64_t lm = __ballot(left);
    if (lane == 0) s_len[wave] = (unsigned)__popcll(lm);
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned total = s_len[0] + s_len[1] + s_len[2] + s_len[3];
        s_base = total ? atomicAdd(queue_len, total) : 0u;
    }
    __syncthreads();
    if (left) {
        unsigned base = s_base;
        for (int q = 0; q < wave; ++q) base += s_len[q];
        queue[base + __popcll(lm & ((1ull << lane) - 1ull))] = (uint32_t)w * 2u + (uint32_t)n_cand;
    }
    add_stats(a, tests, passed);
}

// Per-row hooking of the rows k_hook_tile left (a queue; grid-stride, one wave
// per row): up to max_tests tests in all, in the tiles below the row's own.
__global__ __launch_bounds__(256) void k_hook_queue(LabelArgs a, const uint32_t *__restrict__ queue,
                                                    const unsigned int *__restrict__ queue_len, int max_tests) {
    a = slice(a);
    queue += (int64_t)blockIdx.y * a.n;
    queue_len += blockIdx.y;
    const unsigned nq = *queue_len;
    const int64_t waves = (int64_t)gridDim.x * 4;
    for (int64_t q = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); q < (int64_t)nq; q += waves) {
        const uint32_t e = queue[q];
        hook_row_words(a, (int64_t)(e >> 1), max_tests - (int)(e & 1u), true);
    }
}

// Root hooking: a core point that is still a root tests core neighbours whose
// current root is smaller than itself (either side of it in the list) and
// re-points itself at that root on the first pass.  Only roots write their own
// entry and only to smaller values, so the parents stay a forest.
template <bool WORDS>
__device__ void hook_root(const LabelArgs &a, int64_t w, int max_tests) {
    const int lane = threadIdx.x & 63;
    unsigned tests = 0, passed = 0;
    int attempts = 0;
    if constexpr (WORDS) {
        const int64_t dw = deg_of(a, w);
        const WordRow A = word_row(a, w);
        const int c = csim_of(a, w);
        bool done = false;
        for (int64_t t0 = 0; t0 < A.len && attempts < max_tests && !done; t0 += 64) {
            const int64_t t = t0 + lane;
            uint64_t v = 0ull;
            int C = 0;
            if (t < A.len) {
                v = word_at(A, t);
                C = A.tile[t];
            }
            uint64_t tiles = __ballot(v != 0ull);
            while (tiles && attempts < max_tests && !done) {
                const int src = __ffsll((unsigned long long)tiles) - 1;
                tiles &= tiles - 1;
                const uint32_t vlo = __builtin_amdgcn_readlane((uint32_t)v, src);
                const uint32_t vhi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), src);
                const int Cs = __builtin_amdgcn_readlane(C, src);
                const bool bit = ((lane < 32 ? vlo >> lane : vhi >> (lane - 32)) & 1u) != 0u;
                const int j = Cs * 64 + lane;
                // the parent loads with the core flag (parents are flattened)
                const int pj = bit ? a.parent[j] : INT_MAX;
                const int rj = (bit && a.core[j]) ? pj : INT_MAX;
                uint64_t bits = __ballot(rj < (int)w);
                while (bits && attempts < max_tests) {
                    const int src2 = __ffsll((unsigned long long)bits) - 1;
                    bits &= bits - 1;
                    const int jj = Cs * 64 + src2;
                    const int rr = __shfl(rj, src2, 64);
                    ++attempts;
                    ++tests;
                    const int64_t dj = deg_of(a, jj);
                    if (dw >= c && dj >= c && wave_sim_words(A, word_row(a, jj), c)) {
                        ++passed;
                        if (lane == 0) a.parent[w] = rr;
                        done = true;
                        break;
                    }
                    bits &= ~__ballot(rj == rr);  // one test per neighbouring component
                }
            }
        }
        add_stats(a, tests, passed);
        return;
    }
    const int64_t b = a.row_ptr[w], e = a.row_ptr[w + 1];
    for (int64_t t0 = b; t0 < e && attempts < max_tests; t0 += 64) {
        const int64_t t = t0 + lane;
        const int j = t < e ? a.col[t] : -1;
        const int pj = t < e ? a.parent[j] : INT_MAX;  // with the core flag (parents are flattened)
        const int rj = (t < e && a.core[j]) ? pj : INT_MAX;
        uint64_t bits = __ballot(rj < (int)w);
        bool done = false;
        while (bits && attempts < max_tests) {
            const int src = __ffsll((unsigned long long)bits) - 1;
            bits &= bits - 1;
            const int jj = __shfl(j, src, 64);
            const int rr = __shfl(rj, src, 64);
            const int64_t bj = a.row_ptr[jj], ej = a.row_ptr[jj + 1];
            ++attempts;
            ++tests;
            if (wave_sim(a.col + b, e - b, a.col + bj, ej - bj, csim_of(a, w))) {
                ++passed;
                if (lane == 0) a.parent[w] = rr;
                done = true;
                break;
            }
            bits &= ~__ballot(rj == rr);  // one test per neighbouring component
        }
        if (done) break;
    }
    add_stats(a, tests, passed);
}

// The roots k_compress_roots listed, one wave each (grid-stride): no wave is
// started for the points that are not roots.
template <bool WORDS>
__global__ __launch_bounds__(256) void k_hook_roots_list(LabelArgs a, const int32_t *__restrict__ roots,
                                                         const unsigned int *__restrict__ n_roots, int max_tests) {
    const int64_t nr = *n_roots;
    const int64_t waves = (int64_t)gridDim.x * 4;
    for (int64_t q = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); q < nr; q += waves) {
        const int64_t w = roots[q];
        if (a.parent[w] == (int)w) hook_root<WORDS>(a, w, max_tests);
    }
}

// Row w's part of a full round on row words, over its candidate tiles, 64 a
// step (ascending column tile, so entries come in list order); tiles whose
// points share a rank that is not above w's, or that w has joined, are skipped
// without reading their bits; tests are bitset intersections of the two rows'
// words.
__device__ void round_row_words(const LabelArgs &a, int w, uint64_t rw, int c, unsigned &tests, unsigned &passed) {
    const int lane = threadIdx.x & 63;
    const WordRow A = word_row(a, w);
    const int64_t dw = deg_of(a, w);
    int resolved = -1;  // the snapshot component w is known to have joined
    for (int64_t t0 = 0; t0 < A.len; t0 += 64) {
        const int64_t t = t0 + lane;
        uint64_t v = 0ull, tr = 0ull;
        int C = 0;
        if (t < A.len) {
            // the tile id with the pair's flag, the tile's rank with the word
            C = A.tile[t];
            v = word_at(A, t);
            tr = a.tile_rank ? a.tile_rank[C] : ~0ull;
        }
        uint64_t tiles = __ballot(v != 0ull && (tr == ~0ull || tr > rw));
        while (tiles) {
            const int src = __ffsll((unsigned long long)tiles) - 1;
            tiles &= tiles - 1;
            const uint32_t tlo = __builtin_amdgcn_readlane((uint32_t)tr, src);
            const uint32_t thi = __builtin_amdgcn_readlane((uint32_t)(tr >> 32), src);
            const uint64_t trs = ((uint64_t)thi << 32) | tlo;
            if (trs != ~0ull && (int)tlo == resolved) continue;
            const uint32_t vlo = __builtin_amdgcn_readlane((uint32_t)v, src);
            const uint32_t vhi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), src);
            const bool bit = ((lane < 32 ? vlo >> lane : vhi >> (lane - 32)) & 1u) != 0u;
            const int j = __builtin_amdgcn_readlane(C, src) * 64 + lane;
            uint64_t rj = 0ull;
            if (bit) rj = trs == ~0ull ? a.rank[j] : trs;
            const int kj = (int)(uint32_t)rj;
            uint64_t bits = __ballot(bit && rj > rw && kj != resolved);
            while (bits) {
                const int jsrc = __ffsll((unsigned long long)bits) - 1;
                bits &= bits - 1;
                const int jj = __builtin_amdgcn_readlane(j, jsrc);
                const int kjj = __builtin_amdgcn_readlane(kj, jsrc);
                if (test_and_link_words(a, w, jj, A, dw, c, tests, passed)) {
                    resolved = kjj;
                    bits &= ~__ballot(kj == kjj);
                }
            }
        }
    }
}

// Full round.  Every edge between two different snapshot components is owned
// by the endpoint whose component ranks lower (rank = size << 32 | root, all
// distinct), and only the owner examines it.  A row whose rank is at least the
// largest rank among its candidate tiles owns no edge and is skipped without
// reading its list.  Candidates are filtered with the read-only snapshot (one
// 8-byte gather per entry); a stale snapshot only yields redundant candidates,
// which test_and_link's find() check discards.
template <bool WORDS>
__global__ __launch_bounds__(256) void k_round_b(LabelArgs a) {
    a = slice(a);
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= a.n) return;
    const uint64_t rw = a.rank[w];
    if (rw == 0) return;
    if (a.cand_max && rw >= a.cand_max[w >> 6]) return;
    const int c = csim_of(a, w);
    unsigned tests = 0, passed = 0;
    if constexpr (WORDS) {
        round_row_words(a, (int)w, rw, c, tests, passed);
        add_stats(a, tests, passed, 1);
        return;
    }
    int resolved = -1;  // last snapshot component found joined to w
    // four 64-entry windows per step: their loads and rank lookups are issued
    // together, so a row's scan waits on one memory round trip per 256 entries
    const int64_t b = a.row_ptr[w], e = a.row_ptr[w + 1];
    constexpr int kWin = 4;
    for (int64_t t0 = b; t0 < e; t0 += 64 * kWin) {
        int j[kWin];
        uint64_t rj[kWin];
#pragma unroll
        for (int u = 0; u < kWin; ++u) {
            const int64_t t = t0 + 64 * u + lane;
            j[u] = t < e ? a.col[t] : -1;
        }
#pragma unroll
        for (int u = 0; u < kWin; ++u) {
            uint64_t tr = 0ull;
            if (j[u] >= 0) tr = a.tile_rank ? a.tile_rank[j[u] >> 6] : ~0ull;
            rj[u] = tr;
        }
#pragma unroll
        for (int u = 0; u < kWin; ++u)
            if (rj[u] == ~0ull) rj[u] = a.rank[j[u]];
#pragma unroll
        for (int u = 0; u < kWin; ++u) {
            const int kj = (int)(uint32_t)rj[u];
            const bool cand = rj[u] > rw && kj != resolved;
            uint64_t bits = __ballot(cand);
            while (bits) {
                const int src = __ffsll((unsigned long long)bits) - 1;
                bits &= bits - 1;
                const int jj = __shfl(j[u], src, 64);
                const int kjj = __shfl(kj, src, 64);
                if (test_and_link(a, (int)w, jj, b, e, c, tests, passed)) {
                    // w has joined snapshot component kjj: its other entries are joined too
                    resolved = kjj;
                    bits &= ~__ballot(kj == kjj);
                }
            }
        }
    }
    add_stats(a, tests, passed, 1);
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, int src) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, src);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

// Columns (lanes) of a column tile whose rank, held by lane b for column b,
// lies above rw and belongs to no component numbered `resolved`: one pass per
// distinct rank of the tile (a ballot each), the per-row test folded in.
__device__ __forceinline__ uint64_t columns_above(uint64_t rk, uint64_t rw, int resolved) {
    uint64_t rem = ~0ull, bits = 0ull;
    while (rem) {
        const uint64_t val = readlane_u64(rk, __ffsll((unsigned long long)rem) - 1);
        const uint64_t m = __ballot(rk == val);
        rem &= ~m;
        if (val > rw && (int)(uint32_t)val != resolved) bits |= m;
    }
    return bits;
}

// Column tiles that hold words of both of two row tiles, as pairs of positions
// in the two tiles' candidate lists, written to buf (at most kMatchCap a
// chunk) by the whole wave; a chunk continues where the last one ended.
// 64-wide windows of both ascending lists advance like a two-pointer merge,
// each lane looking its B tile up in the A window by a shuffle binary search.
constexpr int kMatchCap = 256;

struct TileMatch {
    const int32_t *ta, *tb;   // column tiles of the two lists
    const uint8_t *za, *zb;   // flags of the non-empty pairs
    int64_t la, lb;
    int64_t ia = 0, ib = 0;   // first positions not yet matched
    __device__ __forceinline__ bool end() const { return ia >= la || ib >= lb; }
    __device__ __forceinline__ void rewind() { ia = ib = 0; }
    __device__ int next(int2 *buf) {
        const int lane = threadIdx.x & 63;
        const uint64_t below = (1ull << lane) - 1ull;
        int m = 0;
        while (!end() && m + 64 <= kMatchCap) {
            bool hit;
            int64_t pa, pb = ib + lane;
            int64_t na, nb;
            if (ta == tb) {  // the rows of one tile
                hit = pb < lb && zb[pb] != 0;
                pa = pb;
                na = nb = ib + 64;
            } else {
                const int va = (int)min<int64_t>(64, la - ia), vb = (int)min<int64_t>(64, lb - ib);
                const int a = lane < va ? ta[ia + lane] : INT_MAX;
                const int b = lane < vb ? tb[ib + lane] : INT_MAX;
                const int fa = lane < va ? (int)za[ia + lane] : 0;
                const int fb = lane < vb ? (int)zb[ib + lane] : 0;
                const int top = min(__shfl(a, va - 1, 64), __shfl(b, vb - 1, 64));
                int lo = 0, hi = va;
#pragma unroll
                for (int step = 0; step < 7; ++step) {
                    const int mid = (lo + hi) >> 1;
                    const int am = __shfl(a, min(mid, 63), 64);
                    if (lo < hi) {
                        if (am < b) lo = mid + 1;
                        else hi = mid;
                    }
                }
                const int found = __shfl(a, min(lo, 63), 64), ffound = __shfl(fa, min(lo, 63), 64);
                hit = lane < vb && b <= top && lo < va && found == b && ffound != 0 && fb != 0;
                pa = ia + lo;
                na = ia + __popcll(__ballot(lane < va && a <= top));
                nb = ib + __popcll(__ballot(lane < vb && b <= top));
            }
            const uint64_t hm = __ballot(hit);
            if (hit) buf[m + __popcll(hm & below)] = make_int2((int)pa, (int)pb);
            m += __popcll(hm);
            ia = na;
            ib = nb;
        }
        return m;
    }
};

// One row tile of the full round, as its wave holds it (lane r = row 64R + r).
struct RoundRows {
    int64_t R;
    int64_t kb, ke;      // the tile's candidate pairs
    uint64_t rw;         // the row's snapshot rank (0: not core)
    int c;
    int resolved = -1;   // last snapshot component this row was found joined to
    unsigned tests = 0, passed = 0;
};

// The edges of tile pair (R, C), C the column tile at position k of R's list:
// v holds the row words (0 for rows that own nothing), tr the tile's common
// rank (all ones: mixed, rk then holds lane b's rank of column b).  Edges to
// higher ranks whose endpoints are still apart are tested together: up to 64,
// 64 / E lanes each (one edge a row; up to eight columns of a row when few
// rows are open).  Both rows' words over the tiles common to R's and C's lists
// (found once per tile pair) are and-ed and their bits counted, so 64 tests
// share one walk of the lists, and their words the same cache lines.  Stops
// after `budget` such batches (it is counted down); true when no edge is left.
__device__ bool round_pair(const LabelArgs &a, RoundRows &rr, int C, uint64_t v, uint64_t tr, uint64_t rk, int &budget,
                           int2 *match, uint16_t *edge) {
    const int lane = threadIdx.x & 63;
    const int w = (int)(rr.R * 64 + lane);
    const bool common = tr != ~0ull;
    uint64_t bits;
    if (common) bits = (tr > rr.rw && (int)(uint32_t)tr != rr.resolved) ? v : 0ull;
    else bits = columns_above(rk, rr.rw, rr.resolved) & v;
    TileMatch tm;
    int n_match = -1;  // tiles common to R and C (-1: not matched yet)
    while (__ballot(bits != 0ull)) {
        const int col = bits ? __ffsll((unsigned long long)bits) - 1 : 0;
        const uint64_t rb = common ? tr : __shfl(rk, col, 64);
        bool changed = false, open = false;
        if (bits) {
            changed = uf_find(a.parent, w) == uf_find(a.parent, C * 64 + col);
            open = !changed;
        }
        if (changed) rr.resolved = (int)(uint32_t)rb;
        const uint64_t need = __ballot(open);
        if (need) {
            if (budget-- <= 0) return false;
            const int rows = __popcll(need);
            const int quota = rows >= 32 ? 1 : min(8, 32 / rows);
            const int mine = open ? min(__popcll(bits), quota) : 0;
            const int incl = wave_incl_scan(mine), off = incl - mine;
            const int E = __builtin_amdgcn_readlane(incl, 63);
            uint64_t left = bits;
            for (int x = 0; x < mine; ++x) {
                edge[off + x] = (uint16_t)((lane << 6) | (__ffsll((unsigned long long)left) - 1));
                left &= left - 1;
            }
            if (n_match < 0) {
                const int64_t kc = a.tp_ptr[C];
                tm.ta = a.tp_col + rr.kb;
                tm.za = a.pair_nz + rr.kb;
                tm.la = rr.ke - rr.kb;
                tm.tb = a.tp_col + kc;
                tm.zb = a.pair_nz + kc;
                tm.lb = a.tp_ptr[C + 1] - kc;
                n_match = tm.next(match);
            }
            wave_lds_fence();
            int shift = 6;  // 2^shift lanes per edge
            while ((E << shift) > 64) --shift;
            const int grp = lane >> shift, sub = lane & ((1 << shift) - 1);
            const bool on = grp < E;
            const int ed = on ? edge[grp] : 0;
            const int er = ed >> 6, ec = ed & 63;
            const uint64_t *__restrict__ wa = a.mask + rr.kb * 64 + er;
            const uint64_t *__restrict__ wb = a.mask + (tm.tb - a.tp_col) * 64 + ec;
            int cnt = 0, sum = 0;
            bool dec = !on || rr.c <= 0;
            bool again = false;  // the lists took more than one chunk
            for (;;) {
                constexpr int kU = 8;
                for (int t0 = 0; t0 < n_match && __ballot(!dec); t0 += kU << shift) {
                    uint64_t x[kU], y[kU];
#pragma unroll
                    for (int z = 0; z < kU; ++z) {
                        const int t = t0 + (z << shift) + sub;
                        x[z] = y[z] = 0ull;
                        if (!dec && t < n_match) {
                            const int2 m = match[t];
                            x[z] = wa[(int64_t)m.x * 64];
                            y[z] = wb[(int64_t)m.y * 64];
                        }
                    }
#pragma unroll
                    for (int z = 0; z < kU; ++z) cnt += __popcll(x[z] & y[z]);
                    sum = cnt;
                    for (int o = 0; o < shift; ++o) sum += __shfl_xor(sum, 1 << o, 64);
                    dec = dec || sum >= rr.c;
                }
                if (tm.end() || __ballot(!dec) == 0ull) break;
                wave_lds_fence();
                n_match = tm.next(match);
                again = true;
                wave_lds_fence();
            }
            if (again) {  // the next test of this tile pair starts over
                tm.rewind();
                n_match = -1;
            }
            const bool pass = on && (rr.c <= 0 || sum >= rr.c);
            if (pass && sub == 0) uf_union(a.parent, (int)(rr.R * 64 + er), C * 64 + ec);
            const uint64_t pm = __ballot(pass && sub == 0);
            rr.tests += (unsigned)E;
            rr.passed += (unsigned)__popcll(pm);
            // each row takes up the results of its edges
            uint64_t todo = bits;
            for (int x = 0; x < quota; ++x) {
                const int cx = todo ? __ffsll((unsigned long long)todo) - 1 : 0;
                const uint64_t rx = common ? tr : __shfl(rk, cx, 64);
                if (x < mine) {
                    if ((pm >> ((off + x) << shift)) & 1ull) {
                        changed = true;
                        rr.resolved = (int)(uint32_t)rx;
                    }
                    todo &= todo - 1;
                }
            }
            if (open) bits = left;
            wave_lds_fence();
        }
        // a joined component: its remaining columns are joined as well
        if (__ballot(changed)) {
            if (common) {
                if (changed) bits = 0ull;
            } else {
                if (changed && !open) bits &= bits - 1;
                bits &= columns_above(rk, rr.rw, rr.resolved);
            }
        }
    }
    return true;
}

// Full round on a graph's tile-pair words, `split` waves per row tile (lane r
// owns row w = 64R + r; wave q of the tile takes the q-th of `split` equal
// parts of its candidate pairs), with k_round_b's ownership and skip rules: an
// edge is examined by the endpoint of lower snapshot rank, rows at or above
// the tile's candidate maximum own none, and a row drops every column of a
// component it has joined (per wave: the skip is only a saving, every row
// checks with two finds before a test).  The pairs are walked once for all 64
// rows -- pair k's 64 row words are one contiguous 512-byte load, 8 pairs in
// flight -- and the rank filter and the already-joined check run for all rows
// in parallel (round_pair).  A wave runs kInlineTests batches of tests itself:
// a pass usually joins the components of the other open edges too.  After
// them, a pair with open edges goes to a queue ({R, pair}; one counter update
// per 64 pairs) that k_round_queue serves, one wave per pair, so that no wave
// runs the tests of many pairs one after another; a full queue falls back to
// tests here.
// Bound by the latency of dependent loads.  Tested one edge per wave from a
// queue of rows, the round took 622 us at n = 1e6, d = 3, 708 us at n = 2e5,
// d = 64 and 182 us at n = 3e4, d = 3; batched by tile pair
// 284, 198 and 72 us.
__global__ __launch_bounds__(256) void k_round_tile(LabelArgs a, int64_t n_tiles, int split) {
    a = slice(a);
    __shared__ int2 s_match[4][kMatchCap];
    __shared__ uint16_t s_edge[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t g = (int64_t)blockIdx.x * 4 + wave;
    if (g >= n_tiles * split) return;
    const int64_t gR = g / split;
    const int q = (int)(g - gR * split);
    RoundRows rr;
    rr.R = a.tile_order ? (int64_t)a.tile_order[gR] : gR;
    const int64_t w = rr.R * 64 + lane;
    rr.rw = w < a.n ? a.rank[w] : 0ull;
    const uint64_t cmax = a.cand_max ? a.cand_max[rr.R] : ~0ull;
    const bool active = rr.rw != 0ull && rr.rw < cmax;
    const uint64_t act = __ballot(active);
    if (act == 0ull) return;
    // a column tile whose points share a rank not above every active row's has no candidate
    uint64_t rmin = active ? rr.rw : ~0ull;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint64_t o = __shfl_xor(rmin, off, 64);
        rmin = o < rmin ? o : rmin;
    }
    rr.c = csim_of(a, rr.R * 64);
    rr.kb = a.tp_ptr[rr.R];
    rr.ke = a.tp_ptr[rr.R + 1];
    const int64_t per = (rr.ke - rr.kb + split - 1) / split;
    const int64_t kb = rr.kb + q * per, ke = min(rr.ke, kb + per);
    constexpr int kInFlight = 8, kInlineTests = 2;
    int budget = kInlineTests;
    for (int64_t k0 = kb; k0 < ke; k0 += 64) {
        const int64_t kk = k0 + lane;
        int C = 0;
        uint64_t tr = 0ull;
        bool want = false;
        if (kk < ke && a.pair_nz[kk] != 0) {
            C = a.tp_col[kk];
            tr = a.tile_rank ? a.tile_rank[C] : ~0ull;
            want = tr == ~0ull || tr > rmin;
        }
        uint64_t wm = __ballot(want), open = 0ull;
        while (wm) {
            int idx[kInFlight];
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                idx[u] = wm ? __ffsll((unsigned long long)wm) - 1 : -1;
                wm &= wm - 1;
            }
            uint64_t v[kInFlight], rk[kInFlight];
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                v[u] = 0ull;
                rk[u] = 0ull;
                if (idx[u] >= 0) {
                    const int64_t Cu = __builtin_amdgcn_readlane(C, idx[u]);
                    if (active) v[u] = a.mask[(k0 + idx[u]) * 64 + lane];
                    if (readlane_u64(tr, idx[u]) == ~0ull && Cu * 64 + lane < a.n) rk[u] = a.rank[Cu * 64 + lane];
                }
            }
#pragma unroll 1
            for (int u = 0; u < kInFlight; ++u) {
                uint64_t vu = 0ull, rku = 0ull;
                int iu = -1;
                // (a private array indexed at run time would live in memory)
#pragma unroll
                for (int x = 0; x < kInFlight; ++x)
                    if (x == u) {
                        vu = v[x];
                        rku = rk[x];
                        iu = idx[x];
                    }
                if (iu < 0 || __ballot(vu != 0ull) == 0ull) continue;
                if (!round_pair(a, rr, __builtin_amdgcn_readlane(C, iu), vu, readlane_u64(tr, iu), rku, budget,
                                s_match[wave], s_edge[wave]))
                    open |= 1ull << iu;
            }
        }
        if (open) {
            unsigned long long base = 0;
            if (lane == 0) base = atomicAdd(a.rq_len, (unsigned long long)__popcll(open));
            base = __shfl(base, 0, 64);
            const bool mine = ((open >> lane) & 1ull) != 0ull;
            const unsigned long long slot = base + __popcll(open & ((1ull << lane) - 1ull));
            const bool queued = mine && slot < (unsigned long long)a.rq_cap;
            if (queued) a.rq[slot] = make_int2((int)rr.R, (int)(kk - rr.kb));
            open &= ~__ballot(queued);
            while (open) {
                const int iu = __ffsll((unsigned long long)open) - 1;
                open &= open - 1;
                const int Cu = __builtin_amdgcn_readlane(C, iu);
                const uint64_t vu = active ? a.mask[(k0 + iu) * 64 + lane] : 0ull;
                const uint64_t rku = (int64_t)Cu * 64 + lane < a.n ? a.rank[(int64_t)Cu * 64 + lane] : 0ull;
                int all = INT_MAX;
                (void)round_pair(a, rr, Cu, vu, readlane_u64(tr, iu), rku, all, s_match[wave], s_edge[wave]);
            }
        }
    }
    add_stats(a, rr.tests, rr.passed, q == 0 ? (unsigned)__popcll(act) : 0u);
}

// The tile pairs k_round_tile queued, one wave each (grid-stride).
__global__ __launch_bounds__(256) void k_round_queue(LabelArgs a) {
    a = slice(a);
    __shared__ int2 s_match[4][kMatchCap];
    __shared__ uint16_t s_edge[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t nq = (int64_t)min<unsigned long long>(*a.rq_len, (unsigned long long)a.rq_cap);
    const int64_t waves = (int64_t)gridDim.x * 4;
    for (int64_t q = (int64_t)blockIdx.x * 4 + wave; q < nq; q += waves) {
        const int2 e = a.rq[q];
        RoundRows rr;
        rr.R = uniform(e.x);
        rr.kb = a.tp_ptr[rr.R];
        rr.ke = a.tp_ptr[rr.R + 1];
        const int64_t k = rr.kb + uniform(e.y);
        const int C = uniform(a.tp_col[k]);
        const int64_t w = rr.R * 64 + lane, j = (int64_t)C * 64 + lane;
        rr.rw = w < a.n ? a.rank[w] : 0ull;
        const uint64_t v = rr.rw != 0ull ? a.mask[k * 64 + lane] : 0ull;
        const uint64_t rk = j < a.n ? a.rank[j] : 0ull;
        const uint64_t tr = a.tile_rank ? a.tile_rank[C] : ~0ull;
        rr.c = csim_of(a, rr.R * 64);
        int all = INT_MAX;
        (void)round_pair(a, rr, C, v, tr, rk, all, s_match[wave], s_edge[wave]);
        add_stats(a, rr.tests, rr.passed);
    }
}

// Queue entries of one full round over that many tile pairs.
static int64_t round_queue_cap(int64_t n_tile_pairs, int n_c) {
    if (const char *ev = std::getenv("CNN_HIP_ROUND_QUEUE")) return std::max<int64_t>(1, std::atoll(ev));  // tests
    return std::min<int64_t>(std::max<int64_t>(n_tile_pairs, 1), ((int64_t)1 << 21) / n_c);
}

// Waves per row tile for k_round_tile: one per 128 candidate pairs, and with few
// tiles enough for about 4096 waves of at least 8 pairs.  (Twice and half as
// many waves were within 2 % of this from n = 1e3 to 1e6.)
static int round_split(int64_t n_tile_pairs, int64_t n_tiles) {
    if (n_tiles <= 0) return 1;
    const int64_t per_tile = ceil_div(n_tile_pairs, n_tiles);
    const int64_t want = std::max(ceil_div(per_tile, 128), std::min(ceil_div(4096, n_tiles), ceil_div(per_tile, 8)));
    return (int)std::min<int64_t>(64, std::max<int64_t>(1, want));
}

// Largest rank over the candidate column tiles of each row tile, one
// workgroup per row tile: a tile with thousands of candidates takes a few
// steps of 256 instead of a long serial walk by one wave.
__global__ __launch_bounds__(256) void k_cand_max(const uint64_t *__restrict__ tmax, const int64_t *__restrict__ tp_ptr,
                                                  const int32_t *__restrict__ tp_col, int64_t n_tiles,
                                                  uint64_t *__restrict__ cmax) {
    tmax += (int64_t)blockIdx.y * n_tiles;
    cmax += (int64_t)blockIdx.y * n_tiles;
    __shared__ uint64_t sv[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t R = blockIdx.x;
    if (R >= n_tiles) return;  // the whole workgroup
    const int64_t kb = tp_ptr ? tp_ptr[R] : 0, ke = tp_ptr ? tp_ptr[R + 1] : n_tiles;
    uint64_t v = 0;
    for (int64_t k = kb + threadIdx.x; k < ke; k += 256) {
        const int64_t C = tp_ptr ? (int64_t)tp_col[k] : k;
        const uint64_t x = tmax[C];
        v = x > v ? x : v;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint64_t o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    if (lane == 0) sv[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t m = sv[0];
        for (int q = 1; q < 4; ++q) m = sv[q] > m ? sv[q] : m;
        cmax[R] = m;
    }
}

// rank[w] = (component size << 32 | root) of core points, 0 otherwise; with a
// tile structure also, per tile of 64 points, the largest rank (0: no core
// point) and the tile's common rank: the rank of all its points when they
// share one, all ones when they differ.
__global__ __launch_bounds__(256) void k_snapshot(const uint8_t *core, const int *parent, const int32_t *cnt, int64_t n,
                                                  uint64_t *rank, int64_t n_tiles, uint64_t *tmax, uint64_t *tcommon) {
    const int64_t off = (int64_t)blockIdx.y * n;
    const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
    uint64_t mine = 0ull;
    if (w < n) {
        const int r = parent[off + w];
        mine = core[off + w] ? (((uint64_t)(uint32_t)cnt[off + r] << 32) | (uint32_t)r) : 0ull;
        rank[off + w] = mine;
    }
    const int64_t t = w >> 6;  // one wave per tile
    if (t >= n_tiles) return;
    uint64_t v = mine;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const uint64_t x = __shfl_xor(v, o, 64);
        v = x > v ? x : v;
    }
    const bool same = __ballot(w < n && mine != v) == 0ull;  // every real point has the largest rank
    if ((threadIdx.x & 63) == 0) {
        tmax[(int64_t)blockIdx.y * n_tiles + t] = v;
        tcommon[(int64_t)blockIdx.y * n_tiles + t] = same ? v : ~0ull;
    }
}

// Flatten: every entry points at its root afterwards.  The walk only reads
// (entries of other threads may change meanwhile, but only towards their
// roots) and each thread writes only its own entry, so no write can leave an
// entry below its root.
__device__ __forceinline__ int flatten(int *parent, int64_t w) {
    int x = (int)w;
    int p = atomic_load_relaxed(&parent[x]);
    while (p != x) {
        x = p;
        p = atomic_load_relaxed(&parent[x]);
    }
    __hip_atomic_store(&parent[w], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return x;
}

// Flattening that also lists the core points that are roots afterwards, for
// k_hook_roots_list; one counter update per workgroup (the counter is a single
// address).  The chains are walked past the L1 caches, so few points are spread
// over many compute units: n = 2e4, 27 us in workgroups of 1024, 23 of 256.
__global__ __launch_bounds__(1024) void k_compress_roots(int *parent, const uint8_t *__restrict__ core, int64_t n,
                                                         int32_t *__restrict__ roots,
                                                         unsigned int *__restrict__ n_roots) {
    __shared__ unsigned s_cnt[16], s_base;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool root = w < n && flatten(parent, w) == (int)w && core[w] != 0;
    const uint64_t m = __ballot(root);
    if (lane == 0) s_cnt[wave] = (unsigned)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned total = 0;
        for (int q = 0; q < (int)blockDim.x / 64; ++q) {
            const unsigned x = s_cnt[q];
            s_cnt[q] = total;
            total += x;
        }
        s_base = total ? atomicAdd(n_roots, total) : 0u;
    }
    __syncthreads();
    if (root) roots[s_base + s_cnt[wave] + __popcll(m & ((1ull << lane) - 1ull))] = (int32_t)w;
}

// Lanes sharing a key are combined before one atomic per distinct key (points
// of a component are mostly adjacent in the working order).
__device__ __forceinline__ void wave_add_by_key(int32_t *cnt, int32_t *mins, bool active, int key, int val) {
    uint64_t pending = __ballot(active);
    while (pending) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const int k = __shfl(key, leader, 64);
        const bool mine = active && key == k;
        const uint64_t match = __ballot(mine);
        if (mins) {
            int v = mine ? val : INT_MAX;
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
            if (__lane_id() == leader) atomicMin(&mins[k], v);
        }
        if (__lane_id() == leader) atomicAdd(&cnt[k], __popcll(match));
        pending &= ~match;
    }
}

// Per-key sums over consecutive points: a wave walks `steps` steps of 64
// points and keeps one run (key, count, minimum) while every active lane of a
// step has the run's key, so a large component costs one atomic per run, not
// one per wave (same-address atomics serialize).  Few points take few steps:
// 16 steps of dependent loads on 8 workgroups took 22 and 35 us at n = 3e4.
static int run_steps(int64_t n) { return (int)std::min<int64_t>(16, std::max<int64_t>(1, ceil_div(n, 64 * 2048))); }

struct KeyRun {
    int key = -1;
    int cnt = 0;
    int mn = INT_MAX;
};

__device__ __forceinline__ void run_flush(KeyRun &run, int32_t *cnt, int32_t *mins) {
    if (run.key >= 0 && __lane_id() == 0) {
        atomicAdd(&cnt[run.key], run.cnt);
        if (mins) atomicMin(&mins[run.key], run.mn);
    }
    run.key = -1;
    run.cnt = 0;
    run.mn = INT_MAX;
}

__device__ __forceinline__ void run_add(KeyRun &run, int32_t *cnt, int32_t *mins, bool active, int key, int val) {
    const uint64_t act = __ballot(active);
    if (!act) return;
    const int k = __shfl(key, __ffsll((unsigned long long)act) - 1, 64);
    if (__ballot(active && key != k) != 0ull) {  // mixed keys: one atomic per key
        wave_add_by_key(cnt, mins, active, key, val);
        return;
    }
    if (k != run.key) {
        run_flush(run, cnt, mins);
        run.key = k;
    }
    run.cnt += __popcll(act);
    if (mins) {
        int v = active ? val : INT_MAX;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
        run.mn = min(run.mn, v);
    }
}

__device__ __forceinline__ int64_t run_base(int steps) {
    return ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * (64 * steps);
}

// Flattens the forest and counts the core points of every component; the
// components go into the striped statistics.
__global__ __launch_bounds__(256) void k_root_count(LabelArgs a, int32_t *cnt, int steps) {
    a = slice(a);
    cnt += (int64_t)blockIdx.y * a.n;
    const int64_t base = run_base(steps);
    KeyRun run;
    unsigned roots = 0;
    for (int it = 0; it < steps; ++it) {
        const int64_t w = base + it * 64 + __lane_id();
        int r = 0;
        bool active = false;
        if (w < a.n) {
            r = flatten(a.parent, w);
            active = a.core[w] != 0;
        }
        run_add(run, cnt, nullptr, active, r, 0);
        roots += (unsigned)__popcll(__ballot(active && r == (int)w));
    }
    run_flush(run, cnt, nullptr);
    add_stats(a, 0, 0, 0, roots);
}

// ------------------------------------------------------------------ labels

// Flattens the forest; size and smallest caller index of every component, core
// points and components counted into counters[0] and [1].
__global__ __launch_bounds__(256) void k_comp_stats(const uint8_t *core, int *parent, const int32_t *perm, int64_t n,
                                                    int32_t *cmin, int32_t *csize, unsigned long long *counters,
                                                    int steps) {
    const int64_t off = (int64_t)blockIdx.y * n;
    core += off;
    parent += off;
    cmin += off;
    csize += off;
    counters += 8 * blockIdx.y;
    const int64_t base = run_base(steps);
    KeyRun run;
    unsigned nc = 0, nr = 0;
    for (int it = 0; it < steps; ++it) {
        const int64_t w = base + it * 64 + __lane_id();
        bool is_core = false;
        int r = 0, orig = 0;
        if (w < n) {
            r = flatten(parent, w);
            is_core = core[w] != 0;
            if (is_core) orig = perm ? perm[w] : (int32_t)w;
        }
        run_add(run, csize, cmin, is_core, r, orig);
        nc += (unsigned)__popcll(__ballot(is_core));
        nr += (unsigned)__popcll(__ballot(is_core && r == (int)w));
    }
    run_flush(run, csize, cmin);
    // one update per workgroup: the counters are single addresses
    __shared__ unsigned s_nc[4], s_nr[4];
    if (__lane_id() == 0) {
        s_nc[threadIdx.x >> 6] = nc;
        s_nr[threadIdx.x >> 6] = nr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        nc = s_nc[0] + s_nc[1] + s_nc[2] + s_nc[3];
        nr = s_nr[0] + s_nr[1] + s_nr[2] + s_nr[3];
        if (nc) atomicAdd(&counters[0], (unsigned long long)nc);
        if (nr) atomicAdd(&counters[1], (unsigned long long)nr);
    }
}

__global__ void k_collect_clusters(const uint8_t *core, const int *parent, const int32_t *cmin, const int32_t *csize,
                                   int64_t n, int64_t member_cutoff, unsigned long long *K, uint64_t *keys,
                                   int32_t *vals) {
    int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n || !core[w] || parent[w] != (int)w) return;
    const int32_t sz = csize[w];
    if ((int64_t)sz < member_cutoff) return;
    const unsigned long long idx = atomicAdd(K, 1ull);
    keys[idx] = ((uint64_t)(uint32_t)(0x7fffffff - sz) << 32) | (uint32_t)cmin[w];
    vals[idx] = (int32_t)w;
}

__global__ void k_rank_clusters(const int32_t *vals, int64_t K, int64_t max_clusters, int32_t *newlab) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= K) return;
    newlab[vals[t]] = (max_clusters < 0 || t < max_clusters) ? (int32_t)(t + 1) : 0;
}

// sort_by_size without the host: the K cluster keys (K read on the device;
// they are distinct) are sorted by one workgroup in LDS (bitonic, over the
// next power of two at or above K) and ranked as k_rank_clusters does.  More
// than kSmallClusters clusters: *big = 1 and nothing is written (the host
// sorts them after its next read of the counters).
constexpr int kSmallClusters = 1024;
__global__ __launch_bounds__(kSmallClusters) void k_rank_clusters_small(const uint64_t *__restrict__ keys,
                                                                        const int32_t *__restrict__ vals,
                                                                        const unsigned long long *__restrict__ Kp,
                                                                        int64_t max_clusters,
                                                                        int32_t *__restrict__ newlab,
                                                                        unsigned long long *__restrict__ big) {
    __shared__ uint64_t sk[kSmallClusters];
    __shared__ int32_t sv[kSmallClusters];
    const int64_t K = (int64_t)*Kp;
    const int t = threadIdx.x;
    if (K > kSmallClusters) {
        if (t == 0) *big = 1ull;
        return;
    }
    int n2 = 1;
    while (n2 < K) n2 <<= 1;
    sk[t] = t < K ? keys[t] : ~0ull;
    sv[t] = t < K ? vals[t] : -1;
    __syncthreads();
    for (int size = 2; size <= n2; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const int q = t ^ stride;
            if (q > t && q < n2) {
                const bool up = (t & size) == 0;
                const uint64_t ka = sk[t], kb = sk[q];
                if ((ka > kb) == up) {
                    sk[t] = kb;
                    sk[q] = ka;
                    const int32_t v = sv[t];
                    sv[t] = sv[q];
                    sv[q] = v;
                }
            }
            __syncthreads();
        }
    }
    if (t < K) newlab[sv[t]] = (max_clusters < 0 || t < max_clusters) ? (int32_t)(t + 1) : 0;
}

// Packed batches: clusters of all datasets sorted together by
// (dataset, size descending, smallest original index); ranks restart at 1 in
// every dataset.
struct PackedKey {
    int ds_shift, size_shift;
    uint32_t size_max;
    const int32_t *tile_ds;
    const int64_t *ds_offset;  // cmin is stored relative to the dataset's first row when set
};

__global__ void k_collect_clusters_packed(const uint8_t *core, const int *parent, const int32_t *cmin,
                                          const int32_t *csize, int64_t n, int64_t member_cutoff, PackedKey pk,
                                          unsigned long long *K, uint64_t *keys, int32_t *vals) {
    int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n || !core[w] || parent[w] != (int)w) return;
    const int32_t sz = csize[w];
    if ((int64_t)sz < member_cutoff) return;
    const int ds = pk.tile_ds[w >> 6];
    const uint64_t cm = (uint64_t)(cmin[w] - (pk.ds_offset ? pk.ds_offset[ds] : 0));
    const unsigned long long idx = atomicAdd(K, 1ull);
    keys[idx] = ((uint64_t)ds << pk.ds_shift) | ((uint64_t)(pk.size_max - (uint32_t)sz) << pk.size_shift) | cm;
    vals[idx] = (int32_t)w;
}

__global__ void k_first_of_set(const uint64_t *keys, int64_t K, int ds_shift, int32_t *first) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= K) return;
    const uint64_t ds = keys[t] >> ds_shift;
    if (t == 0 || (keys[t - 1] >> ds_shift) != ds) first[ds] = (int32_t)t;
}

__global__ void k_rank_clusters_packed(const uint64_t *keys, const int32_t *vals, int64_t K, int ds_shift,
                                       const int32_t *first, int64_t max_clusters, int32_t *newlab,
                                       unsigned long long *kept) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool keep = false;
    if (t < K) {
        const int64_t r = t - first[keys[t] >> ds_shift] + 1;
        keep = max_clusters < 0 || r <= max_clusters;
        newlab[vals[t]] = keep ? (int32_t)r : 0;
    }
    const uint64_t b = __ballot(keep);
    if ((threadIdx.x & 63) == 0 && b) atomicAdd(kept, (unsigned long long)__popcll(b));
}

__global__ void k_write_sorted(const uint8_t *core, const int *parent, const int32_t *newlab, const int32_t *perm,
                               int64_t n, int64_t *labels) {
    const int64_t off = (int64_t)blockIdx.y * n;
    core += off;
    parent += off;
    newlab += off;
    labels += off;
    int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n) return;
    const int64_t o = perm ? perm[w] : w;
    if (o >= 0) labels[o] = core[w] ? (int64_t)newlab[parent[w]] : 0;
}

__global__ void k_mark_first(const uint8_t *core, const int *parent, const int32_t *cmin, int64_t n,
                             uint8_t *isfirst) {
    int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n || !core[w] || parent[w] != (int)w) return;
    isfirst[cmin[w]] = 1;
}

__global__ void k_write_unsorted(const uint8_t *core, const int *parent, const int32_t *cmin, const int32_t *rank_incl,
                                 const int32_t *perm, int64_t n, int64_t current_start, bool write_all,
                                 int64_t *labels) {
    int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n) return;
    const int64_t o = perm ? perm[w] : w;
    if (o < 0) return;
    if (core[w]) labels[o] = current_start + (int64_t)rank_incl[cmin[parent[w]]] - 1;
    else if (write_all) labels[o] = 0;
}

// ------------------------------------------------------------------ per-row word lists from lists

// Rows of a CSR (strictly ascending) as word lists: one word per distinct
// column tile (index >> 6) of a row.  Count per row, one wave per row.
__global__ __launch_bounds__(256) void k_row_word_count(const int64_t *__restrict__ row_ptr,
                                                        const int32_t *__restrict__ col, int64_t n,
                                                        int32_t *__restrict__ cnt) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= n) return;
    const int64_t b = row_ptr[w], e = row_ptr[w + 1];
    int total = 0;
    // four windows of 64 entries per step, their loads issued together
    for (int64_t t0 = b; t0 < e; t0 += 256) {
        int32_t cur[4], prev[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t t = t0 + 64 * u + lane;
            cur[u] = t < e ? col[t] : 0;
            prev[u] = (t < e && t > b) ? col[t - 1] : 0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t t = t0 + 64 * u + lane;
            const bool head = t < e && (t == b || (prev[u] >> 6) != (cur[u] >> 6));
            total += __popcll(__ballot(head));
        }
    }
    if (lane == 0) cnt[w] = total;
}

// Entries and words of every stride-th row, summed into sums[0] / sums[1]:
// the automatic similarity choice estimates the lists' fill from them.  A few
// hundred workgroups add their sums once each (two updates of the same
// addresses per row took 220 us for 9000 rows and 15 us for 500, the latter 5 us
// as here).
__global__ __launch_bounds__(256) void k_row_word_sample(const int64_t *__restrict__ row_ptr,
                                                         const int32_t *__restrict__ col, int64_t n, int64_t stride,
                                                         unsigned long long *__restrict__ sums) {
    __shared__ unsigned long long s_entries[4], s_words[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long entries = 0, words = 0;
    for (int64_t w = ((int64_t)blockIdx.x * 4 + wave) * stride; w < n; w += (int64_t)gridDim.x * 4 * stride) {
        const int64_t b = row_ptr[w], e = row_ptr[w + 1];
        int total = 0;
        for (int64_t t0 = b; t0 < e; t0 += 64) {
            const int64_t t = t0 + lane;
            bool head = false;
            if (t < e) head = t == b || (col[t - 1] >> 6) != (col[t] >> 6);
            total += __popcll(__ballot(head));
        }
        entries += (unsigned long long)(e - b);
        words += (unsigned long long)total;
    }
    if (lane == 0) {
        s_entries[wave] = entries;
        s_words[wave] = words;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        entries = s_entries[0] + s_entries[1] + s_entries[2] + s_entries[3];
        words = s_words[0] + s_words[1] + s_words[2] + s_words[3];
        if (words) {
            atomicAdd(&sums[0], entries);
            atomicAdd(&sums[1], words);
        }
    }
}

// Fill: the entries of one word are consecutive in the row, so each window of
// 64 entries ors its bits per segment (a segmented scan over the lanes, the
// open segment of the previous window carried in) and the segment's last
// entry writes the word and its tile.
__global__ __launch_bounds__(256) void k_row_word_fill(const int64_t *__restrict__ row_ptr,
                                                       const int32_t *__restrict__ col, int64_t n,
                                                       const int64_t *__restrict__ wptr, int32_t *__restrict__ wtile,
                                                       uint64_t *__restrict__ wword) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= n) return;
    const int64_t b = row_ptr[w], e = row_ptr[w + 1];
    const int64_t base = wptr[w];
    int64_t run = 0;          // words started in earlier windows
    uint64_t carry = 0ull;    // bits of the word still open at the end of the previous window
    const uint64_t upto_mask = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
    for (int64_t t0 = b; t0 < e; t0 += 64) {
        const int64_t t = t0 + lane;
        const bool valid = t < e;
        int tile = 0;
        uint64_t x = 0ull;
        bool head = false, tail = false;
        if (valid) {
            const int v = col[t];
            tile = v >> 6;
            x = 1ull << (v & 63);
            head = t == b || (col[t - 1] >> 6) != tile;
            tail = t + 1 == e || (col[t + 1] >> 6) != tile;
        }
        const uint64_t hm = __ballot(head);
        const uint64_t upto = hm & upto_mask;
        const int start = upto ? 63 - __clzll((long long)upto) : -1;  // this lane's word starts here
        if (start < 0) x |= carry;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint64_t y = __shfl_up(x, off, 64);
            if (lane >= off && lane - off >= start) x |= y;
        }
        const int64_t idx = base + run + __popcll(upto) - 1;
        if (valid && tail) {
            wtile[idx] = tile;
            wword[idx] = x;
        }
        const bool open = __shfl((int)(valid && !tail), 63, 64) != 0;
        const uint64_t last = __shfl(x, 63, 64);
        carry = open ? last : 0ull;
        run += __popcll(hm);
    }
}

static inline unsigned blocks_for(int64_t n, int per = 256) { return (unsigned)std::max<int64_t>(1, ceil_div(n, per)); }


void labels_run(cnn_ctx *ctx, const LabelRequest &req, cnn_label_stats *st) {
    hipStream_t s = ctx->stream;
    const int64_t n = req.n;
    if (req.c_sim < 0 || req.m_core < 0) throw InvalidArg{"c_sim and m_core must be >= 0"};
    if (req.sim_mode != CNN_SIM_AUTO && req.sim_mode != CNN_SIM_MERGE && req.sim_mode != CNN_SIM_BITSET)
        throw InvalidArg{"unknown sim_mode"};
    cnn_label_stats local{};
    if (n == 0) {
        if (st) *st = local;
        return;
    }
    Scratch<uint8_t> core(ctx, n);
    Scratch<uint64_t> rank(ctx, n);
    Scratch<int> parent(ctx, n);
    // the pass's small counters in one buffer, zeroed by k_init:
    // counters (8), striped test statistics (4 per slot), the hook and the round
    // queue length, then one root count per root hooking pass
    const int64_t kSmallSlots = 8 + 4 * kStatSlots + 2 + std::max(req.root_passes, 0);
    Scratch<unsigned long long> small(ctx, kSmallSlots);
    unsigned long long *const counters_p = small.p, *const tstats_p = small.p + 8;
    unsigned long long *const slot_p = small.p + 8 + 4 * kStatSlots;
    LabelArgs a{req.row_ptr, req.col, n, req.c_sim, req.m_core, core.p, parent.p, tstats_p, rank.p, nullptr,
                nullptr, req.selfpos, req.tile_csim, req.tile_mcore};

    CNN_HIP(hipEventRecord(ctx->ev[0], s));
    // similarity form: bitset intersections of row words (the spatial graph's
    // tile-pair masks, or per-row word lists built here from the lists), or the
    // sorted-list merge
    const bool tile_words = req.mask && req.pair_nz && req.tp_ptr;
    bool words = false;
    std::unique_ptr<Scratch<int64_t>> wptr;
    std::unique_ptr<Scratch<int32_t>> wtile;
    std::unique_ptr<Scratch<uint64_t>> wword;
    if (req.sim_mode != CNN_SIM_MERGE && tile_words) {
        words = true;
        a.mask = req.mask;
        a.pair_nz = req.pair_nz;
        a.tp_ptr = req.tp_ptr;
        a.tp_col = req.tp_col;
        a.diag = req.diag;
        a.tile_order = req.tile_order;
    } else if (req.sim_mode != CNN_SIM_MERGE && req.col) {
        bool build = req.sim_mode == CNN_SIM_BITSET;
        if (!build && req.words_min_fill > 0 && req.words_min_fill <= (int64_t)1 << 24) {
            // automatic choice: the fill of every stride-th row decides, the
            // stride at least 16 and large enough to sample about 2^21 entries
            const int64_t nnz = req.nnz >= 0 ? req.nnz : read_scalar(ctx, req.row_ptr + n);
            const int64_t stride = std::max<int64_t>(16, ceil_div(nnz, (int64_t)1 << 21));
            Scratch<unsigned long long> sums(ctx, 2);
            fill_u64(ctx, sums.p, 0, 2);
            const int64_t rows = ceil_div(n, stride);
            k_row_word_sample<<<(unsigned)std::min<int64_t>(blocks_for(rows, 4), 512), 256, 0, s>>>(req.row_ptr, req.col, n, stride, sums.p);
            CNN_HIP(hipGetLastError());
            PinnedReads rd(ctx);
            const unsigned long long *h = rd.get(sums.p, 2);
            rd.wait();
            build = h[1] > 0 && h[0] >= (unsigned long long)req.words_min_fill * h[1];
        }
        if (build) {
            wptr.reset(new Scratch<int64_t>(ctx, n + 1));
            Scratch<int32_t> wcnt(ctx, n);
            k_row_word_count<<<blocks_for(n, 4), 256, 0, s>>>(req.row_ptr, req.col, n, wcnt.p);
            CNN_HIP(hipGetLastError());
            exclusive_scan_i32_to_i64(ctx, wcnt.p, wptr->p, n);
            PinnedReads rd(ctx);
            const int64_t *last_excl = rd.get(wptr->p + (n - 1));
            const int32_t *last_cnt = rd.get(wcnt.p + (n - 1));
            rd.wait();
            const int64_t n_words = *last_excl + *last_cnt;
            set_i64(ctx, wptr->p + n, n_words);
            wtile.reset(new Scratch<int32_t>(ctx, n_words));
            wword.reset(new Scratch<uint64_t>(ctx, n_words));
            k_row_word_fill<<<blocks_for(n, 4), 256, 0, s>>>(req.row_ptr, req.col, n, wptr->p, wtile->p, wword->p);
            CNN_HIP(hipGetLastError());
            words = true;
            a.wptr = wptr->p;
            a.wtile = wtile->p;
            a.wword = wword->p;
        }
    }
    if (!words && !req.col) throw InvalidArg{"the sorted-list merge needs the neighbour lists"};

    Scratch<int32_t> cmin(ctx, n), csize(ctx, n);
    std::unique_ptr<Scratch<int32_t>> snewlab;
    if (req.sort) snewlab.reset(new Scratch<int32_t>(ctx, n));
    std::unique_ptr<Scratch<int32_t>> cnt(new Scratch<int32_t>(ctx, n));  // until the snapshot
    k_init<<<blocks_for(n), 256, 0, s>>>(a, req.consider, req.perm,
                                         ComponentArrays{cnt->p, cmin.p, csize.p, req.sort ? snewlab->p : nullptr},
                                         ClearList{{small.p}, {kSmallSlots}});
    CNN_HIP(hipGetLastError());
    CNN_HIP(hipEventRecord(ctx->ev[8], s));
    if (words && a.mask) {
        // within row tiles, then the rows left, one wave each
        Scratch<uint32_t> hq(ctx, n);
        unsigned int *const hq_len = (unsigned int *)(slot_p + 0);  // zeroed with the counters
        k_hook_tile<<<blocks_for(req.n_tiles, 4), 256, 0, s>>>(a, req.n_tiles, hq.p, hq_len);
        CNN_HIP(hipGetLastError());
        const unsigned qblocks = (unsigned)std::min<int64_t>(blocks_for(n, 4), 4096);
        k_hook_queue<<<qblocks, 256, 0, s>>>(a, hq.p, hq_len, 2);
    } else if (words) {
        k_hook<true><<<blocks_for(n, 4), 256, 0, s>>>(a, 2);
    } else {
        k_hook<false><<<blocks_for(n, 4), 256, 0, s>>>(a, 2);
    }
    CNN_HIP(hipGetLastError());
    CNN_HIP(hipEventRecord(ctx->ev[9], s));
    // lists: root_passes times flatten (every parent becomes its root) listing
    // the core roots, and let those re-point to smaller neighbouring roots.  On
    // tile-pair words the full round joins components for less (no pass against
    // two: 446 against 518 us a fit at n = 3e4, d = 3; 2.11 against 2.17 ms at
    // n = 1e6); on lists its tests run one row a wave and two passes save 8 to
    // 15 % of the label pass.
    if (req.root_passes > 0 && !(words && a.mask)) {
        Scratch<int32_t> roots(ctx, n);
        const unsigned rblocks = (unsigned)std::min<int64_t>(blocks_for(n, 4), 4096);
        const int threads = n < ((int64_t)1 << 18) ? 256 : 1024;
        for (int pass = 0; pass < req.root_passes; ++pass) {
            unsigned int *const n_roots = (unsigned int *)(slot_p + 2 + pass);  // zeroed with the counters
            k_compress_roots<<<blocks_for(n, threads), threads, 0, s>>>(parent.p, core.p, n, roots.p, n_roots);
            if (words) k_hook_roots_list<true><<<rblocks, 256, 0, s>>>(a, roots.p, n_roots, 4);
            else k_hook_roots_list<false><<<rblocks, 256, 0, s>>>(a, roots.p, n_roots, 4);
        }
    }
    CNN_HIP(hipGetLastError());
    const int steps = run_steps(n);
    std::unique_ptr<Scratch<uint64_t>> cand_max, tile_common;
    k_root_count<<<blocks_for(n, 256 * steps), 256, 0, s>>>(a, cnt->p, steps);
    if (req.n_tiles > 0) {
        Scratch<uint64_t> tmax(ctx, req.n_tiles);
        cand_max.reset(new Scratch<uint64_t>(ctx, req.n_tiles));
        tile_common.reset(new Scratch<uint64_t>(ctx, req.n_tiles));
        k_snapshot<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, cnt->p, n, rank.p, req.n_tiles, tmax.p,
                                                 tile_common->p);
        k_cand_max<<<blocks_for(req.n_tiles, 1), 256, 0, s>>>(tmax.p, req.tp_ptr, req.tp_col, req.n_tiles,
                                                              cand_max->p);
        CNN_HIP(hipGetLastError());
        a.cand_max = cand_max->p;
        a.tile_rank = tile_common->p;
    } else {
        k_snapshot<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, cnt->p, n, rank.p, 0, nullptr, nullptr);
        CNN_HIP(hipGetLastError());
        cnt.reset();
    }
    CNN_HIP(hipEventRecord(ctx->ev[10], s));
    if (words && a.mask && req.n_tiles > 0) {
        const int split = round_split(req.n_tile_pairs, req.n_tiles);
        a.rq_cap = round_queue_cap(req.n_tile_pairs, 1);
        Scratch<int2> rq(ctx, a.rq_cap);
        a.rq = rq.p;
        a.rq_len = slot_p + 1;  // zeroed with the counters
        k_round_tile<<<blocks_for(req.n_tiles * split, 4), 256, 0, s>>>(a, req.n_tiles, split);
        k_round_queue<<<(unsigned)std::min<int64_t>(blocks_for(a.rq_cap, 4), 2048), 256, 0, s>>>(a);
        a.rq = nullptr;
    } else if (words) k_round_b<true><<<blocks_for(n, 4), 256, 0, s>>>(a);
    else k_round_b<false><<<blocks_for(n, 4), 256, 0, s>>>(a);
    CNN_HIP(hipEventRecord(ctx->ev[11], s));
    CNN_HIP(hipGetLastError());
    CNN_HIP(hipEventRecord(ctx->ev[1], s));

    k_comp_stats<<<blocks_for(n, 256 * steps), 256, 0, s>>>(core.p, parent.p, req.perm, n, cmin.p, csize.p,
                                                            counters_p + 2, steps);
    CNN_HIP(hipGetLastError());
    // the cluster keys outlive the sort block: a fit with more clusters than
    // k_rank_clusters_small takes sorts them again after the final read
    std::unique_ptr<Scratch<uint64_t>> skeys;
    std::unique_ptr<Scratch<int32_t>> svals;
    bool big_sort = false;
    if (req.sort) {
        skeys.reset(new Scratch<uint64_t>(ctx, n));
        svals.reset(new Scratch<int32_t>(ctx, n));
        Scratch<uint64_t> &keys = *skeys;
        Scratch<int32_t> &vals = *svals, &newlab = *snewlab;
        if (req.packed) {
            // (only the packed keys: their top bits are the dataset, which
            // k_first_of_set and k_rank_clusters_packed use as an index)
            const PackedSort &ps = *req.packed;
            PackedKey pk{ps.ds_shift, ps.size_shift, ps.size_max, ps.tile_ds, ps.ds_offset};
            k_collect_clusters_packed<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, cmin.p, csize.p, n,
                                                                    req.member_cutoff, pk, counters_p + 5, keys.p,
                                                                    vals.p);
            CNN_HIP(hipGetLastError());
            const int64_t K = (int64_t)read_scalar(ctx, counters_p + 5);
            sort_pairs_u64_i32(ctx, keys.p, vals.p, K, ps.key_bits);
            if (K > 0) {
                Scratch<int32_t> first(ctx, ps.n_sets);
                k_first_of_set<<<blocks_for(K), 256, 0, s>>>(keys.p, K, ps.ds_shift, first.p);
                k_rank_clusters_packed<<<blocks_for(K), 256, 0, s>>>(keys.p, vals.p, K, ps.ds_shift, first.p,
                                                                     req.max_clusters, newlab.p, counters_p + 7);
                CNN_HIP(hipGetLastError());
            }
            k_write_sorted<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, newlab.p, req.perm, n, req.labels);
            CNN_HIP(hipGetLastError());
            local.n_clusters = (int64_t)read_scalar(ctx, counters_p + 7);
        } else {
            k_collect_clusters<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, cmin.p, csize.p, n,
                                                             req.member_cutoff, counters_p + 5, keys.p, vals.p);
            // up to kSmallClusters clusters sorted on the device; counters[4]
            // flags more, which the host sorts after the final read below
            k_rank_clusters_small<<<1, kSmallClusters, 0, s>>>(keys.p, vals.p, counters_p + 5, req.max_clusters,
                                                               newlab.p, counters_p + 4);
            k_write_sorted<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, newlab.p, req.perm, n, req.labels);
            CNN_HIP(hipGetLastError());
            big_sort = true;
        }
    } else {
        Scratch<uint8_t> isfirst(ctx, n);
        Scratch<int32_t> rank(ctx, n);
        fill_u8(ctx, isfirst.p, 0, n);
        k_mark_first<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, cmin.p, n, isfirst.p);
        CNN_HIP(hipGetLastError());
        inclusive_scan_u8_to_i32(ctx, isfirst.p, rank.p, n);
        k_write_unsorted<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, cmin.p, rank.p, req.perm, n, req.current_start,
                                                       req.write_all, req.labels);
        CNN_HIP(hipGetLastError());
    }
    if (req.consider) fill_u8(ctx, req.consider, 0, n);
    CNN_HIP(hipEventRecord(ctx->ev[2], s));
    unsigned long long h[8];
    unsigned long long ht[4 * kStatSlots];
    {
        PinnedReads rd(ctx);
        const unsigned long long *hp = rd.get(counters_p, 8 + 4 * kStatSlots);
        rd.wait();
        std::copy(hp, hp + 8, h);
        std::copy(hp + 8, hp + 8 + 4 * kStatSlots, ht);
    }
    if (big_sort) {
        const int64_t K = (int64_t)h[5];
        if (h[4]) {
            // more clusters than one workgroup sorts: sort them here and write the labels again
            fill_i32(ctx, snewlab->p, 0, n);
            sort_pairs_u64_i32(ctx, skeys->p, svals->p, K, 63);
            k_rank_clusters<<<blocks_for(K), 256, 0, s>>>(svals->p, K, req.max_clusters, snewlab->p);
            k_write_sorted<<<blocks_for(n), 256, 0, s>>>(core.p, parent.p, snewlab->p, req.perm, n, req.labels);
            CNN_HIP(hipGetLastError());
            CNN_HIP(hipStreamSynchronize(s));
        }
        local.n_clusters = (req.max_clusters >= 0) ? std::min<int64_t>(K, req.max_clusters) : K;
    }
    h[0] = h[1] = 0;
    unsigned long long rows = 0, sampled = 0;
    for (int i = 0; i < kStatSlots; ++i) {
        h[0] += ht[4 * i];
        h[1] += ht[4 * i + 1];
        rows += ht[4 * i + 2];
        sampled += ht[4 * i + 3];
    }
    local.sampled_components = (int64_t)sampled;
    local.rows_scanned = (int64_t)rows;
    float t1 = 0, t2 = 0;
    CNN_HIP(hipEventElapsedTime(&t1, ctx->ev[0], ctx->ev[1]));
    CNN_HIP(hipEventElapsedTime(&t2, ctx->ev[1], ctx->ev[2]));
    local.tests = (int64_t)h[0];
    local.tests_passed = (int64_t)h[1];
    local.n_core = (int64_t)h[2];
    local.n_components = (int64_t)h[3];
    if (!req.sort) local.n_clusters = local.n_components;
    local.ms_similarity = t1;
    local.ms_labels = t2;
    CNN_HIP(hipEventElapsedTime(&local.ms_hook, ctx->ev[8], ctx->ev[9]));
    CNN_HIP(hipEventElapsedTime(&local.ms_round, ctx->ev[10], ctx->ev[11]));
    local.sim_form = words ? (tile_words ? CNN_SIM_FORM_TILE_WORDS : CNN_SIM_FORM_ROW_WORDS) : CNN_SIM_FORM_MERGE;
    if (st) *st = local;
}

LabelRequest graph_label_request(cnn_ctx *ctx, const cnn_graph *g, int32_t sim_mode) {
    if (g->n > 0 && !g->col && (sim_mode == CNN_SIM_MERGE || !g->mask)) graph_lists(ctx, g);
    LabelRequest r{};
    r.row_ptr = g->row_ptr;
    r.col = g->col;
    r.n = g->n;
    r.perm = g->perm;
    r.sim_mode = sim_mode;
    r.current_start = 1;
    r.member_cutoff = 2;
    r.max_clusters = -1;
    r.tp_ptr = g->tp_ptr;
    r.tp_col = g->tp_col;
    r.n_tiles = g->n_tiles;
    r.selfpos = g->selfpos;
    r.mask = g->mask;
    r.pair_nz = g->pair_nz;
    r.diag = g->diag;
    r.tile_order = g->tile_order;
    r.n_tile_pairs = g->n_tile_pairs;
    r.root_passes = g->tune.root_passes;
    r.words_min_fill = g->tune.words_min_fill;
    return r;
}

// ------------------------------------------------------------------ several cutoff pairs, no host synchronisation

// sort_by_size of every cutoff pair without a library sort (a captured graph
// may hold no memset node, and library sorts record some): the clusters of
// pair y (roots of components with at least member_cutoff points) are
// collected with their keys (size descending, smallest original index
// ascending; all distinct), and each cluster's rank is the number of keys
// below its own, counted against LDS-staged chunks of the pair's keys --
// K^2 / 256 comparisons per block for K clusters.
__global__ void k_collect_multi(const uint8_t *core, const int *parent, const int32_t *cmin, const int32_t *csize,
                                int64_t n, int64_t member_cutoff, uint64_t *ckey, int32_t *cidx,
                                unsigned int *ccount) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t y = blockIdx.y, off = y * n;
    const bool cluster = w < n && core[off + w] && parent[off + w] == (int)w &&
                         (int64_t)csize[off + w] >= member_cutoff;
    const uint64_t b = __ballot(cluster);
    if (!b) return;
    const int lane = threadIdx.x & 63;
    unsigned base = 0;
    if (lane == 0) base = atomicAdd(&ccount[y], (unsigned)__popcll(b));
    base = __shfl(base, 0, 64);
    if (cluster) {
        const unsigned pos = base + (unsigned)__popcll(b & ((1ull << lane) - 1ull));
        ckey[off + pos] = ((uint64_t)(uint32_t)(0x7fffffff - csize[off + w]) << 32) | (uint32_t)cmin[off + w];
        cidx[off + pos] = (int32_t)w;
    }
}

__global__ __launch_bounds__(256) void k_rank_count(const uint64_t *ckey, const int32_t *cidx,
                                                    const unsigned int *ccount, int64_t n, int64_t max_clusters,
                                                    int32_t *newlab, unsigned long long *counters) {
    __shared__ uint64_t chunk[256];
    const int64_t y = blockIdx.y, off = y * n;
    const int64_t K = ccount[y];
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if ((int64_t)blockIdx.x * 256 >= K) return;  // whole block: uniform
    const uint64_t mine = x < K ? ckey[off + x] : ~0ull;
    int64_t rank = 0;
    for (int64_t base = 0; base < K; base += 256) {
        chunk[threadIdx.x] = base + threadIdx.x < K ? ckey[off + base + threadIdx.x] : ~0ull;
        __syncthreads();
        const int m = (int)min<int64_t>(256, K - base);
        for (int t = 0; t < m; ++t) rank += chunk[t] < mine ? 1 : 0;
        __syncthreads();
    }
    const bool keep = x < K && (max_clusters < 0 || rank < max_clusters);
    if (keep) newlab[off + cidx[off + x]] = (int32_t)(rank + 1);
    const uint64_t b = __ballot(keep);
    if ((threadIdx.x & 63) == 0 && b) atomicAdd(&counters[8 * y + 7], (unsigned long long)__popcll(b));
}

void multi_labels_bytes(int64_t n, int64_t n_tiles, int64_t n_tile_pairs, int n_c, MultiLabelSizes &sz) {
    sz.per_point = n * n_c;
    sz.per_tile = std::max<int64_t>(n_tiles, 1) * n_c;
    sz.round_queue = round_queue_cap(n_tile_pairs, n_c);
}

void labels_enqueue_multi(cnn_ctx *ctx, const MultiLabelBufs &b, const MultiLabelSource &src, int64_t member_cutoff,
                          int64_t max_clusters, int64_t *labels, unsigned long long *counters,
                          unsigned long long *tstats) {
    hipStream_t s = ctx->stream;
    const int64_t n = b.n, T = b.n_tiles;
    const unsigned nc = (unsigned)b.n_c;
    if (n == 0 || nc == 0) return;
    unsigned int *const hq_len = b.lens, *const ccount = b.lens + nc;
    LabelArgs a{};
    a.n = n;
    a.core = b.core;
    a.parent = b.parent;
    a.stats = tstats;
    a.rank = b.rank;
    a.mask = src.mask;
    a.pair_nz = src.pair_nz;
    a.tp_ptr = src.tp_ptr;
    a.tp_col = src.tp_col;
    a.deg = src.deg;
    a.csim_y = b.csim;
    a.mcore_y = b.mcore;
    a.tiles = T;
    auto g2 = [&](int64_t items, int per) { return dim3(blocks_for(items, per), nc); };
    const unsigned waves = (unsigned)std::min<int64_t>(blocks_for(n, 4), 4096);
    k_init<<<g2(n, 256), 256, 0, s>>>(a, nullptr, src.perm, ComponentArrays{b.cnt, b.cmin, b.csize, b.newlab},
                                         ClearList{{counters, b.rq_len, tstats, (unsigned long long *)b.lens},
                                                   {8 * (int64_t)nc, (int64_t)nc, 4 * (int64_t)kStatSlots * nc,
                                                    (int64_t)nc}});
    k_hook_tile<<<g2(T, 4), 256, 0, s>>>(a, T, b.hq, hq_len);
    k_hook_queue<<<dim3(waves, nc), 256, 0, s>>>(a, b.hq, hq_len, 2);
    CNN_HIP(hipGetLastError());
    const int steps = run_steps(n * nc);
    k_root_count<<<g2(n, 256 * steps), 256, 0, s>>>(a, b.cnt, steps);
    k_snapshot<<<g2(n, 256), 256, 0, s>>>(b.core, b.parent, b.cnt, n, b.rank, T, b.tmax, b.tile_common);
    k_cand_max<<<g2(T, 1), 256, 0, s>>>(b.tmax, src.tp_ptr, src.tp_col, T, b.cand_max);
    CNN_HIP(hipGetLastError());
    a.cand_max = b.cand_max;
    a.tile_rank = b.tile_common;
    const int split = round_split(src.n_tile_pairs * nc, T * nc);
    a.rq = b.rq;
    a.rq_len = b.rq_len;
    a.rq_cap = b.rq_cap;
    k_round_tile<<<g2(T * split, 4), 256, 0, s>>>(a, T, split);
    k_round_queue<<<dim3((unsigned)std::min<int64_t>(blocks_for(a.rq_cap, 4), 2048), nc), 256, 0, s>>>(a);
    k_comp_stats<<<g2(n, 256 * steps), 256, 0, s>>>(b.core, b.parent, src.perm, n, b.cmin, b.csize, counters + 2,
                                                    steps);
    k_collect_multi<<<g2(n, 256), 256, 0, s>>>(b.core, b.parent, b.cmin, b.csize, n, member_cutoff, b.ckey,
                                               b.cidx, ccount);
    k_rank_count<<<g2(n, 256), 256, 0, s>>>(b.ckey, b.cidx, ccount, n, max_clusters, b.newlab, counters);
    k_write_sorted<<<g2(n, 256), 256, 0, s>>>(b.core, b.parent, b.newlab, src.perm, n, labels);
    CNN_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ caller CSR validation

// Flags rows that are not strictly ascending or hold indices outside [0, n),
// offsets that decrease, and a bad first or last offset; one wave per row (one
// thread per row took 90 us for 8001 rows of 640 entries, 4 us as here).
// Precondition (caller contract): col holds at least row_ptr[n] entries and
// row_ptr is n+1 long.
__global__ __launch_bounds__(256) void k_validate_csr(const int64_t *__restrict__ row_ptr,
                                                      const int32_t *__restrict__ col, int64_t n,
                                                      unsigned long long *bad) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= n) return;
    const int64_t b = row_ptr[w], e = row_ptr[w + 1], nnz = row_ptr[n];
    if (w == 0 && lane == 0 && (b != 0 || nnz < 0)) atomicOr(bad, 4ull);
    if (b < 0 || e < b || e > nnz) {
        if (lane == 0) atomicOr(bad, 1ull);
        return;
    }
    bool wrong = false;
    for (int64_t t = b + lane; t < e; t += 64) {
        const int32_t j = col[t], prev = t > b ? col[t - 1] : -1;
        wrong = wrong || j <= prev || (int64_t)j >= n;
    }
    if (__ballot(wrong) != 0ull && lane == 0) atomicOr(bad, 2ull);
}

int64_t validate_csr(cnn_ctx *ctx, const int64_t *row_ptr, const int32_t *col, int64_t n) {
    if (n == 0) return 0;
    Scratch<unsigned long long> bad(ctx, 1);
    fill_u64(ctx, bad.p, 0ull, 1);
    k_validate_csr<<<(unsigned)ceil_div(n, 4), 256, 0, ctx->stream>>>(row_ptr, col, n, bad.p);
    CNN_HIP(hipGetLastError());
    PinnedReads rd(ctx);
    const unsigned long long *flags = rd.get(bad.p);
    const int64_t *nnz = rd.get(row_ptr + n);
    rd.wait();
    if (*flags & 4ull) throw InvalidArg{"row_ptr must start at 0 and end at nnz >= 0"};
    if (*flags & 1ull) throw InvalidArg{"row_ptr is not non-decreasing within [0, nnz]"};
    if (*flags & 2ull) throw InvalidArg{"neighbour rows must be strictly ascending with indices in [0, n)"};
    return *nnz;
}

// ------------------------------------------------------------------ generic sort_by_size

__global__ void k_iota(int32_t *v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = (int32_t)i;
}

__global__ void k_heads(const int64_t *keys, int64_t n, uint8_t *head) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    head[t] = (t == 0 || keys[t] != keys[t - 1]) ? 1 : 0;
}

__global__ void k_segments(const int64_t *keys, const int32_t *vals, const int32_t *segid, int64_t n,
                           int32_t *seg_start, int32_t *seg_end) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int sid = segid[t] - 1;
    if (t == 0 || keys[t] != keys[t - 1]) seg_start[sid] = (int32_t)t;
    if (t == n - 1 || keys[t + 1] != keys[t]) seg_end[sid] = (int32_t)t;
}

__global__ void k_seg_collect(const int64_t *keys, const int32_t *vals, const int32_t *seg_start,
                              const int32_t *seg_end, const int32_t *n_seg, unsigned long long *K, uint64_t *okeys,
                              int32_t *ovals) {
    int64_t sid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (sid >= *n_seg) return;
    const int32_t b = seg_start[sid];
    if (keys[b] == 0) return;
    const int32_t sz = seg_end[sid] - b + 1;
    const unsigned long long idx = atomicAdd(K, 1ull);
    okeys[idx] = ((uint64_t)(uint32_t)(0x7fffffff - sz) << 32) | (uint32_t)vals[b];
    ovals[idx] = (int32_t)sid;
}

__global__ void k_seg_rank(const uint64_t *okeys, const int32_t *ovals, int64_t K, int64_t member_cutoff,
                           int64_t max_clusters, int32_t *seglab) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= K) return;
    const int64_t sz = 0x7fffffff - (int64_t)(okeys[t] >> 32);
    const bool keep = (max_clusters < 0 || t < max_clusters) && sz >= member_cutoff;
    seglab[ovals[t]] = keep ? (int32_t)(t + 1) : 0;
}

__global__ void k_seg_write(const int32_t *vals, const int32_t *segid, const int32_t *seglab, int64_t n,
                            int64_t *labels) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    labels[vals[t]] = seglab[segid[t] - 1];
}

// sort_by_size through a table over the labels 0 .. n (what the fits assign):
// members and first index per label, the clusters collected and ranked by
// k_rank_clusters_small, labels rewritten.  flags[0] clusters, [1] a label outside
// the table, [2] more clusters than that kernel ranks: nothing is written then.
//
// Runs of one label cost one update; a workgroup counts the first kLabelLds labels
// in LDS, so that labels in any order meet a few hundred updates an address in
// memory (updates from every wave: 930 us for 1e6 points of 5 clusters in random
// order, the sort 320, as here 50).
constexpr int kLabelLds = 2048;
constexpr int kLabelBlocks = 256;

__global__ __launch_bounds__(256) void k_label_table(const int64_t *__restrict__ labels, int64_t n,
                                                     int32_t *__restrict__ cnt, int32_t *__restrict__ first,
                                                     unsigned long long *__restrict__ flags) {
    __shared__ int32_t s_cnt[kLabelLds], s_first[kLabelLds];
    for (int t = threadIdx.x; t < kLabelLds; t += 256) {
        s_cnt[t] = 0;
        s_first[t] = INT_MAX;
    }
    __syncthreads();
    auto add = [&](int key, int count, int at) {
        if (key < kLabelLds) {
            atomicAdd(&s_cnt[key], count);
            atomicMin(&s_first[key], at);
        } else {
            atomicAdd(&cnt[key], count);
            atomicMin(&first[key], at);
        }
    };
    const int lane = __lane_id();
    const int64_t waves = (int64_t)gridDim.x * 4, wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int64_t per = ((n + waves - 1) / waves + 63) / 64 * 64;  // a wave's points, consecutive
    const int64_t end = min(n, (wave + 1) * per);
    bool outside = false;
    KeyRun run;
    constexpr int kU = 4;  // steps of 64 points loaded together
    for (int64_t i0 = wave * per; i0 < end; i0 += 64 * kU) {
        // another wave met a label outside: the table is not used
        if (__hip_atomic_load(&flags[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        int64_t l[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int64_t i = i0 + 64 * u + lane;
            l[u] = i < end ? labels[i] : 0;
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool in = l[u] >= 0 && l[u] <= n;
            if (__ballot(!in) != 0ull && !outside) {
                outside = true;
                if (lane == 0) __hip_atomic_store(&flags[1], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            const int key = in ? (int)l[u] : 0;
            const uint64_t act = __ballot(key != 0);
            if (!act) continue;
            const int at = (int)(i0 + 64 * u), lead = __ffsll((unsigned long long)act) - 1;
            const int k = __shfl(key, lead, 64);
            if (__ballot(key != 0 && key != k) != 0ull) {
                if (key != 0) add(key, 1, at + lane);
                continue;
            }
            if (k != run.key) {
                if (run.key >= 0 && lane == 0) add(run.key, run.cnt, run.mn);
                run.key = k;
                run.cnt = 0;
                run.mn = at + lead;
            }
            run.cnt += __popcll(act);
        }
    }
    if (run.key >= 0 && lane == 0) add(run.key, run.cnt, run.mn);
    __syncthreads();
    for (int t = threadIdx.x; t < kLabelLds; t += 256)
        if (s_cnt[t]) {
            atomicAdd(&cnt[t], s_cnt[t]);
            atomicMin(&first[t], s_first[t]);
        }
}

__global__ void k_label_clusters(const int32_t *__restrict__ cnt, const int32_t *__restrict__ first, int64_t n,
                                 int64_t member_cutoff, unsigned long long *__restrict__ K, uint64_t *__restrict__ keys,
                                 int32_t *__restrict__ vals) {
    const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l > n || K[1] || cnt[l] == 0 || (int64_t)cnt[l] < member_cutoff) return;  // K[1]: a label outside
    const unsigned long long idx = atomicAdd(K, 1ull);
    keys[idx] = ((uint64_t)(uint32_t)(0x7fffffff - cnt[l]) << 32) | (uint32_t)first[l];
    vals[idx] = (int32_t)l;
}

__global__ void k_label_rewrite(int64_t *__restrict__ labels, int64_t n, const int32_t *__restrict__ newlab,
                                const unsigned long long *__restrict__ flags) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && !(flags && (flags[1] || flags[2]))) labels[i] = newlab[labels[i]];
}

__global__ void k_label_clear(int32_t *cnt, int32_t *first, int32_t *newlab, int64_t count,
                              unsigned long long *flags) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 3) flags[i] = 0ull;
    if (i >= count) return;
    cnt[i] = 0;
    first[i] = INT_MAX;
    newlab[i] = 0;
}

// The number of clusters kept, or -1 when the table does not cover the labels
// (they are unchanged then).
static int64_t sort_by_size_table(cnn_ctx *ctx, int64_t *labels, int64_t n, int64_t member_cutoff,
                                  int64_t max_clusters) {
    hipStream_t s = ctx->stream;
    Scratch<int32_t> cnt(ctx, n + 1), first(ctx, n + 1), newlab(ctx, n + 1), vals(ctx, n + 1);
    Scratch<uint64_t> keys(ctx, n + 1);
    Scratch<unsigned long long> flags(ctx, 3);
    k_label_clear<<<blocks_for(n + 1), 256, 0, s>>>(cnt.p, first.p, newlab.p, n + 1, flags.p);
    k_label_table<<<std::min<unsigned>(blocks_for(n), kLabelBlocks), 256, 0, s>>>(labels, n, cnt.p, first.p, flags.p);
    k_label_clusters<<<blocks_for(n + 1), 256, 0, s>>>(cnt.p, first.p, n, member_cutoff, flags.p, keys.p, vals.p);
    k_rank_clusters_small<<<1, kSmallClusters, 0, s>>>(keys.p, vals.p, flags.p, max_clusters, newlab.p, flags.p + 2);
    k_label_rewrite<<<blocks_for(n), 256, 0, s>>>(labels, n, newlab.p, flags.p);
    CNN_HIP(hipGetLastError());
    PinnedReads rd(ctx);
    const unsigned long long *h = rd.get(flags.p, 3);
    rd.wait();
    if (h[1]) return -1;
    const int64_t K = (int64_t)h[0];
    if (h[2]) {  // more clusters than one workgroup ranks: their keys are sorted
        sort_pairs_u64_i32(ctx, keys.p, vals.p, K, 63);
        k_rank_clusters<<<blocks_for(K), 256, 0, s>>>(vals.p, K, max_clusters, newlab.p);
        k_label_rewrite<<<blocks_for(n), 256, 0, s>>>(labels, n, newlab.p, nullptr);
        CNN_HIP(hipGetLastError());
        CNN_HIP(hipStreamSynchronize(s));
    }
    return max_clusters >= 0 ? std::min<int64_t>(K, max_clusters) : K;
}

int64_t sort_by_size_generic(cnn_ctx *ctx, int64_t *labels, int64_t n, int64_t member_cutoff, int64_t max_clusters) {
    hipStream_t s = ctx->stream;
    if (n == 0) return 0;
    if (n >= (int64_t)INT32_MAX) throw InvalidArg{"n exceeds the int32 index range"};
    // labels as the fits assign them (0 .. n) need no sort of the points: five
    // kernels and one host read against 22 launches and four reads
    // (n = 8000: 47 against 330 us of a traced call)
    const int64_t kept_small = sort_by_size_table(ctx, labels, n, member_cutoff, max_clusters);
    if (kept_small >= 0) return kept_small;
    Scratch<int64_t> keys(ctx, n);
    Scratch<int32_t> vals(ctx, n), segid(ctx, n);
    Scratch<uint8_t> head(ctx, n);
    CNN_HIP(hipMemcpyAsync(keys.p, labels, n * sizeof(int64_t), hipMemcpyDeviceToDevice, s));
    k_iota<<<blocks_for(n), 256, 0, s>>>(vals.p, n);
    CNN_HIP(hipGetLastError());
    sort_pairs_i64_i32(ctx, keys.p, vals.p, n);  // stable: equal labels keep ascending index
    k_heads<<<blocks_for(n), 256, 0, s>>>(keys.p, n, head.p);
    inclusive_scan_u8_to_i32(ctx, head.p, segid.p, n);
    // segid[n - 1] segments, at most n: the count stays on the device
    Scratch<int32_t> seg_start(ctx, n), seg_end(ctx, n), seglab(ctx, n);
    k_segments<<<blocks_for(n), 256, 0, s>>>(keys.p, vals.p, segid.p, n, seg_start.p, seg_end.p);
    fill_i32(ctx, seglab.p, 0, n);
    Scratch<unsigned long long> K(ctx, 1);
    fill_u64(ctx, K.p, 0ull, 1);
    Scratch<uint64_t> okeys(ctx, n);
    Scratch<int32_t> ovals(ctx, n);
    k_seg_collect<<<blocks_for(n), 256, 0, s>>>(keys.p, vals.p, seg_start.p, seg_end.p, segid.p + (n - 1), K.p, okeys.p,
                                                ovals.p);
    CNN_HIP(hipGetLastError());
    const int64_t k = (int64_t)read_scalar(ctx, K.p);
    sort_pairs_u64_i32(ctx, okeys.p, ovals.p, k, 63);
    if (k > 0) k_seg_rank<<<blocks_for(k), 256, 0, s>>>(okeys.p, ovals.p, k, member_cutoff, max_clusters, seglab.p);
    k_seg_write<<<blocks_for(n), 256, 0, s>>>(vals.p, segid.p, seglab.p, n, labels);
    CNN_HIP(hipGetLastError());
    // number of survivors
    int64_t kept = 0;
    if (k > 0) {
        std::vector<uint64_t> hk(k);
        CNN_HIP(hipMemcpyAsync(hk.data(), okeys.p, k * sizeof(uint64_t), hipMemcpyDeviceToHost, s));
        CNN_HIP(hipStreamSynchronize(s));
        for (int64_t t = 0; t < k; ++t) {
            const int64_t sz = 0x7fffffff - (int64_t)(hk[t] >> 32);
            if ((max_clusters < 0 || t < max_clusters) && sz >= member_cutoff) ++kept;
        }
    } else {
        CNN_HIP(hipStreamSynchronize(s));
    }
    return kept;
}

}  // namespace cnn

// ================================================================== C-ABI: phase S+U
using namespace cnn;

extern "C" {

int cnn_labels_from_csr(cnn_ctx *ctx, const int64_t *row_ptr, const int32_t *col, int64_t n, int32_t c_sim,
                        int32_t m_core, uint8_t *consider, int64_t current_start, int32_t sim_mode, int64_t *labels,
                        cnn_label_stats *stats_out) {
    if (!ctx) return CNN_ERR_INVALID;
    return guarded(ctx, [&]() {
        if (n < 0) throw InvalidArg{"negative n"};
        if (n > 0 && (!row_ptr || !col || !labels)) throw InvalidArg{"null buffer"};
        if (n >= (int64_t)INT32_MAX) throw InvalidArg{"n exceeds the int32 index range"};
        CNN_HIP(hipSetDevice(ctx->device));
        const int64_t nnz = validate_csr(ctx, row_ptr, col, n);
        LabelRequest r{row_ptr, col, n, nullptr, c_sim, m_core, consider, current_start, sim_mode,
                       false, false, 2, -1, labels};
        r.nnz = nnz;
        const TuneParams t = tune_lookup(0, n, CNN_PLAIN_F64);
        r.root_passes = t.root_passes;
        r.words_min_fill = t.words_min_fill;
        labels_run(ctx, r, stats_out);
        return (int)CNN_OK;
    });
}

int cnn_graph_labels(cnn_ctx *ctx, const cnn_graph *g, int32_t c_sim, int32_t m_core, uint8_t *consider,
                     int64_t current_start, int32_t sim_mode, int64_t *labels, cnn_label_stats *stats_out) {
    if (!ctx || !g) return CNN_ERR_INVALID;
    return guarded(ctx, [&]() {
        if (g->n > 0 && !labels) throw InvalidArg{"null labels"};
        CNN_HIP(hipSetDevice(ctx->device));
        if (sim_mode != CNN_SIM_AUTO && sim_mode != CNN_SIM_MERGE && sim_mode != CNN_SIM_BITSET)
            throw InvalidArg{"unknown sim_mode"};
        LabelRequest r = graph_label_request(ctx, g, sim_mode);
        r.c_sim = c_sim;
        r.m_core = m_core;
        r.consider = consider;
        r.current_start = current_start;
        r.labels = labels;
        labels_run(ctx, r, stats_out);
        return (int)CNN_OK;
    });
}

int cnn_sort_by_size(cnn_ctx *ctx, int64_t *labels, int64_t n, int64_t member_cutoff, int64_t max_clusters,
                     int64_t *n_clusters_out) {
    if (!ctx) return CNN_ERR_INVALID;
    return guarded(ctx, [&]() {
        if (n < 0) throw InvalidArg{"negative n"};
        if (n > 0 && !labels) throw InvalidArg{"null labels"};
        CNN_HIP(hipSetDevice(ctx->device));
        int64_t k = sort_by_size_generic(ctx, labels, n, member_cutoff, max_clusters);
        if (n_clusters_out) *n_clusters_out = k;
        return (int)CNN_OK;
    });
}

int cnn_graph_fit(cnn_ctx *ctx, const cnn_graph *g, int32_t c_sim, int32_t m_core, int32_t sort,
                  int64_t member_cutoff, int64_t max_clusters, int64_t *labels, cnn_label_stats *lstats) {
    if (!ctx || !g) return CNN_ERR_INVALID;
    return guarded(ctx, [&]() {
        if (g->n > 0 && !labels) throw InvalidArg{"null labels"};
        CNN_HIP(hipSetDevice(ctx->device));
        LabelRequest r = graph_label_request(ctx, g, CNN_SIM_AUTO);
        r.c_sim = c_sim;
        r.m_core = m_core;
        r.sort = sort != 0;
        r.write_all = true;
        r.member_cutoff = member_cutoff;
        r.max_clusters = max_clusters;
        r.labels = labels;
        labels_run(ctx, r, lstats);
        return (int)CNN_OK;
    });
}

int cnn_fit(cnn_ctx *ctx, const void *X, int64_t n, int32_t d, int32_t dtype, double r2, int32_t c_sim,
            int32_t m_core, int32_t precision, int32_t sort, int64_t member_cutoff, int64_t max_clusters,
            int64_t *labels, cnn_graph **graph_out, cnn_graph_stats *gstats, cnn_label_stats *lstats) {
    if (!ctx) return CNN_ERR_INVALID;
    if (graph_out) *graph_out = nullptr;
    return guarded(ctx, [&]() {
        if (n > 0 && !labels) throw InvalidArg{"null labels"};
        CNN_HIP(hipSetDevice(ctx->device));
        cnn_graph *g = graph_build(ctx, X, n, d, dtype, r2, precision, nullptr, graph_out == nullptr);
        std::unique_ptr<cnn_graph, void (*)(cnn_graph *)> hold(g, graph_free);
        if (gstats) *gstats = g->stats;
        LabelRequest r = graph_label_request(ctx, g, CNN_SIM_AUTO);
        r.c_sim = c_sim;
        r.m_core = m_core;
        r.sort = sort != 0;
        r.write_all = true;
        r.member_cutoff = member_cutoff;
        r.max_clusters = max_clusters;
        r.labels = labels;
        labels_run(ctx, r, lstats);
        if (graph_out) *graph_out = hold.release();
        return (int)CNN_OK;
    });
}

}  // extern "C"
