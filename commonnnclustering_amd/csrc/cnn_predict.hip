// Label prediction for a second point set: PredictorFirstmatch.predict
// (_fit.pyx:1241-1291) called by Clustering.predict (cluster.pyx:560-653).
//
// For every considered point p of Y, the reference points within r of it
// (NeighboursGetterExtBruteForce._get_other, _types.pyx:1712-1731: same metric,
// operands swapped, which leaves every squared difference unchanged) are
// visited in ascending reference index; p needs more than m_core of them.  The
// first member whose label is allowed, whose own neighbourhood among the
// reference points has more than m_core entries and with which p shares at
// least c_sim reference neighbours gives p its label and clears p's consider
// flag.  Other points of Y keep label and flag.
//
// Device procedure: one radius graph over the concatenation [X; Y] (same
// kernels and precision forms as a fit); one wave per row of Y walks its
// reference neighbours in ascending reference index: each step takes the
// smallest index above the last one tested (a wave minimum) and tests the
// similarity with that member.
// On a graph that holds its tile-pair words, rows are read from them with the
// reference columns of each tile as a mask, and no lists exist.  Otherwise the
// lists are emitted and every list is cut to its reference points (N_X(m) for
// reference rows, the cross list for rows of Y).  n_x = 1e5, d = 3, 300
// neighbours: 1.03 ms through the lists (emission, two passes that cut them and
// the merges 0.6 ms of it), 0.70 ms on the words.
#include <algorithm>
#include <memory>

#include "cnn_internal.hpp"

namespace cnn {

__device__ __forceinline__ int32_t caller_of(const int32_t *perm, int64_t w) {
    return perm ? perm[w] : (int32_t)w;
}

// Entries whose point is a reference point (caller index < n_x), per row:
// counted (FILL = false) or written in list order (FILL = true).
template <bool FILL>
__global__ __launch_bounds__(256) void k_keep_ref(const int64_t *__restrict__ row_ptr,
                                                  const int32_t *__restrict__ col, const int32_t *__restrict__ perm,
                                                  int64_t n, int64_t n_x, int32_t *__restrict__ cnt,
                                                  const int64_t *__restrict__ out_ptr, int32_t *__restrict__ out_col) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= n) return;
    const int64_t b = row_ptr[w], e = row_ptr[w + 1];
    int64_t pos = FILL ? out_ptr[w] : 0;
    int kept = 0;
    for (int64_t t0 = b; t0 < e; t0 += 64) {
        const int64_t t = t0 + lane;
        const int32_t j = t < e ? col[t] : 0;
        const bool keep = t < e && caller_of(perm, j) < n_x;
        const uint64_t m = __ballot(keep);
        if (FILL && keep) {
            const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            out_col[pos + rank] = j;
        }
        pos += __popcll(m);
        kept += __popcll(m);
    }
    if (!FILL && lane == 0) cnt[w] = kept;
}

// Per working row of a reference point: its label, and whether it may give
// its label (label allowed and more than m_core reference neighbours).
__global__ void k_ref_members(const int64_t *__restrict__ rp, const int32_t *__restrict__ perm, int64_t n,
                              int64_t n_x, int32_t m_core, const int64_t *__restrict__ labels_x,
                              const uint8_t *__restrict__ allowed, int64_t n_allowed, int64_t *__restrict__ lab,
                              uint8_t *__restrict__ ok) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n) return;
    const int32_t o = caller_of(perm, w);
    bool good = false;
    int64_t l = 0;
    if (o < n_x) {
        l = labels_x[o];
        good = (rp[w + 1] - rp[w]) > (int64_t)m_core && l >= 0 && l < n_allowed && allowed[l] != 0;
    }
    lab[w] = l;
    ok[w] = good ? 1 : 0;
}

// One wave per working row of a point of Y.
__global__ __launch_bounds__(256) void k_predict_rows(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                      const int32_t *__restrict__ perm, int64_t n, int64_t n_x,
                                                      int32_t c_sim, int32_t m_core, const int64_t *__restrict__ lab,
                                                      const uint8_t *__restrict__ ok, int64_t *__restrict__ labels_y,
                                                      uint8_t *__restrict__ consider_y,
                                                      unsigned long long *__restrict__ tests) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= n) return;
    const int32_t o = caller_of(perm, w);
    if (o < n_x) return;
    const int64_t q = (int64_t)o - n_x;
    if (!consider_y[q]) return;
    const int64_t b = rp[w], e = rp[w + 1];
    if (e - b <= (int64_t)m_core) return;
    unsigned n_tests = 0;
    int64_t last = -1;  // reference index of the last member tested
    for (;;) {
        // next member: the smallest reference index above `last` among the usable ones
        uint64_t best = ~0ull;  // (reference index << 32) | working row
        for (int64_t t0 = b; t0 < e; t0 += 64) {
            const int64_t t = t0 + lane;
            if (t < e) {
                const int32_t j = col[t];
                const int32_t cj = caller_of(perm, j);
                if (ok[j] && (int64_t)cj > last) {
                    const uint64_t key = ((uint64_t)(uint32_t)cj << 32) | (uint32_t)j;
                    best = key < best ? key : best;
                }
            }
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const uint64_t other = __shfl_xor(best, off, 64);
            best = other < best ? other : best;
        }
        if (best == ~0ull) break;
        const int32_t jm = (int32_t)(uint32_t)best;
        ++n_tests;
        if (wave_sim(col + b, e - b, col + rp[jm], rp[jm + 1] - rp[jm], c_sim)) {
            if (lane == 0) {
                labels_y[q] = lab[jm];
                consider_y[q] = 0;
            }
            break;
        }
        last = (int64_t)(best >> 32);
    }
    if (lane == 0 && n_tests) atomicAdd(tests, (unsigned long long)n_tests);
}

// Per tile, the columns that are reference points.
__global__ __launch_bounds__(256) void k_ref_tiles(const int32_t *__restrict__ perm, int64_t n, int64_t n_x,
                                                   int64_t n_tiles, uint64_t *__restrict__ ref) {
    const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const uint64_t m = __ballot(w < n && caller_of(perm, w) < n_x);
    if ((threadIdx.x & 63) == 0 && (w >> 6) < n_tiles) ref[w >> 6] = m;
}

// Reference neighbours per row, and the key a row offers as a member: its
// caller index when it is a reference point that may give its label, else all
// ones.  One workgroup per row tile (lane = row), its waves every fourth window
// of 64 pairs, eight pairs' words in flight.
__global__ __launch_bounds__(256) void k_ref_keys(const uint64_t *__restrict__ mask, const uint8_t *__restrict__ nz,
                                                  const int64_t *__restrict__ tp_ptr,
                                                  const int32_t *__restrict__ tp_col,
                                                  const uint64_t *__restrict__ ref, const int32_t *__restrict__ perm,
                                                  int64_t n, int64_t n_x, int32_t m_core,
                                                  const int64_t *__restrict__ labels_x,
                                                  const uint8_t *__restrict__ allowed, int64_t n_allowed,
                                                  int32_t *__restrict__ rdeg, uint32_t *__restrict__ key) {
    __shared__ int s_deg[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t R = blockIdx.x;
    const int64_t kb = tp_ptr[R], ke = tp_ptr[R + 1];
    int deg = 0;
    for (int64_t k0 = kb + 64 * wave; k0 < ke; k0 += 256) {
        const int64_t kk = k0 + lane;
        const bool on = kk < ke && nz[kk] != 0;
        const uint64_t rm = on ? ref[tp_col[kk]] : 0ull;
        uint64_t todo = __ballot(rm != 0ull);
        while (todo) {
            uint64_t v[8], m[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                v[u] = m[u] = 0ull;
                if (todo) {
                    const int q = __ffsll((unsigned long long)todo) - 1;
                    todo &= todo - 1;
                    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)rm, q);
                    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(rm >> 32), q);
                    m[u] = ((uint64_t)hi << 32) | lo;
                    v[u] = mask[(k0 + q) * 64 + lane];
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) deg += __popcll(v[u] & m[u]);
        }
    }
    s_deg[wave][lane] = deg;
    __syncthreads();
    const int64_t w = R * 64 + lane;
    if (wave != 0 || w >= n) return;
    deg = s_deg[0][lane] + s_deg[1][lane] + s_deg[2][lane] + s_deg[3][lane];
    rdeg[w] = deg;
    const int32_t o = caller_of(perm, w);
    bool good = false;
    if (o < n_x && deg > m_core) {
        const int64_t l = labels_x[o];
        good = l >= 0 && l < n_allowed && allowed[l] != 0;
    }
    key[w] = good ? (uint32_t)o : 0xffffffffu;
}

// One wave per working row of a point of Y, on tile-pair words.
__global__ __launch_bounds__(256) void k_predict_words(
    const uint64_t *__restrict__ mask, const uint8_t *__restrict__ nz, const int64_t *__restrict__ tp_ptr,
    const int32_t *__restrict__ tp_col, const uint64_t *__restrict__ ref, const int32_t *__restrict__ rdeg,
    const uint32_t *__restrict__ key, const int32_t *__restrict__ perm, int64_t n, int64_t n_x, int32_t c_sim,
    int32_t m_core, const int64_t *__restrict__ labels_x, int64_t *__restrict__ labels_y,
    uint8_t *__restrict__ consider_y, unsigned long long *__restrict__ tests) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= n) return;
    const int32_t o = caller_of(perm, w);
    if (o < n_x) return;
    const int64_t q = (int64_t)o - n_x;
    if (!consider_y[q] || rdeg[w] <= m_core) return;
    auto row_of = [&](int64_t r) {
        const int64_t R = r >> 6, kb = tp_ptr[R];
        return WordRow{tp_col + kb, mask + kb * 64 + (r & 63), nz + kb, tp_ptr[R + 1] - kb, 64};
    };
    const WordRow A = row_of(w);
    unsigned n_tests = 0;
    int64_t last = -1;  // reference index of the last member tested
    for (;;) {
        // next member: the smallest reference index above `last` among the usable
        // ones; lane = column, one tile of the row after another, eight in flight
        uint64_t best = ~0ull;  // (reference index << 32) | working row
        for (int64_t t0 = 0; t0 < A.len; t0 += 64) {
            const int64_t t = t0 + lane;
            uint64_t v = 0ull;
            int C = 0;
            if (t < A.len) {
                C = A.tile[t];
                v = word_at(A, t) & ref[C];
            }
            uint64_t todo = __ballot(v != 0ull);
            while (todo) {
                uint32_t kv[8];
                int cs[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    kv[u] = 0xffffffffu;
                    cs[u] = 0;
                    if (todo) {
                        const int s = __ffsll((unsigned long long)todo) - 1;
                        todo &= todo - 1;
                        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, s);
                        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), s);
                        cs[u] = __builtin_amdgcn_readlane(C, s);
                        if ((lane < 32 ? lo >> lane : hi >> (lane - 32)) & 1u) kv[u] = key[cs[u] * 64 + lane];
                    }
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    if (kv[u] != 0xffffffffu && (int64_t)kv[u] > last) {
                        const uint64_t x = ((uint64_t)kv[u] << 32) | (uint32_t)(cs[u] * 64 + lane);
                        best = x < best ? x : best;
                    }
                }
            }
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const uint64_t other = __shfl_xor(best, off, 64);
            best = other < best ? other : best;
        }
        if (best == ~0ull) break;
        const int64_t jm = (int64_t)(uint32_t)best, oj = (int64_t)(best >> 32);
        ++n_tests;
        if (wave_sim_words(A, row_of(jm), c_sim, ref)) {
            if (lane == 0) {
                labels_y[q] = labels_x[oj];
                consider_y[q] = 0;
            }
            break;
        }
        last = oj;
    }
    if (lane == 0 && n_tests) atomicAdd(tests, (unsigned long long)n_tests);
}

}  // namespace cnn

using namespace cnn;

extern "C" {

int cnn_predict(cnn_ctx *ctx, const void *X, int64_t n_x, const void *Y, int64_t n_y, int32_t d, int32_t dtype,
                double r2, int32_t precision, int32_t c_sim, int32_t m_core, const int64_t *labels_x,
                const uint8_t *allowed, int64_t n_allowed, int64_t *labels_y, uint8_t *consider_y,
                int64_t *tests_out) {
    if (!ctx) return CNN_ERR_INVALID;
    return guarded(ctx, [&]() {
        if (n_x < 0 || n_y < 0) throw InvalidArg{"negative size"};
        if (d < 1) throw InvalidArg{"d must be >= 1"};
        if (dtype != CNN_F32 && dtype != CNN_F64) throw InvalidArg{"dtype must be CNN_F32 or CNN_F64"};
        if (n_allowed < 0) throw InvalidArg{"negative n_allowed"};
        if (n_y > 0 && (!Y || !labels_y || !consider_y)) throw InvalidArg{"null buffer for Y"};
        if (n_x > 0 && (!X || !labels_x)) throw InvalidArg{"null buffer for X"};
        if (n_allowed > 0 && !allowed) throw InvalidArg{"null allowed-label table"};
        if (n_x + n_y >= (int64_t)INT32_MAX) throw InvalidArg{"n_x + n_y exceeds the int32 index range"};
        CNN_HIP(hipSetDevice(ctx->device));
        if (tests_out) *tests_out = 0;
        if (n_y == 0 || n_x == 0) return (int)CNN_OK;  // nothing to predict from
        hipStream_t s = ctx->stream;
        const size_t es = dtype == CNN_F32 ? sizeof(float) : sizeof(double);
        const int64_t n = n_x + n_y;
        // [X; Y] in one buffer: one graph holds N_X of both sets' points
        Scratch<uint8_t> Z(ctx, (size_t)n * d * es);
        CNN_HIP(hipMemcpyAsync(Z.p, X, (size_t)n_x * d * es, hipMemcpyDeviceToDevice, s));
        CNN_HIP(hipMemcpyAsync(Z.p + (size_t)n_x * d * es, Y, (size_t)n_y * d * es, hipMemcpyDeviceToDevice, s));
        cnn_graph *g = graph_build(ctx, Z.p, n, d, dtype, r2, precision, nullptr, true);
        std::unique_ptr<cnn_graph, void (*)(cnn_graph *)> hold(g, graph_free);
        const unsigned wblocks = (unsigned)ceil_div(n, 4);
        if (g->mask && g->pair_nz && g->tp_ptr) {
            const int64_t T = g->n_tiles;
            Scratch<uint64_t> ref(ctx, T);
            Scratch<int32_t> rdeg(ctx, n);
            Scratch<uint32_t> key(ctx, n);
            Scratch<unsigned long long> tests(ctx, 1);
            fill_u64(ctx, tests.p, 0ull, 1);
            k_ref_tiles<<<(unsigned)ceil_div(n, 256), 256, 0, s>>>(g->perm, n, n_x, T, ref.p);
            k_ref_keys<<<(unsigned)T, 256, 0, s>>>(g->mask, g->pair_nz, g->tp_ptr, g->tp_col, ref.p, g->perm, n, n_x,
                                                  m_core, labels_x, allowed, n_allowed, rdeg.p, key.p);
            k_predict_words<<<wblocks, 256, 0, s>>>(g->mask, g->pair_nz, g->tp_ptr, g->tp_col, ref.p, rdeg.p, key.p,
                                                    g->perm, n, n_x, c_sim, m_core, labels_x, labels_y, consider_y,
                                                    tests.p);
            CNN_HIP(hipGetLastError());
            const unsigned long long nt = read_scalar(ctx, tests.p);
            if (tests_out) *tests_out = (int64_t)nt;
            return (int)CNN_OK;
        }
        graph_lists(ctx, g);
        Scratch<int32_t> cnt(ctx, n);
        Scratch<int64_t> rp(ctx, n + 1);
        k_keep_ref<false><<<wblocks, 256, 0, s>>>(g->row_ptr, g->col, g->perm, n, n_x, cnt.p, nullptr, nullptr);
        CNN_HIP(hipGetLastError());
        exclusive_scan_i32_to_i64(ctx, cnt.p, rp.p, n);
        const int64_t last_excl = read_scalar(ctx, rp.p + n - 1);
        const int32_t last_cnt = read_scalar(ctx, cnt.p + n - 1);
        const int64_t nnz = last_excl + last_cnt;
        CNN_HIP(hipMemcpyAsync(rp.p + n, &nnz, sizeof(int64_t), hipMemcpyHostToDevice, s));
        Scratch<int32_t> col(ctx, std::max<int64_t>(nnz, 1));
        k_keep_ref<true><<<wblocks, 256, 0, s>>>(g->row_ptr, g->col, g->perm, n, n_x, nullptr, rp.p, col.p);
        CNN_HIP(hipGetLastError());
        Scratch<int64_t> lab(ctx, n);
        Scratch<uint8_t> ok(ctx, n);
        k_ref_members<<<(unsigned)ceil_div(n, 256), 256, 0, s>>>(rp.p, g->perm, n, n_x, m_core, labels_x, allowed,
                                                                 n_allowed, lab.p, ok.p);
        CNN_HIP(hipGetLastError());
        Scratch<unsigned long long> tests(ctx, 1);
        CNN_HIP(hipMemsetAsync(tests.p, 0, sizeof(unsigned long long), s));
        k_predict_rows<<<wblocks, 256, 0, s>>>(rp.p, col.p, g->perm, n, n_x, c_sim, m_core, lab.p, ok.p, labels_y,
                                               consider_y, tests.p);
        CNN_HIP(hipGetLastError());
        unsigned long long nt = 0;
        CNN_HIP(hipMemcpyAsync(&nt, tests.p, sizeof(nt), hipMemcpyDeviceToHost, s));
        CNN_HIP(hipStreamSynchronize(s));
        if (tests_out) *tests_out = (int64_t)nt;
        return (int)CNN_OK;
    });
}

}  // extern "C"
