// Neighbourhoods from a precomputed distance matrix: MetricExtPrecomputed
// (_types.pyx:2105-2127) under NeighboursGetterExtBruteForce._get
// (_types.pyx:1692-1710): N(i) = { j : D[i, j] <= r }, ascending j, with the
// radius used as given (_adjust_radius returns it unchanged).
//
// The decisions of each row are packed into 64-bit words, one per 64 columns
// (mask[i][c], bit b = column 64c + b); the CSR is emitted from the words.  The
// labelling treats the neighbour relation as symmetric (components of the
// passing edges); for an asymmetric matrix the reference's BFS follows
// directed edges, so pairs whose two decisions differ are counted (a bit
// transpose of each 64x64 block against its mirror block) and reported.
#include <algorithm>
#include <memory>

#include "cnn_internal.hpp"

namespace cnn {

// One wave per row: the words of row i, eight at a time (their loads in flight
// together).  Bound by reading D: 512 MB (n = 8001, FP64) in 105 us, the rate of a
// large copy here; one word at a time 121 us.
template <typename T>
__global__ __launch_bounds__(256) void k_pre_masks(const T *__restrict__ D, int64_t n, int64_t n_words, double r,
                                                   uint64_t *__restrict__ mask, int32_t *__restrict__ deg) {
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    const T *row = D + i * n;
    constexpr int kW = 8;
    int count = 0;
    for (int64_t c = 0; c < n_words; c += kW) {
        T v[kW];
#pragma unroll
        for (int u = 0; u < kW; ++u) {
            const int64_t j = (c + u) * 64 + lane;
            v[u] = row[j < n ? j : n - 1];  // clamped: no load past the row
        }
        uint64_t mine = 0ull;
#pragma unroll
        for (int u = 0; u < kW; ++u) {
            const uint64_t w = __ballot((c + u) * 64 + lane < n && (double)v[u] <= r);
            if (lane == u) mine = w;
            count += __popcll(w);
        }
        if (lane < kW && c + lane < n_words) mask[i * n_words + c + lane] = mine;
    }
    if (lane == 0) deg[i] = count;
}

__global__ void k_pre_total(int64_t *row_ptr, int64_t n, const int32_t *deg) {
    row_ptr[n] = row_ptr[n - 1] + deg[n - 1];
}

// Lane l of a wave: transposed bits of the 64x64 block (row block R, column
// block C) against the block (C, R); counts the pairs {i, j} whose two
// decisions differ.
__global__ __launch_bounds__(256) void k_pre_symmetry(const uint64_t *__restrict__ mask, int64_t n, int64_t n_words,
                                                      unsigned long long *__restrict__ n_asym) {
    const int lane = threadIdx.x & 63;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= n_words * n_words) return;
    const int64_t R = item / n_words, C = item - R * n_words;
    if (C < R) return;
    const int64_t i = R * 64 + lane;   // row of block (R, C)
    const int64_t j = C * 64 + lane;   // row of block (C, R)
    const uint64_t a = i < n ? mask[i * n_words + C] : 0ull;
    const uint64_t b = j < n ? mask[j * n_words + R] : 0ull;
    // lane l of the transpose: bit k = bit l of lane k's word, i.e. D[64R + k, 64C + l] <= r
    const uint64_t at = transpose_bits(a);
    // a diagonal block holds both orders of each pair: count bits k < l only
    const uint64_t keep = R == C ? ((1ull << lane) - 1ull) : ~0ull;
    const int diff = __popcll((at ^ b) & keep);
    const int total = wave_sum(diff);
    if (lane == 0 && total) atomicAdd(n_asym, (unsigned long long)total);
}

// One wave per row: the set bits of its words, in ascending column order.
__global__ __launch_bounds__(256) void k_pre_emit(const uint64_t *__restrict__ mask, int64_t n, int64_t n_words,
                                                  const int64_t *__restrict__ row_ptr, int32_t *__restrict__ col) {
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    int64_t pos = row_ptr[i];
    for (int64_t c = 0; c < n_words; ++c) {
        const uint64_t w = mask[i * n_words + c];
        if ((w >> lane) & 1ull) {
            const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(w >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)w, 0u));
            col[pos + rank] = (int32_t)(c * 64 + lane);
        }
        pos += __popcll(w);
    }
}

}  // namespace cnn

// The words of one thresholded matrix (working memory of the context).
struct cnn_precomputed {
    cnn::Scratch<uint64_t> mask;
    int64_t n, n_words, nnz = 0;
    cnn_precomputed(cnn_ctx *ctx, int64_t n_, int64_t w) : mask(ctx, n_ * w), n(n_), n_words(w) {}
};

using namespace cnn;

// Words, row_ptr, entry count and asymmetric pairs; one host synchronisation.
static void pre_threshold(cnn_ctx *ctx, const void *D, int32_t dtype, double r, int64_t *row_ptr, cnn_precomputed &p,
                          int64_t &asymmetric) {
    hipStream_t s = ctx->stream;
    const int64_t n = p.n, n_words = p.n_words;
    Scratch<int32_t> deg(ctx, n);
    Scratch<unsigned long long> asym(ctx, 1);
    fill_u64(ctx, asym.p, 0ull, 1);
    const unsigned wblocks = (unsigned)ceil_div(n, 4);
    if (dtype == CNN_F32)
        k_pre_masks<float><<<wblocks, 256, 0, s>>>((const float *)D, n, n_words, r, p.mask.p, deg.p);
    else
        k_pre_masks<double><<<wblocks, 256, 0, s>>>((const double *)D, n, n_words, r, p.mask.p, deg.p);
    k_pre_symmetry<<<(unsigned)ceil_div(n_words * n_words, 4), 256, 0, s>>>(p.mask.p, n, n_words, asym.p);
    CNN_HIP(hipGetLastError());
    exclusive_scan_i32_to_i64(ctx, deg.p, row_ptr, n);
    k_pre_total<<<1, 1, 0, s>>>(row_ptr, n, deg.p);
    CNN_HIP(hipGetLastError());
    PinnedReads rd(ctx);
    const int64_t *nnz = rd.get(row_ptr + n);
    const unsigned long long *na = rd.get(asym.p);
    rd.wait();
    p.nnz = *nnz;
    asymmetric = (int64_t)*na;
}

static void pre_emit(cnn_ctx *ctx, const cnn_precomputed &p, const int64_t *row_ptr, int32_t *col, int64_t col_cap) {
    if (p.nnz > col_cap)
        throw Capacity{"col_cap " + std::to_string(col_cap) + " < nnz " + std::to_string(p.nnz)};
    if (p.nnz == 0) return;
    if (!col) throw InvalidArg{"null col"};
    k_pre_emit<<<(unsigned)ceil_div(p.n, 4), 256, 0, ctx->stream>>>(p.mask.p, p.n, p.n_words, row_ptr, col);
    CNN_HIP(hipGetLastError());
}

static void check_pre_args(const void *D, int64_t n, int32_t dtype, const int64_t *row_ptr) {
    if (n < 0) throw InvalidArg{"negative n"};
    if (dtype != CNN_F32 && dtype != CNN_F64) throw InvalidArg{"dtype must be CNN_F32 or CNN_F64"};
    if (!row_ptr) throw InvalidArg{"null row_ptr"};
    if (n > 0 && !D) throw InvalidArg{"null distance matrix"};
    if (n >= (int64_t)INT32_MAX) throw InvalidArg{"n exceeds the int32 index range"};
}

extern "C" {

int cnn_precomputed_create(cnn_ctx *ctx, const void *D, int64_t n, int32_t dtype, double r, int64_t *row_ptr,
                           cnn_precomputed **out, int64_t *nnz_out, int64_t *asymmetric_out) {
    if (!ctx || !out) return CNN_ERR_INVALID;
    *out = nullptr;
    return guarded(ctx, [&]() {
        check_pre_args(D, n, dtype, row_ptr);
        CNN_HIP(hipSetDevice(ctx->device));
        std::unique_ptr<cnn_precomputed> p(new cnn_precomputed(ctx, n, ceil_div(n, 64)));
        int64_t asymmetric = 0;
        if (n == 0) {
            fill_i64(ctx, row_ptr, 0, 1);
            CNN_HIP(hipStreamSynchronize(ctx->stream));
        } else {
            pre_threshold(ctx, D, dtype, r, row_ptr, *p, asymmetric);
        }
        if (nnz_out) *nnz_out = p->nnz;
        if (asymmetric_out) *asymmetric_out = asymmetric;
        *out = p.release();
        return (int)CNN_OK;
    });
}

int cnn_precomputed_emit(cnn_ctx *ctx, const cnn_precomputed *p, const int64_t *row_ptr, int32_t *col,
                         int64_t col_cap) {
    if (!ctx || !p || !row_ptr) return CNN_ERR_INVALID;
    return guarded(ctx, [&]() {
        CNN_HIP(hipSetDevice(ctx->device));
        pre_emit(ctx, *p, row_ptr, col, col_cap);
        // the words go back to the context's working memory with the handle, and the
        // context's next call may run on another stream
        CNN_HIP(hipStreamSynchronize(ctx->stream));
        return (int)CNN_OK;
    });
}

int cnn_precomputed_destroy(cnn_precomputed *p) {
    if (!p) return CNN_ERR_INVALID;
    delete p;
    return CNN_OK;
}

int cnn_precomputed_csr(cnn_ctx *ctx, const void *D, int64_t n, int32_t dtype, double r, int64_t *row_ptr,
                        int32_t *col, int64_t col_cap, int64_t *nnz_out, int64_t *asymmetric_out) {
    if (!ctx) return CNN_ERR_INVALID;
    return guarded(ctx, [&]() {
        check_pre_args(D, n, dtype, row_ptr);
        CNN_HIP(hipSetDevice(ctx->device));
        if (nnz_out) *nnz_out = 0;
        if (asymmetric_out) *asymmetric_out = 0;
        if (n == 0) {
            fill_i64(ctx, row_ptr, 0, 1);
            CNN_HIP(hipStreamSynchronize(ctx->stream));
            return (int)CNN_OK;
        }
        cnn_precomputed p(ctx, n, ceil_div(n, 64));
        int64_t asymmetric = 0;
        pre_threshold(ctx, D, dtype, r, row_ptr, p, asymmetric);
        if (nnz_out) *nnz_out = p.nnz;
        if (asymmetric_out) *asymmetric_out = asymmetric;
        pre_emit(ctx, p, row_ptr, col, col_cap);
        CNN_HIP(hipStreamSynchronize(ctx->stream));
        return (int)CNN_OK;
    });
}

}  // extern "C"
