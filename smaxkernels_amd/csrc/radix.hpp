// Stable LSD radix sort of uint32 keys with their positions as values, on the
// GPU.  Each pass: per-tile digit histograms, one prefix sum over the
// digit-major histogram table, then a scatter whose ranks inside a tile come
// from ballots and prefix sums only, so equal keys keep their input order and
// the result is deterministic.
//
// What bounds it: one read and one write of the pairs a pass, so few passes:
// digits of up to 8 bits (20-bit keys in three passes of 7).  A wavefront ranks
// 64 keys at once (the lanes with the same digit, found by one ballot a bit),
// and a tile's pairs are put in digit order in LDS first, so that each digit's
// run leaves as contiguous stores.  With 4-bit digits and each thread storing
// its own 16 pairs to 16 places, five passes over 8.0 M keys took 0.99 ms; now
// three take 0.19 (43 us a scatter, 12 a histogram).
#pragma once

#include <utility>

#include "common.hpp"
#include "scan.hpp"

namespace smaxhip {
namespace {  // kernels get internal linkage in every including unit

constexpr int kRThreads = 256;
constexpr int kRWaves = kRThreads / kWave;
constexpr int kRItems = 16;
constexpr int kRTile = kRThreads * kRItems;
constexpr int kRMaxBits = 8;
constexpr int kRMaxBuckets = 1 << kRMaxBits;

__global__ __launch_bounds__(kRThreads) void radix_hist(
    int64_t n, int shift, int bits, const uint32_t *__restrict__ keys,
    int32_t *__restrict__ hist, int64_t n_tiles) {
    __shared__ int32_t c[kRMaxBuckets];
    const int tid = static_cast<int>(threadIdx.x);
    const uint32_t mask = (1u << bits) - 1;
    c[tid] = 0;
    __syncthreads();
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kRTile + tid;
#pragma unroll
    for (int k = 0; k < kRItems; ++k) {
        const int64_t i = base + static_cast<int64_t>(k) * kRThreads;
        if (i < n) atomicAdd(&c[(keys[i] >> shift) & mask], 1);
    }
    __syncthreads();
    if (tid < (1 << bits)) hist[tid * n_tiles + blockIdx.x] = c[tid];
}

// incl: inclusive scan of hist (digit-major), so (digit d, tile t) starts at
// incl[d*n_tiles+t] - hist[d*n_tiles+t].  vals null: the positions themselves.
// Wavefront w ranks the tile's items [w*1024, (w+1)*1024), 64 at a time.
__global__ __launch_bounds__(kRThreads) void radix_scatter(
    int64_t n, int shift, int bits, const uint32_t *__restrict__ keys,
    const int32_t *__restrict__ vals, const int32_t *__restrict__ incl,
    const int32_t *__restrict__ hist, int64_t n_tiles,
    uint32_t *__restrict__ okeys, int32_t *__restrict__ ovals) {
    static_assert(kRMaxBuckets == kRThreads, "one thread per digit");
    __shared__ uint32_t count[kRWaves][kRMaxBuckets];
    __shared__ int64_t out_base[kRMaxBuckets];  // first output minus first tile position
    __shared__ uint32_t skey[kRTile];
    __shared__ int32_t sval[kRTile];
    const int tid = static_cast<int>(threadIdx.x);
    const int wave = tid / kWave, lane = tid & (kWave - 1);
    const uint32_t mask = (1u << bits) - 1;
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kRTile;
    const int64_t mine = t0 + wave * (kRItems * kWave) + lane;
    uint32_t kk[kRItems];
    int32_t vv[kRItems], rank[kRItems];
#pragma unroll
    for (int k = 0; k < kRItems; ++k) {
        const int64_t i = mine + k * kWave;
        kk[k] = i < n ? keys[i] : 0;
        vv[k] = i < n ? (vals ? vals[i] : static_cast<int32_t>(i)) : 0;
    }
#pragma unroll
    for (int w = 0; w < kRWaves; ++w) count[w][tid] = 0;
    __syncthreads();
    // rounds of one wavefront follow each other through its own counters
    volatile uint32_t *cnt = count[wave];
#pragma unroll
    for (int k = 0; k < kRItems; ++k) {
        const bool valid = mine + k * kWave < n;
        const uint32_t d = (kk[k] >> shift) & mask;
        unsigned long long same = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
            const unsigned long long ones = __ballot((d >> b) & 1);
            same &= (d >> b) & 1 ? ones : ~ones;
        }
        const uint32_t before = __popcll(same & ((1ull << lane) - 1));
        const uint32_t old = cnt[d];
        rank[k] = static_cast<int32_t>(old + before);
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) cnt[d] = old + __popcll(same);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // thread d: digit d's place in the tile, and each wavefront's part of it
    uint32_t total = 0;
#pragma unroll
    for (int w = 0; w < kRWaves; ++w) total += count[w][tid];
    uint32_t all;
    uint32_t at = block_excl_scan(total, &all);
    if (tid < (1 << bits)) {
        const int64_t h = tid * n_tiles + blockIdx.x;
        out_base[tid] = static_cast<int64_t>(incl[h]) - hist[h] - at;
    }
#pragma unroll
    for (int w = 0; w < kRWaves; ++w) {
        const uint32_t c = count[w][tid];
        count[w][tid] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRItems; ++k)
        if (mine + k * kWave < n) {
            const uint32_t p = count[wave][(kk[k] >> shift) & mask] + rank[k];
            skey[p] = kk[k];
            sval[p] = vv[k];
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRItems; ++k) {
        const int p = k * kRThreads + tid;
        if (p < static_cast<int>(all)) {
            const uint32_t key = skey[p];
            const int64_t o = out_base[(key >> shift) & mask] + p;
            okeys[o] = key;
            ovals[o] = sval[p];
        }
    }
}

// t_row_ptr[c] = first sorted position with key >= c, for c in [0, n_cols].
__global__ void transpose_row_ptr(int64_t n_cols, int64_t nnz,
                                  const uint32_t *__restrict__ keys,
                                  int32_t *__restrict__ t_row_ptr) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c > n_cols) return;
    int64_t a = 0, b = nnz;
    while (a < b) {
        const int64_t m = (a + b) >> 1;
        if (keys[m] < static_cast<uint32_t>(c)) a = m + 1; else b = m;
    }
    t_row_ptr[c] = static_cast<int32_t>(a);
}

// row[j] = the row of CRS position j.  A wavefront takes kRowItems x 64
// consecutive positions: it finds its first row once, and a lane goes on from
// the row it holds (past a run of empty ones by search).
constexpr int kRowItems = 8;

__global__ __launch_bounds__(256) void entry_rows(int64_t nnz, int64_t n_rows,
                                                  const int32_t *__restrict__ row_ptr,
                                                  int32_t *__restrict__ row) {
    const int64_t j0 = (static_cast<int64_t>(blockIdx.x) * 256 + (threadIdx.x & ~(kWave - 1))) *
                       kRowItems;
    if (j0 >= nnz) return;  // whole wavefronts
    int64_t r = wave_row_of(row_ptr, n_rows, j0);
    int32_t end = row_ptr[r + 1];
    for (int u = 0; u < kRowItems; ++u) {
        const int64_t j = j0 + u * kWave + (threadIdx.x & (kWave - 1));
        if (j >= nnz) return;
        for (int step = 0; j >= end && step < 8; ++step) end = row_ptr[++r + 1];
        if (j >= end) {
            r = row_of(row_ptr, r, n_rows, j);
            end = row_ptr[r + 1];
        }
        row[j] = static_cast<int32_t>(r);
    }
}

// t_col[p] = row[src[p]]
__global__ void transpose_cols(int64_t nnz, const int32_t *__restrict__ row,
                               const int32_t *__restrict__ src, int32_t *__restrict__ t_col) {
    const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p < nnz) t_col[p] = row[src[p]];
}

// Owner of the ping-pong buffers; keys()/vals() hold the sorted pairs.
class RadixSort {
    smax_hip_ctx ctx_;
    uint32_t *k_[2] = {nullptr, nullptr};
    int32_t *v_[2] = {nullptr, nullptr};
    int32_t *hist_ = nullptr, *incl_ = nullptr, *tmp_ = nullptr, *row_ = nullptr;
    int cur_ = 0;

  public:
    explicit RadixSort(smax_hip_ctx ctx) : ctx_(ctx) {}
    ~RadixSort() {
        (void)hipStreamSynchronize(ctx_->stream);
        for (int i = 0; i < 2; ++i) {
            dev_free(k_[i]);
            dev_free(v_[i]);
        }
        dev_free(hist_);
        dev_free(incl_);
        dev_free(tmp_);
        dev_free(row_);
    }
    uint32_t *keys() { return k_[cur_]; }
    int32_t *vals() { return v_[cur_]; }

    int reserve(int64_t n) {
        const int64_t table = kRMaxBuckets * ceil_div(n, kRTile);
        int rc = 0;
        const auto get = [&](auto **p, int64_t count) {
            if (!rc) rc = dev_alloc(ctx_, reinterpret_cast<void **>(p), 4 * count, "radix sort");
        };
        for (int i = 0; i < 2; ++i) {
            get(&k_[i], n);
            get(&v_[i], n);
        }
        get(&hist_, table);
        get(&incl_, table);
        get(&tmp_, scan_tmp_elems(table));
        get(&row_, n);
        return rc;
    }

    // Sorts input[0..n) (keys < key_bound): keys() ascending, vals() their
    // positions, ascending among equal keys.
    int sort(const uint32_t *input, int64_t n, int64_t key_bound) {
        if (n <= 0) return SMAX_HIP_SUCCESS;
        const int64_t tiles = ceil_div(n, kRTile);
        int bits = 1;
        while (bits < 32 && (1ll << bits) < key_bound) ++bits;
        const int passes = (bits + kRMaxBits - 1) / kRMaxBits;
        const int digit = (bits + passes - 1) / passes;
        for (int pass = 0; pass < passes; ++pass) {
            const int shift = pass * digit;
            const uint32_t *in = pass == 0 ? input : k_[cur_];
            hipLaunchKernelGGL(radix_hist, dim3(static_cast<unsigned>(tiles)),
                               dim3(kRThreads), 0, ctx_->stream, n, shift, digit, in, hist_,
                               tiles);
            int rc = check_launch(ctx_, "radix_hist");
            if (!rc)
                rc = scan_inclusive<int32_t, false>(ctx_, hist_, incl_,
                                                    (int64_t{1} << digit) * tiles, tmp_);
            if (rc) return rc;
            hipLaunchKernelGGL(radix_scatter, dim3(static_cast<unsigned>(tiles)),
                               dim3(kRThreads), 0, ctx_->stream, n, shift, digit, in,
                               pass == 0 ? nullptr : v_[cur_], incl_, hist_, tiles,
                               k_[1 - cur_], v_[1 - cur_]);
            rc = check_launch(ctx_, "radix_scatter");
            if (rc) return rc;
            cur_ = 1 - cur_;
        }
        return SMAX_HIP_SUCCESS;
    }

    // After a sort of a CRS pattern's columns: the pattern of the transpose,
    // row pointers (n_cols + 1) and columns.
    int transposed_pattern(int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *row_ptr,
                           int32_t *t_row_ptr, int32_t *t_col) {
        hipLaunchKernelGGL(transpose_row_ptr, grid_for(n_cols + 1, 256), dim3(256), 0,
                           ctx_->stream, n_cols, nnz, keys(), t_row_ptr);
        int rc = check_launch(ctx_, "transpose_row_ptr");
        if (rc || nnz == 0) return rc;
        hipLaunchKernelGGL(entry_rows, grid_for(nnz, 256 * kRowItems), dim3(256), 0,
                           ctx_->stream, nnz, n_rows, row_ptr, row_);
        rc = check_launch(ctx_, "entry_rows");
        if (rc) return rc;
        hipLaunchKernelGGL(transpose_cols, grid_for(nnz, 256), dim3(256), 0, ctx_->stream, nnz,
                           row_, vals(), t_col);
        return check_launch(ctx_, "transpose_cols");
    }
};

}  // namespace
}  // namespace smaxhip
