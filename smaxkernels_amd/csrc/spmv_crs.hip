// CRS SpMV and SpMM for gfx950.
//
// Every output is the reference's sequential row sum
// (spmv_cpu_crs_impl.hpp:20-33, spmm_cpu_crs_impl.hpp:22-44) computed as one
// fma chain in CRS order, so results are bit-identical to the reference CPU
// kernels built with FMA contraction.  Two SpMV schedules:
//
//  * sequential: one lane per row reading straight from HBM (the reference's
//    CUDA schedule, spmv_cuda_crs_impl.cu:5-22);
//  * blocked: a plan cuts the rows into row blocks of at most T rows whose
//    first nonzeros fall in one W-entry window; a long row (kCrsLongRow)
//    forms a block of its own.  Each workgroup of T threads streams its
//    block's values and column indices through LDS in coalesced W-entry tiles
//    (gathering x on the way), and each row's lane then runs its fma chain out
//    of LDS.  Short rows are thereby reduced lane-per-row while the loads stay
//    fully coalesced; a long row is streamed by its whole workgroup.  Row
//    blocks are dealt to the XCDs in contiguous ranges (xcd_block), so the x
//    band of neighbouring blocks is shared in one L2.  Two geometries:
//    T = 256, W = 1024 for rows of even length, and single-wave blocks,
//    T = 64, W = 512, when the longest row exceeds 4x the mean: a wave then
//    waits at its own tiles' barriers only and pipelines its long rows (4M-row
//    band matrix, FP64: 0.657 ms against 0.766; BF16 values 0.443 against
//    0.692; the 512^2 Laplacian and a 27-point stencil run 6.0 / 25.5 us with
//    the wide blocks against 6.5 / 28.2 us).
#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "scan.hpp"
#include "spmm_long.hpp"

namespace smaxhip {
// The first `count` rows of the plan's row order, its longest: the SpMV's first
// `blocks` (a multiple of 8) workgroups take one each.  Their own blocks are
// marked in block_start when the plan is made, so that each row is run once
// whatever row_ptr says by then.
struct FirstRows {
    int32_t count = 0, blocks = 0;
};
}  // namespace smaxhip

struct smax_hip_crs_plan_s {
    int64_t n_rows = 0, nnz = 0, n_blocks = 0;
    int32_t block_threads = 256;     // row-block geometry: 256 (wide) or 64 (narrow)
    int32_t *block_start = nullptr;  // n_blocks + 1 row indices, ~row: a first row's block
    int32_t *row_order = nullptr;    // row-major SpMM execution order (n_rows)
    smaxhip::LongRows long_rows;     // how many rows, first in row_order, are long
    smaxhip::FirstRows first;        // the SpMV's share of them
};

namespace smaxhip {

constexpr int kCrsThreads = 256;
// Rows at least this long form a block of their own, by threads per block:
// with one wavefront they then take long_row_sum (from 128 on: 1,000,000 rows
// 150 us, from 256: 140, from 512: 147), with four a shorter one is done by
// its thread while the other rows' threads run.
template <int NT>
constexpr int kCrsLongRow = NT == kWave ? 256 : 512;
// row-block geometries: threads per block (= rows at most) and the tile and
// block-start window in nonzeros
constexpr int kBlkWideThreads = 256, kBlkWideTile = 1024;
constexpr int kBlkNarrowThreads = 64, kBlkNarrowTile = 512;

// ------------------------------------------------------------ sequential
template <int VT>
__global__ __launch_bounds__(kCrsThreads) void crs_spmv_lane(
    int64_t n_rows, const int32_t *__restrict__ row_ptr,
    const int32_t *__restrict__ col,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ x,
    typename vt<VT>::vec_t *__restrict__ y) {
    using T = vt<VT>;
    const int64_t r = static_cast<int64_t>(blockIdx.x) * kCrsThreads + threadIdx.x;
    if (r >= n_rows) return;
    const int64_t s = row_ptr[r], e = row_ptr[r + 1];
    typename T::vec_t acc = 0;
    int64_t j = s;
    constexpr int U = 4;
    for (; j + U <= e; j += U) {
        int32_t c[U];
        typename T::val_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = col[j + u];
            v[u] = val[j + u];
        }
        typename T::vec_t xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = x[c[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) acc = T::fma_(T::widen(v[u]), xv[u], acc);
    }
    for (; j < e; ++j) acc = T::fma_(T::widen(val[j]), x[col[j]], acc);
    y[r] = acc;
}

// ------------------------------------------------------------ blocked
// One long row by one wavefront: tiles of TILE entries (half the arrays) go
// through LDS as in crs_spmv_blocked, but the next tile's columns, values and
// x entries are requested while this one's chain runs.  What bounds it is that
// chain, one fma after another in the row's order: 6 cycles an entry from
// registers, 11 (FP32) to 15 (FP64) with groups of eight read from LDS, which
// the compiler overlaps better than reads placed a group ahead by hand (13 and
// 23).  Every lane runs the same chain (broadcast reads).  20,000 rows with
// rows of up to 2000, FP64: 91 us with one entry at a time, 19 now.  FP64
// takes two groups at once (one: 23 us); with 4-byte entries the registers are
// worth more (two: BF16, 300,007 rows 44 us against 42).  Tiles of 512: BF16,
// 4,000,000 rows 12% slower.
template <int VT, int TILE>
__device__ __forceinline__ typename vt<VT>::vec_t long_row_sum(
    typename vt<VT>::vec_t *sv, typename vt<VT>::vec_t *sx, int64_t s, int64_t e,
    const int32_t *__restrict__ col, const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ x) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    constexpr int PER = TILE / kWave, U = 8, kAtOnce = sizeof(A) == 8 ? 2 : 1;
    const int tid = static_cast<int>(threadIdx.x);
    int32_t c[PER];
    typename T::val_t v[PER];
    A xv[PER];
    // Past the row's end its last entry is loaded again: under conditions the
    // loads would be waited for where their results merge.
    const auto at = [&](int64_t t0, int u) {
        const int64_t j = t0 + tid + u * kWave;
        return j < e ? j : e - 1;
    };
    const auto load_columns = [&](int64_t t0) {
#pragma unroll
        for (int u = 0; u < PER; ++u) c[u] = ld_stream(col + at(t0, u));
    };
    const auto gather = [&](int64_t t0) {
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            v[u] = ld_stream(val + at(t0, u));
            xv[u] = x[c[u]];
        }
    };
    load_columns(s);
    gather(s);
    load_columns(s + TILE);
    A acc = 0;
    for (int64_t t0 = s; t0 < e; t0 += TILE) {
        // What is past the row's end is -0 * 0, which leaves the accumulator
        // as it is, signed zeros included.
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const bool in = t0 + tid + u * kWave < e;
            sv[tid + u * kWave] = in ? T::widen(v[u]) : A(-0.0);
            sx[tid + u * kWave] = in ? xv[u] : A(0);
        }
        __syncthreads();
        if (t0 + TILE < e) {
            gather(t0 + TILE);
            load_columns(t0 + 2 * TILE);
        }
        const int nt = static_cast<int>(e - t0 < TILE ? e - t0 : TILE);
#pragma unroll kAtOnce
        for (int j = 0; j < nt; j += U) {
            A w[U], b[U];
            load_run<A, U>(sv + j, w);
            load_run<A, U>(sx + j, b);
#pragma unroll
            for (int u = 0; u < U; ++u) acc = T::fma_(w[u], b[u], acc);
        }
        __syncthreads();
    }
    return acc;
}

template <int VT, int NT, int TILE>
__global__ __launch_bounds__(NT) void crs_spmv_blocked(
    const int32_t *__restrict__ block_start,
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ x,
    typename vt<VT>::vec_t *__restrict__ y, FirstRows first, const int32_t *__restrict__ order) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    __shared__ __align__(16) A sv[TILE];
    __shared__ __align__(16) A sx[TILE];
    const int tid = threadIdx.x;
    int64_t r0, r1;
    if (NT == kWave && static_cast<int32_t>(blockIdx.x) < first.blocks) {
        if (static_cast<int32_t>(blockIdx.x) >= first.count) return;
        r0 = order[blockIdx.x];
        r1 = r0 + 1;
    } else {
        const int64_t b = xcd_block(blockIdx.x - first.blocks, gridDim.x - first.blocks);
        const int32_t b0 = block_start[b], b1 = block_start[b + 1];
        if (NT == kWave && b0 < 0) return;  // one of the first workgroups' rows
        r0 = b0;
        r1 = NT == kWave && b1 < 0 ? ~b1 : b1;
    }
    const int64_t s = row_ptr[r0], e = row_ptr[r1];
    if constexpr (NT == kWave) {
        if (r1 - r0 == 1 && e - s >= kCrsLongRow<NT>) {
            const A sum = long_row_sum<VT, TILE / 2>(sv, sx, s, e, col, val, x);
            if (tid == 0) y[r0] = sum;
            return;
        }
    }
    const int64_t row = r0 + tid;
    const bool has = row < r1;
    const int64_t rs = has ? row_ptr[row] : 0, re = has ? row_ptr[row + 1] : 0;
    A acc = 0;
    constexpr int PER = TILE / NT;
    for (int64_t t0 = s; t0 < e; t0 += TILE) {
        const int64_t nt = e - t0 < TILE ? e - t0 : TILE;
        int32_t c[PER];
        typename T::val_t v[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int64_t k = tid + u * NT;
            if (k < nt) {
                c[u] = ld_stream(col + t0 + k);
                v[u] = ld_stream(val + t0 + k);
            }
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int64_t k = tid + u * NT;
            if (k < nt) {
                sx[k] = x[c[u]];
                sv[k] = T::widen(v[u]);
            }
        }
        __syncthreads();
        if (has) {
            const int64_t lo = rs > t0 ? rs : t0;
            const int64_t hi = re < t0 + nt ? re : t0 + nt;
            int j = static_cast<int>(lo - t0);
            const int m = static_cast<int>(hi - t0);
            if constexpr (NT == kWave) {
                // Four entries' LDS reads at once.  A block waits for its
                // longest row, which waited for each entry: 300,007 rows, FP64
                // 51 -> 44 us, BF16 42 -> 36; 1,000,000, FP64 139 -> 126.
                constexpr int U = 4;
                for (; j + U <= m; j += U) {
                    A w[U], b[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        w[u] = sv[j + u];
                        b[u] = sx[j + u];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) acc = T::fma_(w[u], b[u], acc);
                }
            }
            for (; j < m; ++j) acc = T::fma_(sv[j], sx[j], acc);
        }
        __syncthreads();
    }
    if (has) y[row] = acc;
}

// A new block starts at row r when r is a multiple of nt (the block's
// threads), when r's first nonzero enters a new window of `window` entries,
// or when r or r-1 is a long row.
__global__ void crs_block_flags(int64_t n_rows, const int32_t *__restrict__ row_ptr,
                                int32_t *__restrict__ flag, int32_t nt, int32_t window,
                                int32_t long_row) {
    const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= n_rows) return;
    int32_t f = 1;
    if (r % nt != 0) {
        const int32_t a = row_ptr[r - 1], b = row_ptr[r], c = row_ptr[r + 1];
        f = (a / window != b / window) || (b - a >= long_row) || (c - b >= long_row);
    }
    flag[r] = f;
}

// first_from: rows of so many entries, each a block of its own, are first rows.
__global__ void crs_block_starts(int64_t n_rows,
                                 const int32_t *__restrict__ row_ptr, int64_t first_from,
                                 const int32_t *__restrict__ flag,
                                 const int32_t *__restrict__ pos,
                                 int32_t *__restrict__ block_start) {
    const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= n_rows) return;
    const int32_t start = static_cast<int32_t>(r);
    if (flag[r])
        block_start[pos[r] - 1] = row_ptr[r + 1] - row_ptr[r] >= first_from ? ~start : start;
    if (r == n_rows - 1) block_start[pos[r]] = static_cast<int32_t>(n_rows);
}

// ------------------------------------------------------------ SpMM
struct OrderedRow {  // the i-th row of a plan's order
    const int32_t *__restrict__ order, *__restrict__ row_ptr;
    __device__ __forceinline__ LongRowAt operator()(int64_t i) const {
        const int32_t r = order[i];
        return {row_ptr[r + 1] - row_ptr[r], row_ptr[r], r};
    }
};

// Row-major SpMM for any k: ceil(k / Q) lanes per row, each owning a run of Q
// columns (16 bytes' worth where k allows) read with one access per entry,
// `rows` rows a workgroup (none: one row over `parts` workgroups).  LONG: the
// first workgroups take the plan's long rows.
//
// What bounds it: the X rows gathered through L2, and for small matrices the
// longest row's chain.  One column per lane instead (k lanes a row, a 64-bit
// division each, groups of four entries, no prefetch) took 347 us for 200,003
// rows, k = 10, FP64; this way 82.
template <int VT, int Q, bool LONG>
__global__ __launch_bounds__(kCrsThreads) void crs_spmm_run(
    int64_t n_rows, LongRows longs, int64_t k, int64_t lanes, int32_t rows, FastDiv by_lanes,
    int64_t parts, const int32_t *__restrict__ order, const int32_t *__restrict__ row_ptr,
    const int32_t *__restrict__ col, const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ X, int64_t ldx,
    typename vt<VT>::vec_t *__restrict__ Y, int64_t ldy) {
    using A = typename vt<VT>::vec_t;
    if constexpr (LONG) {
        if (blockIdx.x < longs.blocks()) {
            long_rows<VT, Q>(longs, blockIdx.x, OrderedRow{order, row_ptr}, 1, col, val, k, X, ldx,
                             Y, ldy);
            return;
        }
    }
    const int64_t block = blockIdx.x - (LONG ? longs.blocks() : 0);
    int64_t pos, l;
    if (rows > 0) {
        const int32_t rl = by_lanes(static_cast<int32_t>(threadIdx.x));
        if (rl >= rows) return;
        pos = block * rows + rl;
        l = static_cast<int64_t>(threadIdx.x) - rl * lanes;
    } else {
        pos = block / parts;
        l = (block - pos * parts) * kCrsThreads + threadIdx.x;
        if (l >= lanes) return;
    }
    if (LONG) pos += longs.count;
    if (pos >= n_rows) return;
    const int64_t r = order ? static_cast<int64_t>(order[pos]) : pos;
    const int64_t v = run_start<Q>(l, k);
    const int32_t s = row_ptr[r];
    A acc[Q];
    run_chain<VT, Q, !LONG && VT != SMAX_HIP_F64>(s, 1, row_ptr[r + 1] - s, col, val, X + v, ldx, acc);
    store_cols_run<A, Q>(Y + r * ldy + v, acc);
}

template <int VT, int Q>
static void launch_crs_spmm_run(smax_hip_ctx ctx, int64_t n_rows, int64_t k, LongRows longs,
                                const int32_t *order, const int32_t *row_ptr,
                                const int32_t *col, const void *val, const void *X, int64_t ldx,
                                void *Y, int64_t ldy) {
    using T = vt<VT>;
    const int64_t lanes = run_lanes(k, Q);
    const int64_t rows = kCrsThreads / lanes;
    const int64_t parts = rows > 0 ? 1 : ceil_div(lanes, kCrsThreads);
    const int64_t rest = n_rows - longs.count;
    const int64_t blocks = longs.blocks() + (rows > 0 ? ceil_div(rest, rows) : rest * parts);
    auto v = static_cast<const typename T::val_t *>(val);
    auto xv = static_cast<const typename T::vec_t *>(X);
    auto yv = static_cast<typename T::vec_t *>(Y);
    const FastDiv by = fast_div(rows > 0 ? lanes : 1);
#define SMAX_CRS_RUN(L)                                                                      \
    hipLaunchKernelGGL((crs_spmm_run<VT, Q, L>), dim3(static_cast<unsigned>(blocks)),        \
                       dim3(kCrsThreads), 0, ctx->stream, n_rows, longs, k, lanes,           \
                       static_cast<int32_t>(rows), by, parts, order, row_ptr, col, v, xv, ldx, \
                       yv, ldy)
    if (longs.count > 0) SMAX_CRS_RUN(true);
    else SMAX_CRS_RUN(false);
#undef SMAX_CRS_RUN
}

// Row-major SpMM with k = K a power of two and 16-byte aligned X/Y rows: a
// lane owns Q = 16 / sizeof(vec) consecutive columns v (K / Q lanes per row),
// reads its part of each X row with one 16-byte load and keeps Q fma chains;
// the chain is software-pipelined U elements deep.  Every Y[r, v] is the
// same sequential chain over the row as in crs_spmm_run.
template <int VT, int K, bool LONG>
__global__ __launch_bounds__(kCrsThreads) void crs_spmm_rowvec(
    int64_t n_rows, LongRows longs, const int32_t *__restrict__ order,
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ X, int64_t ldx,
    typename vt<VT>::vec_t *__restrict__ Y, int64_t ldy) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    constexpr int Q = 16 / sizeof(A);
    constexpr int GL = K / Q;
    constexpr int U = 8;
    static_assert(GL * Q == K, "K must be a multiple of the run length");
    if constexpr (LONG) {  // the plan's long rows, as in crs_spmm_run
        if (blockIdx.x < longs.blocks()) {
            long_rows<VT, Q>(longs, blockIdx.x, OrderedRow{order, row_ptr}, 1, col, val, K, X, ldx,
                             Y, ldy);
            return;
        }
    }
    const int64_t t = (static_cast<int64_t>(blockIdx.x) - (LONG ? longs.blocks() : 0)) *
                          kCrsThreads + threadIdx.x;
    int64_t r = t / GL + (LONG ? longs.count : 0);
    const int l = static_cast<int>(t % GL);
    if (r >= n_rows) return;
    if (order) r = order[r];
    const int64_t s = row_ptr[r], e = row_ptr[r + 1];
    A acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] = 0;
    int64_t j = s;
    if constexpr ((GL == U || GL == 2 * U) && sizeof(V) <= 4) {
        // 8 or 16 lanes per row (k = 32 or 64 with 4-byte X entries): lane l
        // loads entry l % 8 of each group of 8 and a swizzle within the 8
        // lanes (a DPP row broadcast within the 16) hands every lane all of
        // them, instead of every lane loading each; the next group's are
        // requested before this group's X rows
        if (e - s >= U) {
            const int le = l % U;  // the entry of each group this lane loads
            int cm = col[j + le];
            int wm = val_bits<V>(val[j + le]);
            for (;;) {
                const bool more = j + 2 * U <= e;
                int cn = 0, wn = 0;
                if (more) {
                    cn = col[j + U + le];
                    wn = val_bits<V>(val[j + U + le]);
                }
                int cs[U], ws[U];
                if constexpr (GL == U)
                    grp8_bcast8(cm, wm, cs, ws, std::make_integer_sequence<int, U>{});
                else
                    row16_bcast8(cm, wm, cs, ws, std::make_integer_sequence<int, U>{});
                A xv[U][Q];
#pragma unroll
                for (int u = 0; u < U; ++u)
                    load_run<A, Q>(X + static_cast<int64_t>(cs[u]) * ldx + l * Q, xv[u]);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        acc[q] = T::fma_(T::widen(bits_val<V>(ws[u])), xv[u][q], acc[q]);
                j += U;
                if (!more) break;
                cm = cn;
                wm = wn;
            }
        }
    } else if (e - s >= U) {
        int32_t c0[U];
        V w0[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c0[u] = col[j + u];
            w0[u] = val[j + u];
        }
        for (;;) {
            const bool more = j + 2 * U <= e;
            int32_t c1[U];
            V w1[U];
            if (more) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    c1[u] = col[j + U + u];
                    w1[u] = val[j + U + u];
                }
            }
            A xv[U][Q];
#pragma unroll
            for (int u = 0; u < U; ++u)
                load_run<A, Q>(X + static_cast<int64_t>(c0[u]) * ldx + l * Q, xv[u]);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int q = 0; q < Q; ++q) acc[q] = T::fma_(T::widen(w0[u]), xv[u][q], acc[q]);
            j += U;
            if (!more) break;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                c0[u] = c1[u];
                w0[u] = w1[u];
            }
        }
    }
    for (; j < e; ++j) {
        A xv[Q];
        load_run<A, Q>(X + static_cast<int64_t>(col[j]) * ldx + l * Q, xv);
        const A w = T::widen(val[j]);
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[q] = T::fma_(w, xv[q], acc[q]);
    }
    store_run<A, Q>(Y + r * ldy + l * Q, acc);
}

// Launches crs_spmm_rowvec when k is a power of two in [4Q, 64] and X, Y and
// their row strides are 16-byte aligned; false otherwise.
template <int VT>
static bool launch_crs_spmm_rowvec(smax_hip_ctx ctx, int64_t n_rows, int64_t k,
                                   LongRows longs, const int32_t *order, const int32_t *row_ptr,
                                   const int32_t *col,
                                   const void *val, const void *X, int64_t ldx, void *Y,
                                   int64_t ldy) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    constexpr int64_t Q = 16 / sizeof(A);
    // at least 4 lanes per row (as for the BCRS SpMM, where 2 lost time)
    if (k < 4 * Q || k > 64 || (k & (k - 1)) != 0 || !aligned16(X, Y) ||
        (ldx * sizeof(A)) % 16 != 0 || (ldy * sizeof(A)) % 16 != 0)
        return false;
    const dim3 g(static_cast<unsigned>(
        longs.blocks() + ceil_div((n_rows - longs.count) * (k / Q), kCrsThreads)));
    auto v = static_cast<const typename T::val_t *>(val);
    auto xv = static_cast<const A *>(X);
    auto yv = static_cast<A *>(Y);
#define SMAX_CRS_ROWVEC(KK)                                                                  \
    case KK:                                                                                  \
        if constexpr (KK >= Q) {                                                              \
            if (longs.count > 0)                                                              \
                hipLaunchKernelGGL((crs_spmm_rowvec<VT, KK, true>), g, dim3(kCrsThreads), 0, \
                                   ctx->stream, n_rows, longs, order, row_ptr, col, v, xv,    \
                                   ldx, yv, ldy);                                             \
            else                                                                              \
                hipLaunchKernelGGL((crs_spmm_rowvec<VT, KK, false>), g, dim3(kCrsThreads), 0, \
                                   ctx->stream, n_rows, longs, order, row_ptr, col, v, xv,    \
                                   ldx, yv, ldy);                                             \
        }                                                                                     \
        return true;
    switch (k) {
        SMAX_CRS_ROWVEC(2)
        SMAX_CRS_ROWVEC(4)
        SMAX_CRS_ROWVEC(8)
        SMAX_CRS_ROWVEC(16)
        SMAX_CRS_ROWVEC(32)
        SMAX_CRS_ROWVEC(64)
    default:
        return false;
    }
#undef SMAX_CRS_ROWVEC
}

// Row-major SpMM execution order: every thread group runs one row's chains,
// so a wave lasts as long as its longest row.  Long rows (long_row_from) come
// first, longest first, and run in workgroups of their own; the rest follow window by window (kSpmmWindow rows, so a
// window's X band stays together), longest first inside each window so that
// the rows sharing a wave have similar lengths.  Results do not depend on
// the order.
constexpr int64_t kSpmmWindow = 65536;

static int build_row_order(smax_hip_ctx ctx, int64_t n_rows, int64_t nnz,
                           const std::vector<int32_t> &rp, int32_t **out, LongRows *longs) {
    *out = nullptr;
    *longs = LongRows{};
    const int64_t thr = long_row_from(nnz, n_rows);
    auto len = [&](int32_t r) { return rp[r + 1] - rp[r]; };
    std::vector<int32_t> ord;
    ord.reserve(static_cast<size_t>(n_rows));
    for (int64_t r = 0; r < n_rows; ++r)
        if (len(static_cast<int32_t>(r)) >= thr) ord.push_back(static_cast<int32_t>(r));
    longs->count = static_cast<int64_t>(ord.size());
    longs->whole = std::count_if(ord.begin(), ord.end(),
                                 [&](int32_t r) { return len(r) >= kLongestRow; });
    auto longer = [&](int32_t a, int32_t b) { return len(a) > len(b); };
    std::stable_sort(ord.begin(), ord.end(), longer);
    for (int64_t w = 0; w < n_rows; w += kSpmmWindow) {
        const size_t first = ord.size();
        for (int64_t r = w; r < std::min(n_rows, w + kSpmmWindow); ++r)
            if (len(static_cast<int32_t>(r)) < thr) ord.push_back(static_cast<int32_t>(r));
        std::stable_sort(ord.begin() + static_cast<std::ptrdiff_t>(first), ord.end(), longer);
    }
    int rc = dev_alloc(ctx, reinterpret_cast<void **>(out), sizeof(int32_t) * n_rows,
                       "crs plan row order");
    if (rc) return rc;
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(*out, ord.data(), sizeof(int32_t) * n_rows,
                                      hipMemcpyHostToDevice, ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    return SMAX_HIP_SUCCESS;
}

// Which rows' workgroups come first in the one-wavefront SpMV.  In row order a
// long row may start when the others are nearly done, and its chain then adds
// to their time; in large matrices (`from` is an entry for every 16,000) the
// longest row no longer decides it and the row order's shared x band does:
// 300,007 rows, FP64 61 -> 52 us, 1,000,000 143 -> 137; with an entry for
// every 64,000, 4,000,000 rows took 684 us instead of 666.
static int64_t first_from(int64_t nnz, int64_t n_rows) {
    return std::max({kLongestRow, long_row_from(nnz, n_rows), nnz / 16000});
}

}  // namespace smaxhip

using namespace smaxhip;

namespace smaxhip {

// Dense rows x k block between column-major (element (r, v) at r + v*ld) and
// row-major (r*k + v) layouts, through a 32 x 33 LDS tile so both the read
// and the write are coalesced.  COL_IN: column-major in, row-major out.
template <typename T, bool COL_IN>
__global__ __launch_bounds__(256) void k_relayout(int64_t rows, int64_t k,
                                                  const T *__restrict__ in,
                                                  int64_t ld, T *__restrict__ out) {
    __shared__ T tile[32][33];
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * 32;
    const int64_t v0 = static_cast<int64_t>(blockIdx.y) * 32;
    const int tx = static_cast<int>(threadIdx.x) & 31, ty = static_cast<int>(threadIdx.x) >> 5;
#pragma unroll
    for (int j = 0; j < 32; j += 8) {
        // the read walks the unit-stride index of `in` with tx
        const int64_t r = COL_IN ? r0 + tx : r0 + ty + j;
        const int64_t v = COL_IN ? v0 + ty + j : v0 + tx;
        if (r < rows && v < k) {
            const T e = COL_IN ? in[r + v * ld] : in[r * k + v];
            if (COL_IN) tile[ty + j][tx] = e;   // tile[v - v0][r - r0]
            else tile[tx][ty + j] = e;          // tile[v - v0][r - r0]
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 32; j += 8) {
        // the write walks the unit-stride index of `out` with tx
        const int64_t r = COL_IN ? r0 + ty + j : r0 + tx;
        const int64_t v = COL_IN ? v0 + tx : v0 + ty + j;
        if (r < rows && v < k) {
            if (COL_IN) out[r * k + v] = tile[tx][ty + j];
            else out[r + v * ld] = tile[ty + j][tx];
        }
    }
}

// The same relayout with 16-byte accesses on both sides, for operands whose
// unit-stride extents (rows and k) and leading dimension are multiples of
// E = 16 / sizeof(T) and whose pointers are 16-byte aligned: a 64-row x
// 32-column tile, the column-major side read or written as runs of E rows of
// one column, the row-major side as runs of E columns of one row.  The LDS
// tile is kept as [column][row] with a pitch of 65 elements, so the E-row
// runs of the column-major side and the E-column gathers of the row-major
// side both spread over the banks.
template <typename T, bool COL_IN>
__global__ __launch_bounds__(256) void k_relayout_vec(int64_t rows, int64_t k,
                                                      const T *__restrict__ in,
                                                      int64_t ld, T *__restrict__ out) {
    constexpr int E = 16 / static_cast<int>(sizeof(T));
    constexpr int TR = 64, TV = 32, P = TR + 1;
    constexpr int VPC = TR / E;   // runs per tile column (column-major side)
    constexpr int CPP = 256 / VPC;
    constexpr int VPR = TV / E;   // runs per tile row (row-major side)
    constexpr int RPP = 256 / VPR;
    using V = T __attribute__((ext_vector_type(E)));
    __shared__ T tile[TV * P];   // tile[(v - v0) * P + (r - r0)]
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * TR;
    const int64_t v0 = static_cast<int64_t>(blockIdx.y) * TV;
    const int t = static_cast<int>(threadIdx.x);
    if (COL_IN) {
#pragma unroll
        for (int p = 0; p < TV; p += CPP) {
            const int vc = p + t / VPC, rc = (t % VPC) * E;
            const int64_t r = r0 + rc, v = v0 + vc;
            if (r < rows && v < k) {
                const V e = *reinterpret_cast<const V *>(in + r + v * ld);
#pragma unroll
                for (int i = 0; i < E; ++i) tile[vc * P + rc + i] = e[i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < TR; p += RPP) {
            const int rr = p + t / VPR, vv = (t % VPR) * E;
            const int64_t r = r0 + rr, v = v0 + vv;
            if (r < rows && v < k) {
                V e;
#pragma unroll
                for (int i = 0; i < E; ++i) e[i] = tile[(vv + i) * P + rr];
                *reinterpret_cast<V *>(out + r * k + v) = e;
            }
        }
    } else {
#pragma unroll
        for (int p = 0; p < TR; p += RPP) {
            const int rr = p + t / VPR, vv = (t % VPR) * E;
            const int64_t r = r0 + rr, v = v0 + vv;
            if (r < rows && v < k) {
                const V e = *reinterpret_cast<const V *>(in + r * k + v);
#pragma unroll
                for (int i = 0; i < E; ++i) tile[(vv + i) * P + rr] = e[i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < TV; p += CPP) {
            const int vc = p + t / VPC, rc = (t % VPC) * E;
            const int64_t r = r0 + rc, v = v0 + vc;
            if (r < rows && v < k) {
                V e;
#pragma unroll
                for (int i = 0; i < E; ++i) e[i] = tile[vc * P + rc + i];
                *reinterpret_cast<V *>(out + r + v * ld) = e;
            }
        }
    }
}

// Column-major <-> row-major copy of a rows x k block (COL_IN: column-major
// `in` with leading dimension ld to row-major `out`; else the reverse), with
// 16-byte accesses where the extents and alignment allow.
template <typename T, bool COL_IN>
static void launch_relayout(smax_hip_ctx ctx, int64_t rows, int64_t k, const T *in, int64_t ld,
                            T *out) {
    constexpr int64_t E = 16 / sizeof(T);
    const bool vec = rows % E == 0 && k % E == 0 && ld % E == 0 &&
                     ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    const unsigned gy = static_cast<unsigned>(ceil_div(k, 32));
    if (vec)
        hipLaunchKernelGGL((k_relayout_vec<T, COL_IN>),
                           dim3(static_cast<unsigned>(ceil_div(rows, 64)), gy), dim3(256), 0,
                           ctx->stream, rows, k, in, ld, out);
    else
        hipLaunchKernelGGL((k_relayout<T, COL_IN>),
                           dim3(static_cast<unsigned>(ceil_div(rows, 32)), gy), dim3(256), 0,
                           ctx->stream, rows, k, in, ld, out);
}

}  // namespace smaxhip

namespace smaxhip {

// Fixed staging area of smax_hip_crs_spmm_noalloc (row-major copies of a
// column block of X and of Y): a file-scope device array, so that entry
// point allocates nothing.  Each device holds its own copy for the life of
// the process, shared by every call on that device.  Host code reaches it
// only through the address hipGetSymbolAddress returns for the current
// device; the name itself is a host-side stand-in.
constexpr size_t kNoAllocScratchBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch[kMaxDevices];

// The scratch array's device address on ctx's device (current on entry),
// looked up once per device.
static int noalloc_scratch(smax_hip_ctx ctx, void **out) {
    *out = nullptr;
    if (ctx->device < 0 || ctx->device >= kMaxDevices)
        return fail(ctx, SMAX_HIP_ERROR_NO_DEVICE,
                    "smax_hip_crs_spmm_noalloc: device %d beyond %d", ctx->device, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[ctx->device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return hip_fail(ctx, e != hipSuccess ? e : hipErrorInvalidSymbol,
                            "hipGetSymbolAddress(scratch)");
        g_scratch[ctx->device] = p;
    }
    *out = g_scratch[ctx->device];
    return SMAX_HIP_SUCCESS;
}

}  // namespace smaxhip

extern "C" {

int smax_hip_crs_plan_create(smax_hip_ctx ctx, int64_t n_rows, int64_t nnz,
                             const int32_t *row_ptr, smax_hip_crs_plan *out) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, out, "smax_hip_crs_plan_create: null output");
    *out = nullptr;
    SMAX_HIP_REQUIRE(ctx, n_rows > 0 && n_rows < INT32_MAX && nnz >= 0 &&
                              nnz <= INT32_MAX && row_ptr,
                     "smax_hip_crs_plan_create: bad arguments");
    // the row lengths decide the block geometry and the SpMM row order
    std::vector<int32_t> rp(static_cast<size_t>(n_rows + 1));
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(rp.data(), row_ptr, sizeof(int32_t) * (n_rows + 1),
                                      hipMemcpyDeviceToHost, ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    int64_t longest = 0;
    for (int64_t r = 0; r < n_rows; ++r)
        longest = std::max<int64_t>(longest, static_cast<int64_t>(rp[r + 1]) - rp[r]);
    const bool narrow = static_cast<double>(longest) >
                        4.0 * static_cast<double>(nnz) / static_cast<double>(n_rows);
    const int32_t nt = narrow ? kBlkNarrowThreads : kBlkWideThreads;
    const int32_t window = narrow ? kBlkNarrowTile : kBlkWideTile;
    const int32_t long_row =
        narrow ? kCrsLongRow<kBlkNarrowThreads> : kCrsLongRow<kBlkWideThreads>;
    int64_t from = INT64_MAX;  // first rows: this long and more
    FirstRows first;
    if (narrow) {
        const int64_t line = first_from(nnz, n_rows);
        for (int64_t r = 0; r < n_rows; ++r) first.count += rp[r + 1] - rp[r] >= line;
        if (first.count > 0) {
            from = line;
            first.blocks = (first.count + 7) / 8 * 8;
        }
    }
    int32_t *flag = nullptr, *tmp = nullptr, *starts = nullptr;
    int rc = dev_alloc(ctx, reinterpret_cast<void **>(&flag),
                       sizeof(int32_t) * n_rows, "crs plan");
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&tmp),
                       sizeof(int32_t) * scan_tmp_elems(n_rows), "crs plan");
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&starts),
                       sizeof(int32_t) * (n_rows + 1), "crs plan");
    int64_t n_blocks = 0;
    if (!rc) {
        hipLaunchKernelGGL(crs_block_flags, grid_for(n_rows, 256), dim3(256), 0,
                           ctx->stream, n_rows, row_ptr, flag, nt, window, long_row);
        rc = check_launch(ctx, "crs_block_flags");
    }
    // flag -> inclusive positions (in place); tmp is the scan scratch.
    if (!rc) rc = scan_inclusive<int32_t, false>(ctx, flag, flag, n_rows, tmp);
    int32_t last = 0;
    if (!rc) {
        hipError_t e = hipMemcpyAsync(&last, flag + n_rows - 1, sizeof(int32_t),
                                      hipMemcpyDeviceToHost, ctx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) rc = hip_fail(ctx, e, "crs plan read-back");
        n_blocks = last;
    }
    if (!rc) {
        // Recompute the flags (the scan overwrote them) into tmp-sized reuse.
        int32_t *flag2 = nullptr;
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&flag2),
                       sizeof(int32_t) * n_rows, "crs plan");
        if (!rc) {
            hipLaunchKernelGGL(crs_block_flags, grid_for(n_rows, 256), dim3(256),
                               0, ctx->stream, n_rows, row_ptr, flag2, nt, window, long_row);
            rc = check_launch(ctx, "crs_block_flags");
        }
        if (!rc) {
            hipLaunchKernelGGL(crs_block_starts, grid_for(n_rows, 256), dim3(256),
                               0, ctx->stream, n_rows, row_ptr, from,
                               flag2, flag, starts);
            rc = check_launch(ctx, "crs_block_starts");
        }
        (void)hipStreamSynchronize(ctx->stream);
        dev_free(flag2);
    }
    dev_free(flag);
    dev_free(tmp);
    int32_t *order = nullptr;
    LongRows longs;
    if (!rc) rc = build_row_order(ctx, n_rows, nnz, rp, &order, &longs);
    if (rc) {
        dev_free(starts);
        dev_free(order);
        return rc;
    }
    smax_hip_crs_plan p = new smax_hip_crs_plan_s();
    p->n_rows = n_rows;
    p->nnz = nnz;
    p->n_blocks = n_blocks;
    p->block_threads = nt;
    p->block_start = starts;
    p->row_order = order;
    p->long_rows = longs;
    p->first = first;
    *out = p;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_crs_plan_destroy(smax_hip_ctx ctx, smax_hip_crs_plan plan) {
    if (!plan) return SMAX_HIP_SUCCESS;
    if (ctx) {
        (void)bind(ctx);
        (void)hipStreamSynchronize(ctx->stream);
    }
    dev_free(plan->block_start);
    dev_free(plan->row_order);
    delete plan;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_crs_spmv(smax_hip_ctx ctx, int value_type, int64_t n_rows,
                      int64_t n_cols, int64_t nnz, const int32_t *row_ptr,
                      const int32_t *col, const void *val, const void *x,
                      void *y, smax_hip_crs_plan plan) {
    SMAX_HIP_CHECK_CTX(ctx);
    if (!valid_value_type(value_type))
        return fail(ctx, SMAX_HIP_ERROR_UNSUPPORTED,
                    "smax_hip_crs_spmv: value type %d", value_type);
    SMAX_HIP_REQUIRE(ctx, n_rows > 0 && n_cols > 0 && nnz >= 0 &&
                              nnz <= INT32_MAX,
                     "smax_hip_crs_spmv: bad shape");
    if (n_rows > INT32_MAX || n_cols > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW, "smax_hip_crs_spmv: %lld x %lld exceeds int32",
                    (long long)n_rows, (long long)n_cols);
    SMAX_HIP_REQUIRE(ctx, row_ptr && x && y && (nnz == 0 || (col && val)),
                     "smax_hip_crs_spmv: null pointer");
    if (plan)
        SMAX_HIP_REQUIRE(ctx, plan->n_rows == n_rows && plan->nnz == nnz,
                         "smax_hip_crs_spmv: plan built for another pattern");
    SMAX_HIP_DISPATCH_VT(value_type, {
        using T = vt<VT>;
        auto v = static_cast<const typename T::val_t *>(val);
        auto xv = static_cast<const typename T::vec_t *>(x);
        auto yv = static_cast<typename T::vec_t *>(y);
        if (plan) {
            const dim3 g(static_cast<unsigned>(plan->n_blocks + plan->first.blocks));
            if (plan->block_threads == kBlkNarrowThreads)
                hipLaunchKernelGGL((crs_spmv_blocked<VT, kBlkNarrowThreads, kBlkNarrowTile>), g,
                                   dim3(kBlkNarrowThreads), 0, ctx->stream, plan->block_start,
                                   row_ptr, col, v, xv, yv, plan->first, plan->row_order);
            else
                hipLaunchKernelGGL((crs_spmv_blocked<VT, kBlkWideThreads, kBlkWideTile>), g,
                                   dim3(kBlkWideThreads), 0, ctx->stream, plan->block_start,
                                   row_ptr, col, v, xv, yv, FirstRows{}, nullptr);
            SMAX_HIP_LAUNCHED(ctx, "crs_spmv_blocked");
        } else {
            hipLaunchKernelGGL((crs_spmv_lane<VT>), grid_for(n_rows, kCrsThreads),
                               dim3(kCrsThreads), 0, ctx->stream, n_rows,
                               row_ptr, col, v, xv, yv);
            SMAX_HIP_LAUNCHED(ctx, "crs_spmv_lane");
        }
        return SMAX_HIP_SUCCESS;
    });
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_crs_spmm(smax_hip_ctx ctx, int value_type, int64_t n_rows,
                      int64_t n_cols, int64_t nnz, const int32_t *row_ptr,
                      const int32_t *col, const void *val, int64_t k,
                      int row_major, const void *X, int64_t ldx, void *Y,
                      int64_t ldy, smax_hip_crs_plan plan) {
    SMAX_HIP_CHECK_CTX(ctx);
    if (!valid_value_type(value_type))
        return fail(ctx, SMAX_HIP_ERROR_UNSUPPORTED,
                    "smax_hip_crs_spmm: value type %d", value_type);
    SMAX_HIP_REQUIRE(ctx, n_rows > 0 && n_cols > 0 && nnz >= 0 && k > 0,
                     "smax_hip_crs_spmm: bad shape");
    if (!extent_ok(n_rows, k) || n_cols > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW, "%s: %lld rows x %lld columns exceed the "
                    "launch limits", __func__, (long long)n_rows, (long long)k);
    SMAX_HIP_REQUIRE(ctx, row_ptr && X && Y && (nnz == 0 || (col && val)),
                     "smax_hip_crs_spmm: null pointer");
    if (row_major)
        SMAX_HIP_REQUIRE(ctx, ldx >= k && ldy >= k,
                         "smax_hip_crs_spmm: row-major ld must be >= k");
    else
        SMAX_HIP_REQUIRE(ctx, (ldx >= n_cols || ldx >= n_rows) && (k == 1 || ldy >= n_rows),
                         "smax_hip_crs_spmm: column-major ld too small (need ldx >= "
                         "min(n_rows, n_cols) and ldy >= n_rows)");
    if (plan)
        SMAX_HIP_REQUIRE(ctx, plan->n_rows == n_rows && plan->nnz == nnz,
                         "smax_hip_crs_spmm: plan built for another pattern");
    if (!row_major && k >= 2) {
        // Column-major operands run through row-major copies in the context's
        // workspace: each X row (the k values a nonzero multiplies) becomes
        // contiguous, so the row-major kernels and the plan's row order apply.
        // Every output is the same chain, so Y is unchanged bit for bit.
        SMAX_HIP_DISPATCH_VT(value_type, {
            using A = typename vt<VT>::vec_t;
            const size_t xb = (static_cast<size_t>(n_cols) * k * sizeof(A) + 255) / 256 * 256;
            const size_t yb = static_cast<size_t>(n_rows) * k * sizeof(A);
            void *w = nullptr;
            int rc = ctx_workspace(ctx, xb + yb, &w);
            if (rc) return rc;
            A *Xr = static_cast<A *>(w);
            A *Yr = reinterpret_cast<A *>(static_cast<char *>(w) + xb);
            launch_relayout<A, true>(ctx, n_cols, k, static_cast<const A *>(X), ldx, Xr);
            SMAX_HIP_LAUNCHED(ctx, "k_relayout");
            rc = smax_hip_crs_spmm(ctx, value_type, n_rows, n_cols, nnz, row_ptr, col, val,
                                   k, 1, Xr, k, Yr, k, plan);
            if (rc) return rc;
            launch_relayout<A, false>(ctx, n_rows, k, Yr, ldy, static_cast<A *>(Y));
            SMAX_HIP_LAUNCHED(ctx, "k_relayout");
            return SMAX_HIP_SUCCESS;
        });
        return SMAX_HIP_ERROR_UNSUPPORTED;
    }
    const int32_t *order = plan ? plan->row_order : nullptr;
    const LongRows longs = plan ? plan->long_rows : LongRows{};
    // one column (k = 1): both layouts are the row-major one with unit strides
    if (!row_major) ldx = ldy = 1;
    SMAX_HIP_DISPATCH_VT(value_type, {
        constexpr int64_t Q = 16 / sizeof(typename vt<VT>::vec_t);
        if (!launch_crs_spmm_rowvec<VT>(ctx, n_rows, k, longs, order, row_ptr, col, val, X,
                                        ldx, Y, ldy)) {
            // the widest runs that k columns hold; narrower ones, and so more
            // lanes, where no plan takes the long rows out and the chip is not
            // full (5000 rows, k = 4, FP32 64 -> 56 us, BF16 70 -> 57; 10,000
            // rows, k = 8 (20,000 lanes), 79 both)
            const bool few = longs.count == 0 && n_rows * run_lanes(k, Q) < 16384;
            if (k >= Q && !few)
                launch_crs_spmm_run<VT, Q>(ctx, n_rows, k, longs, order, row_ptr, col, val,
                                           X, ldx, Y, ldy);
            else if (Q > 2 && k >= 2)
                launch_crs_spmm_run<VT, 2>(ctx, n_rows, k, longs, order, row_ptr, col, val,
                                           X, ldx, Y, ldy);
            else
                launch_crs_spmm_run<VT, 1>(ctx, n_rows, k, longs, order, row_ptr, col, val,
                                           X, ldx, Y, ldy);
        }
        SMAX_HIP_LAUNCHED(ctx, "crs_spmm");
        return SMAX_HIP_SUCCESS;
    });
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_crs_spmm_noalloc(smax_hip_ctx ctx, int value_type, int64_t n_rows,
                              int64_t n_cols, int64_t nnz, const int32_t *row_ptr,
                              const int32_t *col, const void *val, int64_t k,
                              int row_major, const void *X, int64_t ldx, void *Y,
                              int64_t ldy, smax_hip_crs_plan plan) {
    SMAX_HIP_CHECK_CTX(ctx);
    // row-major products and k = 1 stage nothing: the same kernels, no scratch
    if (row_major || k == 1)
        return smax_hip_crs_spmm(ctx, value_type, n_rows, n_cols, nnz, row_ptr, col, val, k,
                                 row_major, X, ldx, Y, ldy, plan);
    if (!valid_value_type(value_type))
        return fail(ctx, SMAX_HIP_ERROR_UNSUPPORTED,
                    "smax_hip_crs_spmm_noalloc: value type %d", value_type);
    SMAX_HIP_REQUIRE(ctx, n_rows > 0 && n_cols > 0 && nnz >= 0 && k > 0,
                     "smax_hip_crs_spmm_noalloc: bad shape");
    if (!extent_ok(n_rows, k) || n_cols > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW, "%s: %lld rows x %lld columns exceed the "
                    "launch limits", __func__, (long long)n_rows, (long long)k);
    SMAX_HIP_REQUIRE(ctx, row_ptr && X && Y && (nnz == 0 || (col && val)),
                     "smax_hip_crs_spmm_noalloc: null pointer");
    SMAX_HIP_REQUIRE(ctx, (ldx >= n_cols || ldx >= n_rows) && ldy >= n_rows,
                     "smax_hip_crs_spmm_noalloc: column-major ld too small (need ldx >= "
                     "min(n_rows, n_cols) and ldy >= n_rows)");
    if (plan)
        SMAX_HIP_REQUIRE(ctx, plan->n_rows == n_rows && plan->nnz == nnz,
                         "smax_hip_crs_spmm_noalloc: plan built for another pattern");
    SMAX_HIP_DISPATCH_VT(value_type, {
        using A = typename vt<VT>::vec_t;
        const int64_t s = static_cast<int64_t>(sizeof(A));
        // columns per pass: the X block (rounded up to 256 bytes) and the Y
        // block must fit the scratch together
        const int64_t per_col = (n_cols + n_rows) * s;
        const int64_t kb_max = (static_cast<int64_t>(kNoAllocScratchBytes) - 256) / per_col;
        if (kb_max < 1)
            return fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                        "smax_hip_crs_spmm_noalloc: one column of X and Y takes %lld bytes, "
                        "more than the %zu-byte scratch (n_rows + n_cols <= %lld for this "
                        "type); use smax_hip_crs_spmm",
                        static_cast<long long>(per_col), kNoAllocScratchBytes,
                        static_cast<long long>((static_cast<int64_t>(kNoAllocScratchBytes) - 256) / s));
        int64_t kb = std::min(k, kb_max);
        if (kb < k && kb >= 16) {
            // a power of two in [16, 64] takes the 16-byte-run kernel
            int64_t p = 16;
            while (p * 2 <= std::min<int64_t>(kb, 64)) p *= 2;
            kb = p;
        }
        void *base = nullptr;
        int rc = noalloc_scratch(ctx, &base);
        if (rc) return rc;
        A *Xr = static_cast<A *>(base);
        const int64_t xbytes = (n_cols * kb * s + 255) / 256 * 256;
        A *Yr = reinterpret_cast<A *>(static_cast<char *>(base) + xbytes);
        for (int64_t v0 = 0; v0 < k; v0 += kb) {
            const int64_t kc = std::min(kb, k - v0);
            launch_relayout<A, true>(ctx, n_cols, kc, static_cast<const A *>(X) + v0 * ldx, ldx,
                                     Xr);
            SMAX_HIP_LAUNCHED(ctx, "k_relayout");
            rc = smax_hip_crs_spmm(ctx, value_type, n_rows, n_cols, nnz, row_ptr, col, val,
                                   kc, 1, Xr, kc, Yr, kc, plan);
            if (rc) return rc;
            launch_relayout<A, false>(ctx, n_rows, kc, Yr, ldy, static_cast<A *>(Y) + v0 * ldy);
            SMAX_HIP_LAUNCHED(ctx, "k_relayout");
        }
        return SMAX_HIP_SUCCESS;
    });
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

}  // extern "C"
