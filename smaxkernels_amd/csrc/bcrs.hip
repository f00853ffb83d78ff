// BCRS SpMV / SpMM and CRS -> BCRS conversion for gfx950.
//
// Block row r, block j (CRS order over blocks), block column jx:
//   y[r*h_pad + ix] = sum_j sum_jx val[j*h_pad*w_pad + off(ix, jx)] *
//                     x[col[j]*w_pad + jx]
// with off = jx*h_pad + ix (column-major blocks) or ix*w_pad + jx
// (row-major), accumulated per output in (j, jx) order exactly as
// naive_bcrs_spmv does (spmv_cpu_bcrs_impl.hpp:45-74): bit-identical.
//
// SpMV, b_w <= 8: a thread per output row reads its row of each block itself
// (bcrs_spmv_rows).  Wider blocks are staged through LDS: the values of
// 256/b_h block rows are contiguous in memory, so the workgroup streams them
// (and the x entries their columns select) with coalesced loads, then lane
// (r, ix) runs its fma chain out of LDS.
#include "common.hpp"
#include "scan.hpp"
#include "spmm_long.hpp"

#include <type_traits>
#include <utility>

struct smax_hip_bcrs_s {
    smax_hip_bcrs_info info;
};

namespace smaxhip {

constexpr int kBThreads = 256;
constexpr int kBTileVals = 2048;  // block values staged per LDS tile

template <int VT>
__global__ __launch_bounds__(kBThreads) void bcrs_spmv_lds(
    int64_t n_block_rows, int b_h, int b_w, int h_pad, int w_pad, int col_major,
    const int32_t *__restrict__ col, const int32_t *__restrict__ row_ptr,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ x,
    typename vt<VT>::vec_t *__restrict__ y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    __shared__ A sv[kBTileVals];
    __shared__ A sx[kBTileVals];
    const int rows_per_wg = kBThreads / b_h;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_wg;
    const int64_t r1 = min<int64_t>(r0 + rows_per_wg, n_block_rows);
    const int tid = threadIdx.x;
    const int64_t my_r = r0 + tid / b_h;
    const int ix = tid % b_h;
    const bool has = tid < rows_per_wg * b_h && my_r < r1;
    const int64_t bs = static_cast<int64_t>(h_pad) * w_pad;
    const int64_t s = row_ptr[r0], e = row_ptr[r1];
    const int64_t js = has ? row_ptr[my_r] : 0, je = has ? row_ptr[my_r + 1] : 0;
    // blocks per tile: values and gathered x entries both fit
    const int64_t tb = min<int64_t>(kBTileVals / bs, kBTileVals / w_pad);
    A acc = 0;
    for (int64_t t0 = s; t0 < e; t0 += tb) {
        const int64_t nb = min<int64_t>(tb, e - t0);
        const int64_t nv = nb * bs;
        const typename T::val_t *vsrc = val + t0 * bs;
        for (int64_t k = tid; k < nv; k += kBThreads) sv[k] = T::widen(ld_stream(vsrc + k));
        const int64_t nx = nb * w_pad;
        for (int64_t k = tid; k < nx; k += kBThreads) {
            const int64_t b = k / w_pad, jx = k - b * w_pad;
            sx[k] = jx < b_w ? x[static_cast<int64_t>(col[t0 + b]) * w_pad + jx] : A(0);
        }
        __syncthreads();
        if (has) {
            const int64_t lo = max(js, t0), hi = min(je, t0 + nb);
            for (int64_t j = lo; j < hi; ++j) {
                const int64_t b = j - t0;
                for (int jx = 0; jx < b_w; ++jx) {
                    const int64_t off = col_major ? jx * h_pad + ix : ix * w_pad + jx;
                    acc = T::fma_(sv[b * bs + off], sx[b * w_pad + jx], acc);
                }
            }
        }
        __syncthreads();
    }
    if (has) y[my_r * h_pad + ix] = acc;
}

// Q values side by side, aligned as a value is.
template <typename V, int Q>
__device__ __forceinline__ void load_vals(const V *__restrict__ p, V (&out)[Q]) {
    if constexpr (sizeof(V) >= 4) {
        load_cols_run<V, Q>(p, out);
    } else {
#pragma unroll
        for (int i = 0; i < Q; ++i) out[i] = p[i];
    }
}

// SpMV, b_w = BW <= 8: thread (r, ix) reads its row of each block itself, G
// blocks at a time (their columns, then all their values and x entries, then
// the fmas): no barrier between loading and the chains, and a block row's
// lanes are neighbours, so a block's lines are read by one wavefront.  RM:
// row-major blocks, the row's BW values side by side.  Bound by the blocks'
// bytes (3x3 FP64, 48^3 block rows: 4.4 TB/s).  7-point block matrices,
// staged in LDS -> so: 3x3 FP64 of 48^3 43.7 -> 12.8 us, 5x5 of 40^3 70 ->
// 16.7, 6x6 89 -> 21.5, 6x6 BF16 of 32^3 38 -> 5.1; a thread per block row
// -> so: 2x2 FP64 of 48^3 10.1 -> 6.2, 4x4 24.4 -> 16.7, 4x4 FP32 of 64^3
// 28.7 -> 20.9, BF16 of 96^3 55.8 -> 46.7.  Half as many
// blocks at a time: 3x3 13.8 us, 6x6 22.5.
template <int VT, int BW, int G, bool RM>
__global__ __launch_bounds__(kBThreads) void bcrs_spmv_rows(
    int64_t n_rows, int b_h, FastDiv by_h, int h_pad, int w_pad,
    const int32_t *__restrict__ col,
    const int32_t *__restrict__ row_ptr, const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ x, typename vt<VT>::vec_t *__restrict__ y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    const int64_t t = xcd_block(blockIdx.x, gridDim.x) * kBThreads + threadIdx.x;
    if (t >= n_rows) return;
    const int32_t r = by_h(static_cast<int32_t>(t));
    const int32_t ix = static_cast<int32_t>(t) - r * b_h;
    const int64_t bs = static_cast<int64_t>(h_pad) * w_pad;
    const V *vrow = val + (RM ? ix * w_pad : ix);
    const int32_t je = row_ptr[r + 1];
    A acc = 0;
    for (int32_t j = row_ptr[r]; j < je; j += G) {
        int32_t c[G];
        V w[G][BW];
        A xv[G][BW];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) c[g] = col[j + g];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
                const V *blk = vrow + (j + g) * bs;
                if constexpr (RM) {
                    load_vals<V, BW>(blk, w[g]);
                } else {
#pragma unroll
                    for (int jx = 0; jx < BW; ++jx) w[g][jx] = blk[jx * h_pad];
                }
                load_cols_run<A, BW>(x + static_cast<int64_t>(c[g]) * w_pad, xv[g]);
            }
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
#pragma unroll
                for (int jx = 0; jx < BW; ++jx) acc = T::fma_(T::widen(w[g][jx]), xv[g][jx], acc);
            }
    }
    y[static_cast<int64_t>(r) * h_pad + ix] = acc;
}

// Thread (r, ix, v), v fastest: the k lanes of one output row share each
// block value (broadcast) and read one contiguous row of X per (j, jx).
// BW > 0 fixes b_w at compile time: a block's b_w values and X entries are
// then loaded together, and the next block's while this one's fmas run, so
// the chain waits about one memory round trip per block.  The fma order is
// the reference's (j, then jx) either way.
template <int VT, int BW>
__global__ __launch_bounds__(kBThreads) void bcrs_spmm_kernel(
    int64_t n_block_rows, int b_h, int b_w_rt, int h_pad, int w_pad, int col_major,
    int64_t k, const int32_t *__restrict__ col,
    const int32_t *__restrict__ row_ptr,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ X,
    typename vt<VT>::vec_t *__restrict__ Y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBThreads + threadIdx.x;
    const int64_t v = t % k, rix = t / k;
    const int64_t r = rix / b_h;
    const int ix = static_cast<int>(rix - r * b_h);
    if (r >= n_block_rows) return;
    const int64_t bs = static_cast<int64_t>(h_pad) * w_pad;
    // value (ix, jx) of a block sits at ix*vs_i + jx*vs_j
    const int64_t vs_i = col_major ? 1 : w_pad, vs_j = col_major ? h_pad : 1;
    const V *vrow = val + ix * vs_i;
    A acc = 0;
    int64_t j = row_ptr[r];
    const int64_t je = row_ptr[r + 1];
    if (BW == 0) {
        for (; j < je; ++j) {
            const V *blk = vrow + j * bs;
            const A *xr = X + static_cast<int64_t>(col[j]) * w_pad * k + v;
            for (int jx = 0; jx < b_w_rt; ++jx)
                acc = T::fma_(T::widen(blk[jx * vs_j]), xr[jx * k], acc);
        }
    } else if (j < je) {
        V w0[BW > 0 ? BW : 1];
        A x0[BW > 0 ? BW : 1];
        {
            const V *blk = vrow + j * bs;
            const A *xr = X + static_cast<int64_t>(col[j]) * w_pad * k + v;
#pragma unroll
            for (int jx = 0; jx < BW; ++jx) {
                w0[jx] = blk[jx * vs_j];
                x0[jx] = xr[jx * k];
            }
        }
        for (; j + 1 < je; ++j) {
            V w1[BW > 0 ? BW : 1];
            A x1[BW > 0 ? BW : 1];
            const V *blk = vrow + (j + 1) * bs;
            const A *xr = X + static_cast<int64_t>(col[j + 1]) * w_pad * k + v;
#pragma unroll
            for (int jx = 0; jx < BW; ++jx) {
                w1[jx] = blk[jx * vs_j];
                x1[jx] = xr[jx * k];
            }
#pragma unroll
            for (int jx = 0; jx < BW; ++jx) acc = T::fma_(T::widen(w0[jx]), x0[jx], acc);
#pragma unroll
            for (int jx = 0; jx < BW; ++jx) {
                w0[jx] = w1[jx];
                x0[jx] = x1[jx];
            }
        }
#pragma unroll
        for (int jx = 0; jx < BW; ++jx) acc = T::fma_(T::widen(w0[jx]), x0[jx], acc);
    }
    Y[(r * h_pad + ix) * k + v] = acc;
}

// SpMM in parts of a block, b_w = BW and b_h a multiple of H, X and Y of any
// alignment and any k >= Q: thread (r, h, l) keeps H outputs of block row r in
// one run of Q columns (the last run is moved back to end at k), G blocks at a
// time.  RM: row-major blocks.  Bound by the blocks' lines, which each of a
// block row's lanes reads through L1.  Against a thread per output (k = 8 /
// 10 / 32): 3x3 FP64 of 48^3 63 / 78 / 225 -> 23 / 29 / 65 us, 5x5 of 40^3 87
// / 110 / 327 -> 28 / 37 / 84, 6x6 121 / 153 / 523 -> 33 / 41 / 144, 6x6 BF16
// of 32^3 44 / 72 / 175 -> 8.4 / 11.6 / 23.  One block at a time: 6x6 FP64 59
// / 60 / 143.
// One argument: a launch costs the host time for each (the four launches of a
// training step of 12^3 3x3 BF16 blocks, k = 4: 18.7 us, 18.1 this way and with
// LineSizes).
struct PartSizes {
    int64_t n_threads, k;
    FastDiv by_lanes, by_parts;
    int lanes, parts, h_pad, w_pad;
};

template <int VT, int H, int BW, int Q, int G, bool RM>
__global__ __launch_bounds__(kBThreads) void bcrs_spmm_part(
    PartSizes a, const int32_t *__restrict__ col, const int32_t *__restrict__ row_ptr,
    const typename vt<VT>::val_t *__restrict__ val, const typename vt<VT>::vec_t *__restrict__ X,
    typename vt<VT>::vec_t *__restrict__ Y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    const int64_t t = xcd_block(blockIdx.x, gridDim.x) * kBThreads + threadIdx.x;
    if (t >= a.n_threads) return;
    const int h_pad = a.h_pad, w_pad = a.w_pad;
    const int64_t k = a.k;
    const int32_t rh = a.by_lanes(static_cast<int32_t>(t));
    const int32_t l = static_cast<int32_t>(t) - rh * a.lanes;
    const int32_t r = a.by_parts(rh);
    const int32_t ix = (rh - r * a.parts) * H;
    const int64_t v = run_start<Q>(l, k);
    const int64_t bs = static_cast<int64_t>(h_pad) * w_pad;
    const V *vpart = val + (RM ? ix * w_pad : ix);
    const A *xpart = X + v;
    A acc[H][Q];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[h][q] = 0;
    const int32_t je = row_ptr[r + 1];
    for (int32_t j = row_ptr[r]; j < je; j += G) {
        int32_t c[G];
        V w[G][RM ? H : BW][RM ? BW : H];
        A xv[G][BW][Q];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) c[g] = col[j + g];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
                const A *xr = xpart + static_cast<int64_t>(c[g]) * w_pad * k;
#pragma unroll
                for (int jx = 0; jx < BW; ++jx) load_cols_run<A, Q>(xr + jx * k, xv[g][jx]);
                const V *blk = vpart + (j + g) * bs;
#pragma unroll
                for (int i = 0; i < (RM ? H : BW); ++i)
                    load_vals<V, RM ? BW : H>(blk + i * (RM ? w_pad : h_pad), w[g][i]);
            }
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
#pragma unroll
                for (int h = 0; h < H; ++h)
#pragma unroll
                    for (int jx = 0; jx < BW; ++jx)
#pragma unroll
                        for (int q = 0; q < Q; ++q)
                            acc[h][q] = T::fma_(T::widen(w[g][RM ? h : jx][RM ? jx : h]),
                                                xv[g][jx][q], acc[h][q]);
            }
    }
#pragma unroll
    for (int h = 0; h < H; ++h)
        store_cols_run<A, Q>(Y + (static_cast<int64_t>(r) * h_pad + ix + h) * k + v, acc[h]);
}

// One block's values, widened to the accumulation type.  DENSE: h_pad == BH
// and w_pad == BW, so the block is BH*BW contiguous values (row- or
// column-major), read as 16-byte loads when that size is a multiple of 16
// bytes (val is then 16-byte aligned, checked by the host); BF16 blocks are
// read as 32-bit words holding two values each.
template <int VT, int BH, int BW, bool DENSE, bool CM>
__device__ __forceinline__ void load_block(const typename vt<VT>::val_t *__restrict__ blk,
                                           int64_t vs_i, int64_t vs_j,
                                           typename vt<VT>::vec_t (&w)[BH][BW]) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    if constexpr (DENSE) {
        A flat[BH * BW];
        if constexpr (VT == SMAX_HIP_BF16 && (BH * BW) % 2 == 0) {
            uint32_t words[BH * BW / 2];
            load_run<uint32_t, BH * BW / 2>(reinterpret_cast<const uint32_t *>(blk), words);
#pragma unroll
            for (int i = 0; i < BH * BW / 2; ++i) {
                flat[2 * i] = __uint_as_float(words[i] << 16);
                flat[2 * i + 1] = __uint_as_float(words[i] & 0xffff0000u);
            }
        } else {
            typename T::val_t raw[BH * BW];
            load_run<typename T::val_t, BH * BW>(blk, raw);
#pragma unroll
            for (int i = 0; i < BH * BW; ++i) flat[i] = T::widen(raw[i]);
        }
#pragma unroll
        for (int ix = 0; ix < BH; ++ix)
#pragma unroll
            for (int jx = 0; jx < BW; ++jx)
                w[ix][jx] = CM ? flat[jx * BH + ix] : flat[ix * BW + jx];
    } else {
#pragma unroll
        for (int jx = 0; jx < BW; ++jx)
#pragma unroll
            for (int ix = 0; ix < BH; ++ix) w[ix][jx] = T::widen(blk[ix * vs_i + jx * vs_j]);
    }
}

// Register-blocked SpMM for compile-time block shapes: thread (r, l) keeps
// the BH outputs of block row r in columns v = l*Q .. l*Q+Q-1, so each X row
// of a block is loaded once for all BH rows (instead of once per row), and
// the BH*Q chains give independent fmas.  Q = 16 bytes' worth (16-byte runs:
// k a multiple of Q, X and Y 16-byte aligned) reads each lane's part of an X
// row with one 16-byte load; Q = 2 with 4-byte entries takes column pairs
// (no alignment needed).  Blocks go in groups of G: the G column indices,
// then all G blocks' values and X entries are requested before any fma, so a
// row of G blocks costs two memory round trips.  Per output the fma order is
// still the reference's (block j, then jx).
template <int VT, int BH, int BW, int Q, bool DENSE, bool CM, int G>
__global__ __launch_bounds__(kBThreads) void bcrs_spmm_reg(
    int64_t n_block_rows, int h_pad, int w_pad, int col_major, int64_t k,
    const int32_t *__restrict__ col, const int32_t *__restrict__ row_ptr,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ X,
    typename vt<VT>::vec_t *__restrict__ Y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    const int64_t gl = k / Q;  // lanes per block row
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBThreads + threadIdx.x;
    const int64_t r = t / gl, v = (t - r * gl) * Q;
    if (r >= n_block_rows) return;
    const int64_t bs = static_cast<int64_t>(h_pad) * w_pad;
    const int64_t vs_i = col_major ? 1 : w_pad, vs_j = col_major ? h_pad : 1;
    A acc[BH][Q];
#pragma unroll
    for (int ix = 0; ix < BH; ++ix)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[ix][q] = 0;
    const int64_t je = row_ptr[r + 1];
    for (int64_t j = row_ptr[r]; j < je; j += G) {
        int32_t c[G];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) c[g] = col[j + g];
        A w[G][BH][BW];
        A xv[G][BW][Q];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
                const A *xr = X + static_cast<int64_t>(c[g]) * w_pad * k + v;
#pragma unroll
                for (int jx = 0; jx < BW; ++jx) load_run<A, Q>(xr + jx * k, xv[g][jx]);
                load_block<VT, BH, BW, DENSE, CM>(val + (j + g) * bs, vs_i, vs_j, w[g]);
            }
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
#pragma unroll
                for (int ix = 0; ix < BH; ++ix)
#pragma unroll
                    for (int jx = 0; jx < BW; ++jx)
#pragma unroll
                        for (int q = 0; q < Q; ++q)
                            acc[ix][q] = T::fma_(w[g][ix][jx], xv[g][jx][q], acc[ix][q]);
            }
    }
#pragma unroll
    for (int ix = 0; ix < BH; ++ix) store_run<A, Q>(Y + (r * h_pad + ix) * k + v, acc[ix]);
}

// Lane N of each 16-lane DPP row, handed to every lane of that row
// (row_newbcast).
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + N, 0xf, 0xf, false));
}

template <int... N>
__device__ __forceinline__ void row_bcast16(float mine, float (&out)[16],
                                            std::integer_sequence<int, N...>) {
    ((out[N] = row_bcast<N>(mine)), ...);
}

// bcrs_spmm_reg for dense 4x4 blocks and k = 64 four-byte columns, where a
// block row's 16 lanes (four columns each) are exactly one DPP row.  There,
// every lane loading the whole 16-value block makes a third of the bytes the
// vector memory path (texture address unit busy ~88 % of the kernel's cycles
// on the 96^3 block matrix) hands back.  Here each lane loads one value of
// the block and 16 row broadcasts give every lane all of them; the next
// group's column indices are requested while this group's X rows are in
// flight.  Per output the fma order is bcrs_spmm_reg's (block j,
// then jx), so Y is bit-identical.
template <int VT, bool CM, int G>
__global__ __launch_bounds__(kBThreads) void bcrs_spmm_bcast(
    int64_t n_block_rows, int64_t k, const int32_t *__restrict__ col,
    const int32_t *__restrict__ row_ptr, const typename vt<VT>::val_t *__restrict__ val,
    const float *__restrict__ X, float *__restrict__ Y) {
    using T = vt<VT>;
    constexpr int BH = 4, BW = 4, Q = 4, kRow = 16;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBThreads + threadIdx.x;
    const int64_t r = t / kRow;  // whole DPP rows leave together
    const int l = static_cast<int>(threadIdx.x) % kRow;
    const int64_t v = static_cast<int64_t>(l) * Q;
    if (r >= n_block_rows) return;
    float acc[BH][Q];
#pragma unroll
    for (int ix = 0; ix < BH; ++ix)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[ix][q] = 0;
    const int64_t jb = row_ptr[r], je = row_ptr[r + 1];
    int32_t cn[G];
#pragma unroll
    for (int g = 0; g < G; ++g) cn[g] = jb + g < je ? col[jb + g] : 0;
    for (int64_t j = jb; j < je; j += G) {
        int32_t c[G];
        float mine[G];
        float xv[G][BW][Q];
#pragma unroll
        for (int g = 0; g < G; ++g) c[g] = cn[g];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
                const float *xr = X + static_cast<int64_t>(c[g]) * BW * k + v;
#pragma unroll
                for (int jx = 0; jx < BW; ++jx) load_run<float, Q>(xr + jx * k, xv[g][jx]);
                mine[g] = T::widen(val[(j + g) * (BH * BW) + l]);
            }
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + G + g < je) cn[g] = col[j + G + g];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
                float w[BH * BW];
                row_bcast16(mine[g], w, std::make_integer_sequence<int, BH * BW>{});
#pragma unroll
                for (int ix = 0; ix < BH; ++ix)
#pragma unroll
                    for (int jx = 0; jx < BW; ++jx)
#pragma unroll
                        for (int q = 0; q < Q; ++q)
                            acc[ix][q] = T::fma_(w[CM ? jx * BH + ix : ix * BW + jx],
                                                 xv[g][jx][q], acc[ix][q]);
            }
    }
#pragma unroll
    for (int ix = 0; ix < BH; ++ix) store_run<float, Q>(Y + (r * BH + ix) * k + v, acc[ix]);
}

// Dword v of lane S of each DPP quad, handed to the quad's four lanes
// (quad_perm [S,S,S,S]).
template <int S>
__device__ __forceinline__ uint32_t quad_bcast(uint32_t v) {
    return static_cast<uint32_t>(
        __builtin_amdgcn_mov_dpp(static_cast<int>(v), S * 0x55, 0xf, 0xf, false));
}

// Dword v of lane S of each aligned group of NL lanes (4: a DPP quad, 8: a
// ds_swizzle group), handed to the group's lanes.
template <int NL, int S>
__device__ __forceinline__ uint32_t group_bcast(uint32_t v) {
    if constexpr (NL == 4)
        return quad_bcast<S>(v);
    else
        return static_cast<uint32_t>(grp8_bcast<S>(static_cast<int>(v)));
}

template <int NL, int M, int... S>
__device__ __forceinline__ void group_bcast_all(const uint32_t (&mine)[M],
                                                uint32_t (&words)[NL * M],
                                                std::integer_sequence<int, S...>) {
#pragma unroll
    for (int d = 0; d < M; ++d) ((words[S * M + d] = group_bcast<NL, S>(mine[d])), ...);
}

// bcrs_spmm_reg for dense 4x4 blocks with four-byte columns and NL = 4 or 8
// lanes per block row (k = 8 in column pairs, Q = 2; k = 16 or 32 in
// 16-byte runs, Q = 4), so that a block row's lanes are one DPP quad or one
// swizzle group of 8: each lane loads 1/NL of the block and broadcasts
// within the group give every lane the whole block, instead of every lane
// loading all of it.  Blocks go in groups of 4 (the quarters take few registers),
// with the next group's column indices requested while this group's X rows
// are in flight.  Per output the fma order is bcrs_spmm_reg's (block j, then
// jx), so Y is bit-identical.
template <int VT, int Q, int NL, bool CM, int G>
__global__ __launch_bounds__(kBThreads) void bcrs_spmm_quad(
    int64_t n_block_rows, int64_t k, const int32_t *__restrict__ col,
    const int32_t *__restrict__ row_ptr, const typename vt<VT>::val_t *__restrict__ val,
    const float *__restrict__ X, float *__restrict__ Y) {
    using T = vt<VT>;
    using V = typename T::val_t;
    constexpr int BH = 4, BW = 4;
    constexpr int kWords = BH * BW * static_cast<int>(sizeof(V)) / 4;  // dwords per block
    constexpr int kMine = kWords / NL;                                 // loaded per lane
    static_assert(kMine * NL == kWords, "a block splits evenly over the group");
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBThreads + threadIdx.x;
    const int64_t r = t / NL;  // whole groups leave together
    const int l = static_cast<int>(threadIdx.x) % NL;
    const int64_t v = static_cast<int64_t>(l) * Q;
    if (r >= n_block_rows) return;
    float acc[BH][Q];
#pragma unroll
    for (int ix = 0; ix < BH; ++ix)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[ix][q] = 0;
    const int64_t jb = row_ptr[r], je = row_ptr[r + 1];
    int32_t cn[G];
#pragma unroll
    for (int g = 0; g < G; ++g) cn[g] = jb + g < je ? col[jb + g] : 0;
    const uint32_t *vw = reinterpret_cast<const uint32_t *>(val);
    for (int64_t j = jb; j < je; j += G) {
        int32_t c[G];
        uint32_t mine[G][kMine];
        float xv[G][BW][Q];
#pragma unroll
        for (int g = 0; g < G; ++g) c[g] = cn[g];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
                const float *xr = X + static_cast<int64_t>(c[g]) * BW * k + v;
#pragma unroll
                for (int jx = 0; jx < BW; ++jx) load_run<float, Q>(xr + jx * k, xv[g][jx]);
                load_run<uint32_t, kMine>(vw + (j + g) * kWords + l * kMine, mine[g]);
            }
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + G + g < je) cn[g] = col[j + G + g];
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (j + g < je) {
                uint32_t words[kWords];
                group_bcast_all<NL>(mine[g], words, std::make_integer_sequence<int, NL>{});
                float w[BH * BW];
#pragma unroll
                for (int i = 0; i < BH * BW; ++i) {
                    if constexpr (sizeof(V) == 2)  // BF16: two values per dword, low first
                        w[i] = __uint_as_float((i & 1) ? (words[i >> 1] & 0xffff0000u)
                                                       : (words[i >> 1] << 16));
                    else
                        w[i] = __uint_as_float(words[i]);
                }
#pragma unroll
                for (int ix = 0; ix < BH; ++ix)
#pragma unroll
                    for (int jx = 0; jx < BW; ++jx)
#pragma unroll
                        for (int q = 0; q < Q; ++q)
                            acc[ix][q] = T::fma_(w[CM ? jx * BH + ix : ix * BW + jx],
                                                 xv[g][jx][q], acc[ix][q]);
            }
    }
#pragma unroll
    for (int ix = 0; ix < BH; ++ix) store_run<float, Q>(Y + (r * BH + ix) * k + v, acc[ix]);
}

template <int VT, int BH, int BW>
static void launch_bcrs_spmm_reg(smax_hip_ctx ctx, int64_t n_block_rows, int64_t h_pad,
                                 int64_t w_pad, bool cm, int64_t k, const int32_t *col,
                                 const int32_t *row_ptr, const void *val, const void *X,
                                 void *Y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    constexpr int Q = 16 / sizeof(A);
    auto v = static_cast<const typename T::val_t *>(val);
    auto xv = static_cast<const A *>(X);
    auto yv = static_cast<A *>(Y);
    // 16-byte runs need at least 4 lanes per block row: with fewer (k = 8 in
    // FP32) the per-lane chains run longer than the saved instructions pay for
    const bool runs = k % Q == 0 && k >= 4 * Q && aligned16(X, Y);
    // unpadded blocks load as one contiguous run (16-byte loads if the block
    // size is a multiple of 16 bytes and val is aligned)
    constexpr bool kBlock16 = (BH * BW * sizeof(typename T::val_t)) % 16 == 0;
    const bool dense = h_pad == BH && w_pad == BW && (!kBlock16 || aligned16(val, val));
    // otherwise, with 4-byte X entries and an even k >= 8, each lane takes two
    // columns: every lane loads its block row's blocks whole, so half as many
    // lanes load half as many copies (96^3 block matrix, k = 8: BF16 values
    // 0.155 -> 0.151 ms, FP32 0.198 -> 0.183 ms)
    const bool pairs = !runs && dense && sizeof(A) == 4 && k % 2 == 0 && k >= 8;
    const int64_t lanes = runs ? k / Q : pairs ? k / 2 : k;  // per block row
    const dim3 g = grid_for(n_block_rows * lanes, kBThreads);
    // 4x4 dense blocks at k = 64 (16 lanes per block row): one value per lane
    // and DPP row broadcasts, in groups of 4 blocks (96^3 block matrix, BF16
    // values: 0.646 -> 0.615 ms forward and through the transpose; groups of
    // 2: 0.621 ms)
    if constexpr (BH == 4 && BW == 4 && sizeof(A) == 4) {
        if (runs && dense && lanes == 16) {
            if (cm)
                hipLaunchKernelGGL((bcrs_spmm_bcast<VT, true, 4>), g, dim3(kBThreads), 0,
                                   ctx->stream, n_block_rows, k, col, row_ptr, v, xv, yv);
            else
                hipLaunchKernelGGL((bcrs_spmm_bcast<VT, false, 4>), g, dim3(kBThreads), 0,
                                   ctx->stream, n_block_rows, k, col, row_ptr, v, xv, yv);
            return;
        }
        // 4 lanes per block row (k = 8 in pairs, k = 16 in runs): a quarter of
        // each block per lane and DPP quad broadcasts, in groups of 4 blocks
        // (k = 8: BF16 values 0.152 -> 0.139 ms forward and through the
        // transpose, FP32 0.183 -> 0.160 ms; groups of 2: 0.150 / 0.171 ms;
        // k = 16, FP32 values: 0.240 -> 0.223 ms).  8 lanes (k = 32 in runs):
        // an eighth per lane and swizzles within the 8 (BF16 values 0.331 ->
        // 0.318 ms, FP32 0.368 -> 0.345 ms)
#define SMAX_BCRS_QUAD(QQ, NN)                                                             \
    if (cm)                                                                                \
        hipLaunchKernelGGL((bcrs_spmm_quad<VT, QQ, NN, true, 4>), g, dim3(kBThreads), 0,   \
                           ctx->stream, n_block_rows, k, col, row_ptr, v, xv, yv);         \
    else                                                                                   \
        hipLaunchKernelGGL((bcrs_spmm_quad<VT, QQ, NN, false, 4>), g, dim3(kBThreads), 0,  \
                           ctx->stream, n_block_rows, k, col, row_ptr, v, xv, yv)
        if (pairs && lanes == 4) {
            SMAX_BCRS_QUAD(2, 4);
            return;
        }
        if (runs && dense && lanes == 4) {
            SMAX_BCRS_QUAD(4, 4);
            return;
        }
        if (runs && dense && lanes == 8) {
            SMAX_BCRS_QUAD(4, 8);
            return;
        }
#undef SMAX_BCRS_QUAD
    }
    // block groups of 2 (measured on the 96^3 block matrix: k = 8 0.173 ->
    // 0.160 ms, k = 64 0.663 -> 0.649 ms in BF16)
#define SMAX_BCRS_REG_LAUNCH(QQ, DD, CC, GG)                                                \
    hipLaunchKernelGGL((bcrs_spmm_reg<VT, BH, BW, QQ, DD, CC, GG>), g, dim3(kBThreads), 0,  \
                       ctx->stream, n_block_rows, static_cast<int>(h_pad),                 \
                       static_cast<int>(w_pad), cm ? 1 : 0, k, col, row_ptr, v, xv, yv)
    // of 8 where one thread has a whole block row of 2x2 BF16 values, the one
    // shape of which spmv_by_rows leaves k = 1 to this kernel
    if constexpr (VT == SMAX_HIP_BF16 && BH == 2 && BW == 2) {
        if (dense && k == 1) {
            if (cm) { SMAX_BCRS_REG_LAUNCH(1, true, true, 8); }
            else { SMAX_BCRS_REG_LAUNCH(1, true, false, 8); }
            return;
        }
    }
    if (runs && dense && cm) { SMAX_BCRS_REG_LAUNCH(Q, true, true, 2); }
    else if (runs && dense) { SMAX_BCRS_REG_LAUNCH(Q, true, false, 2); }
    else if (runs) { SMAX_BCRS_REG_LAUNCH(Q, false, false, 2); }
    else if (pairs && cm) { SMAX_BCRS_REG_LAUNCH(2, true, true, 2); }
    else if (pairs) { SMAX_BCRS_REG_LAUNCH(2, true, false, 2); }
    else if (dense && cm) { SMAX_BCRS_REG_LAUNCH(1, true, true, 2); }
    else if (dense) { SMAX_BCRS_REG_LAUNCH(1, true, false, 2); }
    else { SMAX_BCRS_REG_LAUNCH(1, false, false, 2); }
#undef SMAX_BCRS_REG_LAUNCH
}

template <int VT, int BW>
static void launch_bcrs_spmm(smax_hip_ctx ctx, int64_t threads, int64_t n_block_rows,
                             int64_t b_h, int64_t b_w, int64_t h_pad, int64_t w_pad,
                             bool cm, int64_t k, const int32_t *col,
                             const int32_t *row_ptr, const void *val, const void *X,
                             void *Y) {
    using T = vt<VT>;
    hipLaunchKernelGGL((bcrs_spmm_kernel<VT, BW>), grid_for(threads, kBThreads),
                       dim3(kBThreads), 0, ctx->stream, n_block_rows,
                       static_cast<int>(b_h), static_cast<int>(b_w),
                       static_cast<int>(h_pad), static_cast<int>(w_pad), cm ? 1 : 0, k,
                       col, row_ptr, static_cast<const typename T::val_t *>(val),
                       static_cast<const typename T::vec_t *>(X),
                       static_cast<typename T::vec_t *>(Y));
}


// False: more threads than the kernel's index arithmetic holds.
template <int VT, int H, int BW, int G>
static bool launch_bcrs_spmm_part(smax_hip_ctx ctx, int64_t n_block_rows, int64_t b_h,
                                  int64_t h_pad, int64_t w_pad, bool cm, int64_t k,
                                  const int32_t *col, const int32_t *row_ptr, const void *val,
                                  const void *X, void *Y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    constexpr int Q = 16 / sizeof(A);
    const bool runs = k >= Q;
    const int64_t lanes = runs ? run_lanes(k, Q) : k, parts = b_h / H;
    const int64_t threads = n_block_rows * parts * lanes;
    if (threads > INT32_MAX - kBThreads) return false;
    if constexpr (H > 1) {
        // Fewer threads than fill the chip: one output row each instead of H.
        // us at H and at one, 7-point matrices, k = 4: 5x5 BF16 of 10^3 10.2 and
        // 4.7, 3x3 FP64 of 16^3 5.6 and 3.7; from 2^14 threads on the block
        // values that H rows share count again (5x5 FP64 of 24^3, k = 8, 28,000
        // threads: 9.0 and 12.2).  BF16 values are loaded one by one, which
        // moves the line for the smaller blocks (3x3 of 16^3, k = 16, 16,400
        // threads: 5.8 and 4.0; 6x3 of 16^3, k = 3, 24,600: 5.4 and 4.0), and so
        // do 2x2 blocks with 4-byte X (32^3, k = 4, 32,800: 4.1 and 3.7).
        const bool small = (sizeof(A) == 4 && BW == 2) || (VT == SMAX_HIP_BF16 && BW == 3);
        const int64_t few = !small ? 1 << 14 : BW == 2 || runs || parts == 1 ? 3 << 14 : 1 << 18;
        if (threads < few)
            return launch_bcrs_spmm_part<VT, 1, BW, G>(ctx, n_block_rows, b_h, h_pad, w_pad, cm, k,
                                                       col, row_ptr, val, X, Y);
    }
    const PartSizes sizes{threads,
                          k,
                          fast_div(lanes),
                          fast_div(parts),
                          static_cast<int>(lanes),
                          static_cast<int>(parts),
                          static_cast<int>(h_pad),
                          static_cast<int>(w_pad)};
#define SMAX_BCRS_PART(QQ, RM)                                                               \
    hipLaunchKernelGGL((bcrs_spmm_part<VT, H, BW, QQ, G, RM>), grid_for(threads, kBThreads), \
                       dim3(kBThreads), 0, ctx->stream, sizes, col, row_ptr,                 \
                       static_cast<const typename T::val_t *>(val), static_cast<const A *>(X), \
                       static_cast<A *>(Y))
    if (runs && cm) SMAX_BCRS_PART(Q, false);
    else if (runs) SMAX_BCRS_PART(Q, true);
    else if (cm) SMAX_BCRS_PART(1, false);
    else SMAX_BCRS_PART(1, true);
#undef SMAX_BCRS_PART
    return true;
}

// Which block shapes take it: 3x3, 5x5, 6x6 and stacks of them; 2x2 and, in FP64
// from k = 8 on, 4x4 (FP32 and BF16 values have broadcast kernels), except where
// the register-blocked kernel is faster (us, this against that):
//   2x2, 16-byte runs (k >= 16) once Y is 90 MB (FP64 of 64^3, k = 20, 84 MB 61
//     / 64, of 72^3, k = 16, 96 MB 86 / 81) or, with 4-byte X, 100 MB (FP32 of
//     80^3, k = 24, 98 MB 83 / 91, k = 32, 131 MB 110 / 105)
//   2x2 BF16 values for k < 4 (96^3, k = 3 49 / 40, k = 4 33 / 39) and from k =
//     32 on (96^3 182 / 164)
//   2x2 FP32, k = 3, from 2^13 block rows to a Y of 5 MB (24^3 3.8 / 3.7, 40^3
//     5.8 / 5.3, 56^3, 4.2 MB 12.9 / 12.6, 64^3, 6.3 MB 16.9 / 17.5; its three
//     lanes a block row of one column each save too little)
//   4x4 FP64, even k, once Y is 64 MB (48^3, k = 16, 57 MB 48 / 53, 64^3, k = 8,
//     67 MB 95 / 92; 56^3, k = 13, 73 MB 101 / 138)
static bool spmm_in_parts(smax_hip_ctx ctx, int value_type, int64_t n_block_rows, int64_t b_h,
                          int64_t b_w, int64_t h_pad, int64_t w_pad, bool cm, int64_t k,
                          const int32_t *col, const int32_t *row_ptr, const void *val,
                          const void *X, void *Y) {
#define SMAX_BCRS_PARTS(VT, H, W, G)                                                       \
    return launch_bcrs_spmm_part<VT, H, W, G>(ctx, n_block_rows, b_h, h_pad, w_pad, cm, k, \
                                              col, row_ptr, val, X, Y)
    SMAX_HIP_DISPATCH_VT(value_type, {
        if (b_w == 3 && b_h % 3 == 0) SMAX_BCRS_PARTS(VT, 3, 3, 4);
        if (b_w == 5 && b_h % 5 == 0) SMAX_BCRS_PARTS(VT, 5, 5, 2);
        if (b_w == 6 && b_h % 3 == 0) SMAX_BCRS_PARTS(VT, 3, 6, 2);
        constexpr int64_t kItem = sizeof(typename vt<VT>::vec_t);
        const int64_t y_bytes = n_block_rows * b_h * k * kItem;
        const bool wide = k >= 16 && k * kItem % 16 == 0 &&
                          y_bytes >= (kItem == 8 ? 90'000'000 : 100'000'000);
        const bool three = VT == SMAX_HIP_F32 && k == 3 && n_block_rows >= 1 << 13 &&
                           y_bytes < 5'000'000;
        if (b_w == 2 && b_h == 2 && !wide && !three &&
            !(VT == SMAX_HIP_BF16 && (k < 4 || k >= 32)))
            SMAX_BCRS_PARTS(VT, 2, 2, 4);
        if (VT == SMAX_HIP_F64 && b_w == 4 && b_h == 4 && k >= 8 &&
            (k % 2 != 0 || y_bytes < 64'000'000))
            SMAX_BCRS_PARTS(SMAX_HIP_F64, 4, 4, 2);
    });
#undef SMAX_BCRS_PARTS
    return false;
}

// b_w <= 8, except unpadded 2x2 blocks of BF16 values, whose 8 bytes a thread
// per block row reads at once (48^3: 4.4 us against 5.3, 96^3: 24.1 against
// 24.8).  False also with more rows than the kernel's arithmetic holds.
static bool spmv_by_rows(smax_hip_ctx ctx, int value_type, int64_t n_block_rows, int64_t b_h,
                         int64_t b_w, int64_t h_pad, int64_t w_pad, bool cm, const int32_t *col,
                         const int32_t *row_ptr, const void *val, const void *x, void *y) {
    const int64_t rows = n_block_rows * b_h;
    if (b_w > 8 || rows > INT32_MAX - kBThreads) return false;
    if (value_type == SMAX_HIP_BF16 && h_pad == 2 && w_pad == 2 && b_h == 2 && b_w == 2)
        return false;
#define SMAX_BCRS_ROWS(W, RM)                                                                \
    hipLaunchKernelGGL((bcrs_spmv_rows<VT, W, (W <= 3 ? 8 : 4), RM>), grid_for(rows, kBThreads), \
                       dim3(kBThreads), 0, ctx->stream, rows, static_cast<int>(b_h),         \
                       fast_div(b_h), static_cast<int>(h_pad), static_cast<int>(w_pad), col, \
                       row_ptr, static_cast<const typename T::val_t *>(val),                 \
                       static_cast<const typename T::vec_t *>(x),                            \
                       static_cast<typename T::vec_t *>(y))
#define SMAX_BCRS_ROWS_W(W)                                                    \
    case W:                                                                    \
        if (cm) SMAX_BCRS_ROWS(W, false); else SMAX_BCRS_ROWS(W, true);        \
        break;
    SMAX_HIP_DISPATCH_VT(value_type, {
        using T = vt<VT>;
        switch (b_w) {
            SMAX_BCRS_ROWS_W(1) SMAX_BCRS_ROWS_W(2) SMAX_BCRS_ROWS_W(3) SMAX_BCRS_ROWS_W(4)
            SMAX_BCRS_ROWS_W(5) SMAX_BCRS_ROWS_W(6) SMAX_BCRS_ROWS_W(7) SMAX_BCRS_ROWS_W(8)
        }
        return true;
    });
#undef SMAX_BCRS_ROWS_W
#undef SMAX_BCRS_ROWS
    return false;
}

// ------------------------------------------------------------ conversion
// Sorted unique block columns of each block row: a merge of its b_h rows,
// whose block-column sequences must be non-decreasing (the reference's fill
// loop, convert_formats.hpp:222-234, throws otherwise).
//
// A workgroup takes 256/GS consecutive block rows (GS the power of two >=
// b_h), whose CRS entries are one contiguous range; when the range fits the
// LDS tile it is loaded once, coalesced (columns, and values in the fill
// pass), and the merge reads LDS.  A group of GS lanes takes one block row,
// lane l its CRS row br*b_h + l, read front to back.  Each step the group's
// smallest head block column m is found with an xor-butterfly; every lane
// then steps past its entries in block column m, and m is the block row's
// next block column.  In the fill pass a lane places each value it steps
// past, in row order, so of two entries with the same column the later one
// stays, as in the reference's fill loop.

template <typename V>
struct BcrsBuild {
    int64_t nbr, n_cols;
    int b_h, b_w, h_pad, w_pad, col_major;
    int cap;  // entries the LDS tile holds
    FastDiv div;
    const int32_t *row_ptr, *col;
    const V *val;
    int64_t *cnt;        // count pass: blocks per block row
    int64_t *bad;        // count pass: [0] descending rows, [1] columns out of range
    const int64_t *incl; // fill pass: inclusive scan of cnt
    int32_t *brow_ptr, *bcol;
    V *bval;
};

// Entry j of the CRS arrays, from the LDS tile (which starts at entry
// base) or from memory.
template <bool STAGED, typename T>
struct Entries {
    const T *p;
    int32_t base;
    __device__ T operator[](int32_t j) const { return STAGED ? p[j - base] : p[j]; }
};

template <int GS, bool FILL, bool STAGED, typename V>
__device__ void merge_block_row(const BcrsBuild<V> &a, int64_t br, bool row_valid,
                                Entries<STAGED, int32_t> cs, Entries<STAGED, V> vs) {
    const int lane = static_cast<int>(threadIdx.x) & (GS - 1);
    const bool mine = row_valid && lane < a.b_h;
    int32_t pos = 0, end = 0;
    if (mine) {
        const int64_t r = br * a.b_h + lane;
        pos = a.row_ptr[r];
        end = a.row_ptr[r + 1];
    }
    int desc = 0, range = 0;
    if (!FILL && mine) {
        int32_t prev = -1;
        for (int32_t j = pos; j < end; ++j) {
            const int32_t c = cs[j];
            range |= static_cast<uint32_t>(c) >= static_cast<uint64_t>(a.n_cols);
            const int32_t bc = a.div(c);
            desc |= bc < prev;
            prev = bc;
        }
    }
    if (!FILL) {
#pragma unroll
        for (int off = GS / 2; off >= 1; off >>= 1) {
            desc |= __shfl_xor(desc, off, GS);
            range |= __shfl_xor(range, off, GS);
        }
        if (desc || range) {
            if (row_valid && lane == 0) {
                a.cnt[br] = 0;
                if (desc) atomicAdd(reinterpret_cast<unsigned long long *>(a.bad), 1ull);
                if (range) atomicAdd(reinterpret_cast<unsigned long long *>(a.bad + 1), 1ull);
            }
            return;
        }
    }
    const int64_t start = FILL && row_valid ? (br == 0 ? 0 : a.incl[br - 1]) : 0;
    const int64_t bs = static_cast<int64_t>(a.h_pad) * a.w_pad;
    int64_t u = 0;
    for (;;) {
        int32_t m = pos < end ? a.div(cs[pos]) : INT32_MAX;
#pragma unroll
        for (int off = GS / 2; off >= 1; off >>= 1) m = min(m, __shfl_xor(m, off, GS));
        if (m == INT32_MAX) break;
        const int64_t blk = start + u;
        while (pos < end) {
            const int32_t c = cs[pos];
            if (a.div(c) != m) break;
            if (FILL) {
                const int64_t in = c - static_cast<int64_t>(m) * a.b_w;
                const int64_t inc = a.col_major ? static_cast<int64_t>(a.h_pad) * in + lane
                                                : static_cast<int64_t>(a.w_pad) * lane + in;
                a.bval[blk * bs + inc] = vs[pos];
            }
            ++pos;
        }
        if (FILL && lane == 0) a.bcol[blk] = m;
        ++u;
    }
    if (row_valid && lane == 0) {
        if (FILL) {
            a.brow_ptr[br + 1] = static_cast<int32_t>(a.incl[br]);
            if (br == 0) a.brow_ptr[0] = 0;
        } else {
            a.cnt[br] = u;
        }
    }
}

// Count pass (FILL false): blocks per block row, descending rows and
// out-of-range columns.  Fill pass: block row pointers, block columns and
// values (into zeroed blocks).  Dynamic LDS: cap columns, then (fill pass)
// cap values.
template <int GS, bool FILL, typename V>
__global__ __launch_bounds__(256) void bcrs_build(BcrsBuild<V> a) {
    extern __shared__ int32_t tile_col[];
    V *tile_val = reinterpret_cast<V *>(tile_col + a.cap);
    constexpr int kRows = 256 / GS;
    const int64_t br0 = static_cast<int64_t>(blockIdx.x) * kRows;
    const int64_t br1 = min<int64_t>(br0 + kRows, a.nbr);
    const int64_t br = br0 + static_cast<int>(threadIdx.x) / GS;
    const bool row_valid = br < br1;
    const int32_t base = a.row_ptr[br0 * a.b_h];
    const int32_t len = a.row_ptr[br1 * a.b_h] - base;
    if (len >= 0 && len <= a.cap) {
        for (int32_t t = threadIdx.x; t < len; t += 256) {
            tile_col[t] = a.col[base + t];
            if (FILL) tile_val[t] = a.val[base + t];
        }
        __syncthreads();
        merge_block_row<GS, FILL, true>(a, br, row_valid, Entries<true, int32_t>{tile_col, base},
                                        Entries<true, V>{tile_val, base});
    } else {
        merge_block_row<GS, FILL, false>(a, br, row_valid, Entries<false, int32_t>{a.col, 0},
                                         Entries<false, V>{a.val, 0});
    }
}

// Lanes per block row of the conversion: the power of two >= b_h (<= 64).
inline int bcrs_group(int64_t b_h) {
    int g = 1;
    while (g < b_h) g <<= 1;
    return g;
}

// LDS tile of a pass: room for 1.25x a workgroup's average entries (plus
// slack), at most 64 KB.
inline int bcrs_tile_entries(int64_t nnz, int64_t n_wg, int64_t entry_bytes) {
    const int64_t avg = nnz / (n_wg > 0 ? n_wg : 1);
    const int64_t most = (65536 / entry_bytes) / 256 * 256;
    const int64_t want = (avg + avg / 4 + 256 + 255) / 256 * 256;
    return static_cast<int>(want < most ? want : most);
}

template <bool FILL, typename V>
static int launch_bcrs_build(smax_hip_ctx ctx, BcrsBuild<V> a, int64_t nnz) {
    const int gs = bcrs_group(a.b_h);
    const int64_t n_wg = (a.nbr + 256 / gs - 1) / (256 / gs);
    const int64_t entry = 4 + (FILL ? sizeof(V) : 0);
    a.cap = bcrs_tile_entries(nnz, n_wg, entry);
    const size_t lds = static_cast<size_t>(a.cap) * entry;
    switch (gs) {
#define SMAX_BCRS_BUILD(G)                                                                \
    case G:                                                                               \
        hipLaunchKernelGGL((bcrs_build<G, FILL, V>), dim3(static_cast<unsigned>(n_wg)),   \
                           dim3(256), lds, ctx->stream, a);                               \
        break;
        SMAX_BCRS_BUILD(1)
        SMAX_BCRS_BUILD(2)
        SMAX_BCRS_BUILD(4)
        SMAX_BCRS_BUILD(8)
        SMAX_BCRS_BUILD(16)
        SMAX_BCRS_BUILD(32)
        SMAX_BCRS_BUILD(64)
#undef SMAX_BCRS_BUILD
    }
    return check_launch(ctx, FILL ? "bcrs_build(fill)" : "bcrs_build(count)");
}

static int check_bcrs(smax_hip_ctx ctx, const char *fn, int value_type,
                      int64_t nbr, int64_t b_h, int64_t b_w, int64_t h_pad,
                      int64_t w_pad) {
    if (!valid_value_type(value_type))
        return fail(ctx, SMAX_HIP_ERROR_UNSUPPORTED, "%s: value type %d", fn,
                    value_type);
    SMAX_HIP_REQUIRE(ctx, nbr > 0 && b_h > 0 && b_w > 0 && h_pad >= b_h &&
                              w_pad >= b_w,
                     "%s: bad block shape (%lld rows, %lldx%lld pad %lldx%lld)",
                     fn, (long long)nbr, (long long)b_h, (long long)b_w,
                     (long long)h_pad, (long long)w_pad);
    SMAX_HIP_REQUIRE(ctx, b_h <= kBThreads && h_pad * w_pad <= kBTileVals,
                     "%s: blocks larger than %d values are not supported", fn,
                     kBTileVals);
    if (nbr > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW, "%s: %lld block rows exceed int32", fn,
                    (long long)nbr);
    return SMAX_HIP_SUCCESS;
}

}  // namespace smaxhip

using namespace smaxhip;

extern "C" {

int smax_hip_bcrs_spmv(smax_hip_ctx ctx, int value_type,
                       int64_t n_block_rows, int64_t b_h, int64_t b_w,
                       int64_t h_pad, int64_t w_pad, const int32_t *col,
                       const int32_t *row_ptr, const void *val,
                       int block_col_major, const void *x, void *y) {
    SMAX_HIP_CHECK_CTX(ctx);
    int rc = check_bcrs(ctx, "smax_hip_bcrs_spmv", value_type, n_block_rows,
                        b_h, b_w, h_pad, w_pad);
    if (rc) return rc;
    SMAX_HIP_REQUIRE(ctx, row_ptr && x && y, "smax_hip_bcrs_spmv: null pointer");
    // b_h, b_w in {1, 2, 4}: the SpMM with one right-hand side
    if ((b_h == 1 || b_h == 2 || b_h == 4) && (b_w == 1 || b_w == 2 || b_w == 4))
        return smax_hip_bcrs_spmm(ctx, value_type, n_block_rows, b_h, b_w, h_pad, w_pad, col,
                                  row_ptr, val, block_col_major, 1, x, y);
    if (spmv_by_rows(ctx, value_type, n_block_rows, b_h, b_w, h_pad, w_pad,
                     block_col_major != 0, col, row_ptr, val, x, y)) {
        SMAX_HIP_LAUNCHED(ctx, "bcrs_spmv_rows");
        return SMAX_HIP_SUCCESS;
    }
    const int64_t rows_per_wg = kBThreads / b_h;
    SMAX_HIP_DISPATCH_VT(value_type, {
        using T = vt<VT>;
        hipLaunchKernelGGL((bcrs_spmv_lds<VT>), grid_for(n_block_rows, rows_per_wg),
                           dim3(kBThreads), 0, ctx->stream, n_block_rows,
                           static_cast<int>(b_h), static_cast<int>(b_w),
                           static_cast<int>(h_pad), static_cast<int>(w_pad),
                           block_col_major ? 1 : 0, col, row_ptr,
                           static_cast<const typename T::val_t *>(val),
                           static_cast<const typename T::vec_t *>(x),
                           static_cast<typename T::vec_t *>(y));
        SMAX_HIP_LAUNCHED(ctx, "bcrs_spmv_lds");
        return SMAX_HIP_SUCCESS;
    });
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_bcrs_spmm(smax_hip_ctx ctx, int value_type,
                       int64_t n_block_rows, int64_t b_h, int64_t b_w,
                       int64_t h_pad, int64_t w_pad, const int32_t *col,
                       const int32_t *row_ptr, const void *val,
                       int block_col_major, int64_t k, const void *X, void *Y) {
    SMAX_HIP_CHECK_CTX(ctx);
    int rc = check_bcrs(ctx, "smax_hip_bcrs_spmm", value_type, n_block_rows,
                        b_h, b_w, h_pad, w_pad);
    if (rc) return rc;
    SMAX_HIP_REQUIRE(ctx, k > 0 && row_ptr && X && Y,
                     "smax_hip_bcrs_spmm: bad k or null pointer");
    if (!extent_ok(n_block_rows * h_pad, k))
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "smax_hip_bcrs_spmm: %lld rows x %lld columns exceed the launch limits",
                    (long long)(n_block_rows * h_pad), (long long)k);
    const int64_t threads = n_block_rows * b_h * k;
    const bool cm = block_col_major != 0;
    if (k == 1 && spmv_by_rows(ctx, value_type, n_block_rows, b_h, b_w, h_pad, w_pad, cm, col,
                               row_ptr, val, X, Y)) {
        SMAX_HIP_LAUNCHED(ctx, "bcrs_spmv_rows");
        return SMAX_HIP_SUCCESS;
    }
    if (spmm_in_parts(ctx, value_type, n_block_rows, b_h, b_w, h_pad, w_pad, cm, k, col, row_ptr,
                      val, X, Y)) {
        SMAX_HIP_LAUNCHED(ctx, "bcrs_spmm_part");
        return SMAX_HIP_SUCCESS;
    }
    // What the two kernels above leave of (b_h, b_w) in {1, 2, 4} x {1, 2, 4}
    // runs in registers: for one right-hand side 2x2 BF16 blocks, for more the
    // shapes that spmm_in_parts does not take (it takes square ones, up to the
    // sizes of Y named there).
    const bool reg = (b_h == 1 || b_h == 2 || b_h == 4) && (b_w == 1 || b_w == 2 || b_w == 4);
#define SMAX_BCRS_REG(H, W)                                                            \
    if (b_h == H && b_w == W) {                                                        \
        launch_bcrs_spmm_reg<VT, H, W>(ctx, n_block_rows, h_pad, w_pad, cm, k, col,    \
                                       row_ptr, val, X, Y);                            \
        SMAX_HIP_LAUNCHED(ctx, "bcrs_spmm_reg");                                       \
        return SMAX_HIP_SUCCESS;                                                       \
    }
    if (reg) {
        SMAX_HIP_DISPATCH_VT(value_type, {
            SMAX_BCRS_REG(1, 1) SMAX_BCRS_REG(1, 2) SMAX_BCRS_REG(1, 4)
            SMAX_BCRS_REG(2, 1) SMAX_BCRS_REG(2, 2) SMAX_BCRS_REG(2, 4)
            SMAX_BCRS_REG(4, 1) SMAX_BCRS_REG(4, 2) SMAX_BCRS_REG(4, 4)
        });
    }
#undef SMAX_BCRS_REG
    SMAX_HIP_DISPATCH_VT(value_type, {
        switch (b_w) {
        case 1:
            launch_bcrs_spmm<VT, 1>(ctx, threads, n_block_rows, b_h, b_w, h_pad, w_pad,
                                    cm, k, col, row_ptr, val, X, Y);
            break;
        case 2:
            launch_bcrs_spmm<VT, 2>(ctx, threads, n_block_rows, b_h, b_w, h_pad, w_pad,
                                    cm, k, col, row_ptr, val, X, Y);
            break;
        case 4:
            launch_bcrs_spmm<VT, 4>(ctx, threads, n_block_rows, b_h, b_w, h_pad, w_pad,
                                    cm, k, col, row_ptr, val, X, Y);
            break;
        case 8:
            launch_bcrs_spmm<VT, 8>(ctx, threads, n_block_rows, b_h, b_w, h_pad, w_pad,
                                    cm, k, col, row_ptr, val, X, Y);
            break;
        default:
            launch_bcrs_spmm<VT, 0>(ctx, threads, n_block_rows, b_h, b_w, h_pad, w_pad,
                                    cm, k, col, row_ptr, val, X, Y);
            break;
        }
        SMAX_HIP_LAUNCHED(ctx, "bcrs_spmm_kernel");
        return SMAX_HIP_SUCCESS;
    });
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_bcrs_from_crs(smax_hip_ctx ctx, int64_t n_rows, int64_t n_cols,
                           int64_t nnz, const int32_t *row_ptr,
                           const int32_t *col, const void *val,
                           int64_t val_bytes, int64_t b_h, int64_t b_w,
                           int64_t h_pad, int64_t w_pad, int block_col_major,
                           smax_hip_bcrs *out) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, out, "smax_hip_bcrs_from_crs: null output");
    *out = nullptr;
    SMAX_HIP_REQUIRE(ctx, n_rows > 0 && n_cols > 0 && nnz >= 0 && row_ptr &&
                              (nnz == 0 || (col && val)),
                     "smax_hip_bcrs_from_crs: bad input");
    if (n_rows > INT32_MAX || n_cols > INT32_MAX || nnz > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "smax_hip_bcrs_from_crs: %lld x %lld with %lld entries exceeds int32",
                    (long long)n_rows, (long long)n_cols, (long long)nnz);
    SMAX_HIP_REQUIRE(ctx, val_bytes == 2 || val_bytes == 4 || val_bytes == 8,
                     "smax_hip_bcrs_from_crs: val_bytes must be 2, 4 or 8");
    // convert_formats.hpp:142-157
    SMAX_HIP_REQUIRE(ctx, b_h > 0 && b_w > 0 && n_rows % b_h == 0,
                     "Target block height does not divide number of input rows");
    SMAX_HIP_REQUIRE(ctx, n_cols % b_w == 0,
                     "Target block width does not divide number of input columns");
    SMAX_HIP_REQUIRE(ctx, h_pad >= b_h,
                     "Height padding has to be at least target block height");
    SMAX_HIP_REQUIRE(ctx, w_pad >= b_w,
                     "Width padding has to be at least target block width");
    SMAX_HIP_REQUIRE(ctx, b_h <= 64, "smax_hip_bcrs_from_crs: b_h > 64");
    const int64_t nbr = n_rows / b_h;
    int64_t *cnt = nullptr, *incl = nullptr, *tmp = nullptr, *bad = nullptr;
    smax_hip_bcrs_info info{};
    int rc = dev_alloc(ctx, reinterpret_cast<void **>(&cnt), 8 * nbr, "bcrs");
    if (!rc) rc = dev_alloc(ctx, reinterpret_cast<void **>(&incl), 8 * nbr, "bcrs");
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&tmp),
                       8 * scan_tmp_elems(nbr), "bcrs");
    if (!rc) rc = dev_alloc(ctx, reinterpret_cast<void **>(&bad), 16, "bcrs");
    if (!rc) rc = smax_hip_zero(ctx, bad, 16);
    BcrsBuild<uint32_t> args{};
    args.nbr = nbr;
    args.n_cols = n_cols;
    args.b_h = static_cast<int>(b_h);
    args.b_w = static_cast<int>(b_w);
    args.h_pad = static_cast<int>(h_pad);
    args.w_pad = static_cast<int>(w_pad);
    args.col_major = block_col_major ? 1 : 0;
    args.div = fast_div(b_w);
    args.row_ptr = row_ptr;
    args.col = col;
    args.cnt = cnt;
    args.bad = bad;
    int64_t n_blocks = 0, nbad[2] = {0, 0};
    if (!rc) rc = launch_bcrs_build<false>(ctx, args, nnz);
    if (!rc) rc = scan_inclusive<int64_t, false>(ctx, cnt, incl, nbr, tmp);
    if (!rc) rc = read_i64(ctx, bad, &nbad[0]);
    if (!rc) rc = read_i64(ctx, bad + 1, &nbad[1]);
    if (!rc) rc = read_i64(ctx, incl + nbr - 1, &n_blocks);
    if (!rc && nbad[1])
        rc = fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                  "smax_hip_bcrs_from_crs: %lld block rows hold column indices outside "
                  "[0, %lld)", (long long)nbad[1], (long long)n_cols);
    if (!rc && nbad[0])
        rc = fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                  "Blocked Column array does not fit with crs columns "
                  "(%lld block rows with descending columns)", (long long)nbad[0]);
    if (!rc && n_blocks * h_pad * w_pad > INT32_MAX * 4LL)
        rc = fail(ctx, SMAX_HIP_ERROR_OVERFLOW, "bcrs: too many blocks");
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&info.row_ptr),
                       4 * (nbr + 1), "bcrs row_ptr");
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&info.col), 4 * n_blocks,
                       "bcrs col");
    if (!rc)
        rc = dev_alloc(ctx, &info.val, val_bytes * n_blocks * h_pad * w_pad,
                       "bcrs val");
    if (!rc) rc = smax_hip_zero(ctx, info.val, val_bytes * n_blocks * h_pad * w_pad);
    if (!rc) {
        auto fill = [&](auto *vals) {
            using V = std::remove_const_t<std::remove_pointer_t<decltype(vals)>>;
            BcrsBuild<V> f{};
            f.nbr = args.nbr;
            f.n_cols = args.n_cols;
            f.b_h = args.b_h;
            f.b_w = args.b_w;
            f.h_pad = args.h_pad;
            f.w_pad = args.w_pad;
            f.col_major = args.col_major;
            f.div = args.div;
            f.row_ptr = row_ptr;
            f.col = col;
            f.val = vals;
            f.incl = incl;
            f.brow_ptr = info.row_ptr;
            f.bcol = info.col;
            f.bval = static_cast<V *>(info.val);
            return launch_bcrs_build<true>(ctx, f, nnz);
        };
        if (val_bytes == 8)
            rc = fill(static_cast<const uint64_t *>(val));
        else if (val_bytes == 4)
            rc = fill(static_cast<const uint32_t *>(val));
        else
            rc = fill(static_cast<const uint16_t *>(val));
    }
    (void)hipStreamSynchronize(ctx->stream);
    dev_free(cnt);
    dev_free(incl);
    dev_free(tmp);
    dev_free(bad);
    if (rc) {
        dev_free(info.row_ptr);
        dev_free(info.col);
        dev_free(info.val);
        return rc;
    }
    info.n_block_rows = nbr;
    info.n_block_cols = n_cols / b_w;
    info.n_blocks = n_blocks;
    info.b_h = b_h;
    info.b_w = b_w;
    info.h_pad = h_pad;
    info.w_pad = w_pad;
    info.val_bytes = val_bytes;
    info.block_col_major = block_col_major ? 1 : 0;
    smax_hip_bcrs m = new smax_hip_bcrs_s();
    m->info = info;
    *out = m;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_bcrs_get_info(smax_hip_bcrs bcrs, smax_hip_bcrs_info *info) {
    if (!bcrs || !info)
        return fail(nullptr, SMAX_HIP_ERROR_INVALID_VALUE,
                    "smax_hip_bcrs_get_info: null argument");
    *info = bcrs->info;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_bcrs_destroy(smax_hip_ctx ctx, smax_hip_bcrs bcrs) {
    if (!bcrs) return SMAX_HIP_SUCCESS;
    if (ctx) {
        (void)bind(ctx);
        (void)hipStreamSynchronize(ctx->stream);
    }
    dev_free(bcrs->info.row_ptr);
    dev_free(bcrs->info.col);
    dev_free(bcrs->info.val);
    dev_free(bcrs->info.src_block);
    delete bcrs;
    return SMAX_HIP_SUCCESS;
}

}  // extern "C"

// ------------------------------------------------------------ adjoint
#include "radix.hpp"

namespace smaxhip {

// Block p of `out` = block src_block[p] of `src`, a block being `per` units of
// type U.  A thread moves UNITS units, 256 apart; one unit's index is below
// 2^31, with more the block of each is counted from its workgroup's first.
// Past the end the last unit is loaded again: the loads are requested
// together, not one after another.
//
// What bounds it: one read and one write of the blocks (96^3 matrix of 4x4
// BF16 blocks, 417 MB: 97 us, 75 at the copy rate), in units of 16 bytes where
// the block size and alignment allow; in small matrices two dependent loads
// (10^3: 2.3 us).  Value by value with a 64-bit division each: 278 and 2.3 us.
// Four units a thread pay below 16 bytes once there are enough of them: 5x5
// FP32 of 32^3 (5.6 M units) 15.0 -> 12.5 us, 3x3 FP64 (2.0 M) 9.0 -> 8.3,
// 3x3 BF16 of 16^3 (0.2 M) 2.4 -> 2.6; with 16-byte units they change nothing.
// (Quad is a built-in vector: an array of HIP's uint4 is kept in LDS, which
// made 24^3 of 2x2 FP64 blocks 14.9 us, 2.8 now.)
typedef uint32_t Quad __attribute__((ext_vector_type(4)));
constexpr int kGatherUnits = 4;
constexpr int64_t kGatherWide = 1 << 20;

template <typename U, int UNITS>
__global__ __launch_bounds__(256) void bcrs_gather_blocks(
    int64_t total, int32_t per, FastDiv by_per, const int32_t *__restrict__ src_block,
    const U *__restrict__ src, U *__restrict__ out) {
    const int64_t base = static_cast<int64_t>(blockIdx.x) * (256 * UNITS);
    const int64_t p0 = UNITS == 1 ? 0 : base / per;
    const int32_t first = static_cast<int32_t>(base - p0 * per);
    const int32_t left = static_cast<int32_t>(total - base < 256 * UNITS ? total - base : 256 * UNITS);
    int32_t at[UNITS], blk[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int32_t q = u * 256 + static_cast<int32_t>(threadIdx.x);
        const int32_t i = first + (q < left ? q : left - 1), p = by_per(i);
        at[u] = i - p * per;
        blk[u] = src_block[p0 + p];
    }
    U v[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) v[u] = src[static_cast<int64_t>(blk[u]) * per + at[u]];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int32_t q = u * 256 + static_cast<int32_t>(threadIdx.x);
        if (q < left) out[base + q] = v[u];
    }
}

template <typename U>
static void launch_gather_blocks(smax_hip_ctx ctx, int64_t n_blocks, int64_t block_bytes,
                                 const int32_t *src_block, const void *src, void *out) {
    const int64_t per = block_bytes / static_cast<int64_t>(sizeof(U)), total = n_blocks * per;
    const bool one = total < (sizeof(U) == 16 ? INT32_MAX : kGatherWide);
    const auto launch = [&](auto kernel, int units) {
        hipLaunchKernelGGL(kernel, grid_for(total, 256 * units), dim3(256), 0, ctx->stream, total,
                           static_cast<int32_t>(per), fast_div(per), src_block,
                           static_cast<const U *>(src), static_cast<U *>(out));
    };
    if (one) launch(bcrs_gather_blocks<U, 1>, 1);
    else launch(bcrs_gather_blocks<U, kGatherUnits>, kGatherUnits);
}

static int gather_blocks(smax_hip_ctx ctx, const smax_hip_bcrs_info &T,
                         const void *src) {
    if (T.n_blocks == 0) return SMAX_HIP_SUCCESS;
    const int64_t bytes = T.h_pad * T.w_pad * T.val_bytes;
    // the widest unit that divides a block and both addresses
    const uintptr_t all = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(T.val) |
                          static_cast<uintptr_t>(bytes);
    if (all % 16 == 0)
        launch_gather_blocks<Quad>(ctx, T.n_blocks, bytes, T.src_block, src, T.val);
    else if (all % 8 == 0)
        launch_gather_blocks<uint64_t>(ctx, T.n_blocks, bytes, T.src_block, src, T.val);
    else if (all % 4 == 0)
        launch_gather_blocks<uint32_t>(ctx, T.n_blocks, bytes, T.src_block, src, T.val);
    else
        launch_gather_blocks<uint16_t>(ctx, T.n_blocks, bytes, T.src_block, src, T.val);
    SMAX_HIP_LAUNCHED(ctx, "bcrs_gather_blocks");
    return SMAX_HIP_SUCCESS;
}

// VL entries from p in one access (VL * sizeof(A) is 16 with p 16-byte
// aligned, or VL is 1), predicated per run on v < k.
template <typename A, int KP, int VL>
__device__ __forceinline__ void load_cols(const A *__restrict__ p, int64_t k, A (&out)[KP]) {
#pragma unroll
    for (int v = 0; v < KP; v += VL) {
        A run[VL];
#pragma unroll
        for (int i = 0; i < VL; ++i) run[i] = 0;
        if (v < k) load_run<A, VL>(p + v, run);
#pragma unroll
        for (int i = 0; i < VL; ++i) out[v + i] = run[i];
    }
}

// One thread per block line, the positions of a block that are contiguous in
// memory: a row of a row-major block (its G row against the block's w_pad X
// rows), a column of a column-major one (its X row against the h_pad G rows).
// The thread keeps the line's own operand row in registers (k <= 32) and
// forms each position's sum by itself, in the tree of a group of KP lanes (KP
// the power of two >= k, at most 64): lane l's chain over v = l, l + KP, ...,
// then the xor-butterfly's halves, KP/2 first.
//
// What bounds it: the vector memory path, 16 bytes a lane and load (b + 1
// operand rows of k entries per line of b results), and the store of dvals.
// The results do not depend on who computes them, so the split is free: with
// a group of KP lanes per position (each lane searching the position's block
// row in row_ptr, 20 dependent loads) the 96^3 matrix of 4x4 blocks took
// 9.74 ms at k = 8, 4-byte entries.
//
// A workgroup takes `iters` x 256 consecutive lines, so stores are contiguous
// whatever the block shape and block rows may have any length; it finds its
// first block's row once (wave_row_of) and writes the row of each of its
// blocks to LDS.
constexpr int kSddmmIters = 8;  // at most: 2048 lines a workgroup

// Lines of M results load all their operand rows before the sums where 64
// bytes a row or less leave the registers for it; by itself the compiler keeps
// two or three loads in flight (96^3, 4x4, 4-byte entries, k = 8: 302 -> 266
// us; 64^3, 3x3, FP64, k = 8: 89 -> 77).
template <typename A, int KP>
constexpr bool kSddmmAtOnce = KP * sizeof(A) <= 64;

struct LineSizes {  // one argument, as PartSizes
    int64_t n_blocks, n_block_rows, k;
    int iters, n_lines, lines_real, n_out, outs_real, h_pad, w_pad, col_major;
};

template <typename A, int KP, int VL, int M>
__global__ __launch_bounds__(256) void bcrs_sddmm_lines(
    LineSizes sizes, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
    const A *__restrict__ Gm, const A *__restrict__ X, A *__restrict__ dvals) {
    const int64_t n_blocks = sizes.n_blocks, n_block_rows = sizes.n_block_rows, k = sizes.k;
    const int iters = sizes.iters, n_lines = sizes.n_lines, lines_real = sizes.lines_real;
    const int n_out = sizes.n_out, outs_real = sizes.outs_real;
    const int h_pad = sizes.h_pad, w_pad = sizes.w_pad;
    const bool col_major = sizes.col_major != 0;
    __shared__ int32_t row_of[256 * kSddmmIters + 1];
    const int span = iters * 256;
    const int64_t t0 = xcd_block(blockIdx.x, gridDim.x) * span;
    const int64_t j0 = t0 / n_lines;
    const int first = static_cast<int>(t0 - j0 * n_lines);
    // blocks of this workgroup: [j0, j1)
    const int64_t jn = j0 + (first + span - 1) / n_lines + 1;
    const int64_t j1 = jn < n_blocks ? jn : n_blocks;
    if (j0 >= n_blocks) return;  // whole workgroups
    for (int64_t r = wave_row_of(row_ptr, n_block_rows, j0) + threadIdx.x;
         r < n_block_rows; r += 256) {
        const int64_t s = row_ptr[r], e = row_ptr[r + 1];
        if (s >= j1) break;
        for (int64_t j = s > j0 ? s : j0; j < (e < j1 ? e : j1); ++j)
            row_of[j - j0] = static_cast<int32_t>(r);
    }
    __syncthreads();
    constexpr bool kKeep = KP <= 32;  // the line's own operand row stays in registers
    constexpr bool kAtOnce = kSddmmAtOnce<A, KP>;
    for (int it = 0; it < iters; ++it) {
        const int q = first + it * 256 + static_cast<int>(threadIdx.x);
        const int jl = q / n_lines, i = q - jl * n_lines;
        const int64_t j = j0 + jl;
        if (j >= n_blocks) break;
        A *out = dvals + (j * n_lines + i) * n_out;
        const int64_t r = row_of[jl], c = col[j];
        const A *grow = Gm + r * h_pad * k, *xrow = X + c * w_pad * k;
        const A *own = (col_major ? xrow : grow) + i * k;
        const A *others = col_major ? grow : xrow;
        A f[kKeep ? KP : 1];
        if constexpr (kKeep)
            if (i < lines_real) load_cols<A, KP, VL>(own, k, f);
        const auto halve = [](A (&p)[KP]) {
#pragma unroll
            for (int off = KP / 2; off >= 1; off >>= 1)
#pragma unroll
                for (int v = 0; v < off; ++v) p[v] += p[v + off];
        };
        auto position = [&](int m) -> A {
            if (i >= lines_real || m >= outs_real) return 0;
            const A *w = others + m * k;
            A p[KP];
            if constexpr (kKeep) {
                A b[KP];
                load_cols<A, KP, VL>(w, k, b);
#pragma unroll
                for (int v = 0; v < KP; ++v) p[v] = __builtin_elementwise_fma(f[v], b[v], A(0));
            } else {
#pragma unroll
                for (int v = 0; v < KP; ++v) p[v] = 0;
                for (int64_t v0 = 0; v0 < k; v0 += KP) {
#pragma unroll
                    for (int v = 0; v < KP; v += VL) {
                        if (v0 + v >= k) continue;
                        A a[VL], b[VL];
                        load_run<A, VL>(own + v0 + v, a);
                        load_run<A, VL>(w + v0 + v, b);
#pragma unroll
                        for (int u = 0; u < VL; ++u)
                            p[v + u] = __builtin_elementwise_fma(a[u], b[u], p[v + u]);
                    }
                }
            }
            halve(p);
            return p[0];
        };
        if constexpr (M > 0 && kAtOnce) {
            A sums[M] = {};
            if (i < lines_real) {
                A b[M][KP];
#pragma unroll
                for (int m = 0; m < M; ++m)
                    load_cols<A, KP, VL>(others + (m < outs_real ? m : 0) * k, k, b[m]);
                __builtin_amdgcn_sched_barrier(0);  // every row requested before the sums
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    A p[KP];
#pragma unroll
                    for (int v = 0; v < KP; ++v)
                        p[v] = __builtin_elementwise_fma(f[v], b[m][v], A(0));
                    halve(p);
                    if (m < outs_real) sums[m] = p[0];
                }
            }
            store_run<A, M>(out, sums);
        } else if constexpr (M > 0) {
            A sums[M];
#pragma unroll
            for (int m = 0; m < M; ++m) sums[m] = position(m);
            store_run<A, M>(out, sums);
        } else {
            for (int m = 0; m < n_out; ++m) out[m] = position(m);
        }
    }
}

template <typename A, int KP, int VL, int M>
static void launch_bcrs_sddmm_lines(smax_hip_ctx ctx, const smax_hip_bcrs_info &in, int64_t k,
                                    const void *Gm, const void *X, void *dv) {
    const bool cm = in.block_col_major != 0;
    const int64_t n_lines = cm ? in.w_pad : in.h_pad, lines = in.n_blocks * n_lines;
    // fewer lines a workgroup while that leaves CUs idle
    int64_t iters = lines / (256 * 2048);
    iters = iters < 1 ? 1 : iters > kSddmmIters ? kSddmmIters : iters;
    const LineSizes sizes{in.n_blocks,
                          in.n_block_rows,
                          k,
                          static_cast<int>(iters),
                          static_cast<int>(n_lines),
                          static_cast<int>(cm ? in.b_w : in.b_h),
                          static_cast<int>(cm ? in.h_pad : in.w_pad),
                          static_cast<int>(cm ? in.b_h : in.b_w),
                          static_cast<int>(in.h_pad),
                          static_cast<int>(in.w_pad),
                          cm ? 1 : 0};
    hipLaunchKernelGGL((bcrs_sddmm_lines<A, KP, VL, M>),
                       grid_for(lines, static_cast<int>(256 * iters)), dim3(256), 0, ctx->stream,
                       sizes, in.row_ptr, in.col, static_cast<const A *>(Gm),
                       static_cast<const A *>(X), static_cast<A *>(dv));
}

// 16-byte loads when every operand row is 16-byte aligned; 16-byte stores for
// lines of four results.
template <typename A, int KP, int VL>
static void launch_bcrs_sddmm_vl(smax_hip_ctx ctx, const smax_hip_bcrs_info &in, int64_t k,
                                 const void *Gm, const void *X, void *dv) {
    const int64_t out = aligned16(dv, dv) ? (in.block_col_major ? in.h_pad : in.w_pad) : 0;
    if constexpr (kSddmmAtOnce<A, KP>) {
        if (out == 2) return launch_bcrs_sddmm_lines<A, KP, VL, 2>(ctx, in, k, Gm, X, dv);
        if (out == 3) return launch_bcrs_sddmm_lines<A, KP, VL, 3>(ctx, in, k, Gm, X, dv);
    }
    if (out == 4) return launch_bcrs_sddmm_lines<A, KP, VL, 4>(ctx, in, k, Gm, X, dv);
    launch_bcrs_sddmm_lines<A, KP, VL, 0>(ctx, in, k, Gm, X, dv);
}

template <typename A, int KP>
static void launch_bcrs_sddmm(smax_hip_ctx ctx, const smax_hip_bcrs_info &in, int64_t k,
                              const void *Gm, const void *X, void *dv) {
    constexpr int Q = 16 / static_cast<int>(sizeof(A));
    if constexpr (KP >= Q) {
        if (k % Q == 0 && aligned16(Gm, X))
            return launch_bcrs_sddmm_vl<A, KP, Q>(ctx, in, k, Gm, X, dv);
    }
    launch_bcrs_sddmm_vl<A, KP, 1>(ctx, in, k, Gm, X, dv);
}

template <typename A>
static int bcrs_sddmm(smax_hip_ctx ctx, const smax_hip_bcrs_info &in, int64_t k, const void *Gm,
                      const void *X, void *dv) {
    if (k <= 1) launch_bcrs_sddmm<A, 1>(ctx, in, k, Gm, X, dv);
    else if (k <= 2) launch_bcrs_sddmm<A, 2>(ctx, in, k, Gm, X, dv);
    else if (k <= 4) launch_bcrs_sddmm<A, 4>(ctx, in, k, Gm, X, dv);
    else if (k <= 8) launch_bcrs_sddmm<A, 8>(ctx, in, k, Gm, X, dv);
    else if (k <= 16) launch_bcrs_sddmm<A, 16>(ctx, in, k, Gm, X, dv);
    else if (k <= 32) launch_bcrs_sddmm<A, 32>(ctx, in, k, Gm, X, dv);
    else launch_bcrs_sddmm<A, 64>(ctx, in, k, Gm, X, dv);
    SMAX_HIP_LAUNCHED(ctx, "bcrs_sddmm_lines");
    return SMAX_HIP_SUCCESS;
}

}  // namespace smaxhip

extern "C" {

int smax_hip_bcrs_transpose(smax_hip_ctx ctx, smax_hip_bcrs A, smax_hip_bcrs *out) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, A && out, "smax_hip_bcrs_transpose: null argument");
    *out = nullptr;
    const smax_hip_bcrs_info &a = A->info;
    const int64_t nb = a.n_blocks, m = nb > 0 ? nb : 1;
    smax_hip_bcrs_info t{};
    t.n_block_rows = a.n_block_cols;
    t.n_block_cols = a.n_block_rows;
    t.n_blocks = nb;
    t.b_h = a.b_w;
    t.b_w = a.b_h;
    t.h_pad = a.w_pad;
    t.w_pad = a.h_pad;
    t.val_bytes = a.val_bytes;
    t.block_col_major = a.block_col_major ? 0 : 1;
    RadixSort sorter(ctx);
    int rc = sorter.reserve(m);
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&t.row_ptr),
                       4 * (t.n_block_rows + 1), "bcrs transpose");
    if (!rc) rc = dev_alloc(ctx, reinterpret_cast<void **>(&t.col), 4 * m, "bcrs transpose");
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&t.src_block), 4 * m,
                       "bcrs transpose");
    if (!rc) rc = dev_alloc(ctx, &t.val, a.val_bytes * m * a.h_pad * a.w_pad, "bcrs transpose");
    if (!rc) rc = sorter.sort(reinterpret_cast<const uint32_t *>(a.col), nb, a.n_block_cols);
    if (!rc)
        rc = sorter.transposed_pattern(a.n_block_rows, t.n_block_rows, nb, a.row_ptr, t.row_ptr,
                                       t.col);
    if (!rc && nb > 0) {
        const hipError_t e = hipMemcpyAsync(t.src_block, sorter.vals(), 4 * nb,
                                            hipMemcpyDeviceToDevice, ctx->stream);
        if (e != hipSuccess) rc = hip_fail(ctx, e, "src_block copy");
        if (!rc) rc = gather_blocks(ctx, t, a.val);
    }
    (void)hipStreamSynchronize(ctx->stream);
    if (rc) {
        dev_free(t.row_ptr);
        dev_free(t.col);
        dev_free(t.src_block);
        dev_free(t.val);
        return rc;
    }
    smax_hip_bcrs h = new smax_hip_bcrs_s();
    h->info = t;
    *out = h;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_bcrs_refresh_values(smax_hip_ctx ctx, smax_hip_bcrs T,
                                 const void *src_val) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, T && src_val && T->info.src_block,
                     "smax_hip_bcrs_refresh_values: not a transpose or null input");
    return gather_blocks(ctx, T->info, src_val);
}

int smax_hip_bcrs_sddmm(smax_hip_ctx ctx, int value_type, smax_hip_bcrs A, int64_t k,
                        const void *G, const void *X, void *dvals) {
    SMAX_HIP_CHECK_CTX(ctx);
    if (!valid_value_type(value_type))
        return fail(ctx, SMAX_HIP_ERROR_UNSUPPORTED, "smax_hip_bcrs_sddmm: value type %d",
                    value_type);
    SMAX_HIP_REQUIRE(ctx, A && k > 0 && G && X && dvals,
                     "smax_hip_bcrs_sddmm: bad arguments");
    if (!extent_ok(A->info.n_block_rows * A->info.h_pad, k) ||
        !extent_ok(A->info.n_block_cols * A->info.w_pad, k))
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "smax_hip_bcrs_sddmm: k = %lld exceeds the launch limits", (long long)k);
    if (A->info.n_blocks == 0) return SMAX_HIP_SUCCESS;
    return value_type == SMAX_HIP_F64 ? bcrs_sddmm<double>(ctx, A->info, k, G, X, dvals)
                                      : bcrs_sddmm<float>(ctx, A->info, k, G, X, dvals);
}

}  // extern "C"
