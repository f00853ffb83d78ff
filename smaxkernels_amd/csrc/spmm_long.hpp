// What the CRS and the SELL SpMM share beyond the tuned power-of-two kernels:
// runs of columns of any alignment, and the long-row path.
#pragma once

#include "common.hpp"

namespace smaxhip {

// Q consecutive entries at p, aligned only as an entry is (one 16-byte access
// where Q entries are 16 bytes; the hardware takes dword-aligned ones).
template <typename A, int Q>
struct __attribute__((packed, aligned(4))) RunOf {
    A e[Q];
};
template <typename A, int Q>
__device__ __forceinline__ void load_cols_run(const A *__restrict__ p, A (&out)[Q]) {
    const RunOf<A, Q> v = *reinterpret_cast<const RunOf<A, Q> *>(p);
#pragma unroll
    for (int i = 0; i < Q; ++i) out[i] = v.e[i];
}
template <typename A, int Q>
__device__ __forceinline__ void store_cols_run(A *__restrict__ p, const A (&in)[Q]) {
    RunOf<A, Q> v;
#pragma unroll
    for (int i = 0; i < Q; ++i) v.e[i] = in[i];
    *reinterpret_cast<RunOf<A, Q> *>(p) = v;
}

// k columns in runs of Q <= k: lane l of a row's ceil(k / Q) lanes owns the
// columns from run_start(l); the last run is moved back to end at k, so it may
// share columns with the one before (both form the same chains).
template <int Q>
__device__ __forceinline__ int64_t run_start(int64_t l, int64_t k) {
    return l * Q + Q <= k ? l * Q : k - Q;
}
inline int64_t run_lanes(int64_t k, int64_t q) { return ceil_div(k, q); }

// Long rows: at least this many entries and eight times the mean length (so
// that they are few).  They run in long_row, a wavefront each, from
// kLongestRow entries on a workgroup each.
constexpr int64_t kLongRow = 128, kLongestRow = 512;
inline int64_t long_row_from(int64_t nnz, int64_t n_rows) {
    const int64_t eight = (8 * nnz + n_rows - 1) / n_rows;
    return eight > kLongRow ? eight : kLongRow;
}

// In SELL a long slot alone also pays for its columns and values, one line an
// entry that the other slots of its chunk would share; in large matrices, where
// the longest rows no longer decide the time, fewer slots are long.  Band
// matrices with rows of up to 2000 entries, us with this rule, then with a line
// of 128 / 256 / 512 / 1024 entries and without long slots:
//   40,013 rows, FP64 k = 10       32 |  32 /  34 /  56 / 100, 208
//   200,003, FP64 k = 10           78 |  78 /  79 / 103 / 133, 274
//   200,003, FP32 k = 32           62 |  65 /  63 /  76 / 117, 205
//   500,009, FP64 k = 16          166 | 169 / 171 / 165 / 169, 258
//   1,000,000, FP32 k = 32        315 | 329 / 323 / 323 / 317, 427
//   1,000,000, FP64 k = 16        356 | 377 / 368 / 367 / 358, 381
//   2,000,003, FP64 k = 8         615 | 661 / 631 / 644 / 615, 655
inline int64_t long_slot_from(int64_t nnz, int64_t n_rows) {
    const int64_t row = long_row_from(nnz, n_rows), part = nnz / 16000;
    const int64_t most = part < 1024 ? part : 1024;
    return row > most ? row : most;
}

// Long rows in front of a launch's other rows: the first `whole` workgroups
// take one row each, the next ceil((count - whole) / 4) take four.
struct LongRows {
    int64_t whole = 0, count = 0;
    __host__ __device__ int64_t blocks() const { return whole + (count - whole + 3) / 4; }
};

// One row's outputs by NT threads, a wavefront (64) or a workgroup (256).  A
// row is one fma chain per column whatever its length, so a lane that gathers
// and chains by itself pays a memory round trip every eight entries: a row of
// 2000 entries took 128 us, longer than all other rows of a matrix of 40,013
// (16 us).  Here all lanes gather X runs, a tile of R x NT runs (at most NT
// entries) ahead, into LDS, column by column; a lane per column then chains
// its entries from there, which lie side by side, at about 11 cycles an entry
// (6 of them the fma), the next tile's gathers in flight meanwhile.  The
// chain's order, and so Y, is unchanged.  Wavefronts for the many rows that
// are just long: three of a workgroup's four would only wait.
//   entry j of the row: column col[base + j * stride], value val[...] alike;
//   lds: LongRowLds<A, Q, NT>::kStore elements, 16-byte aligned.
constexpr int kLongRuns = 4;
constexpr int kLongCols = 64;  // columns of a pass, a lane of one wavefront each

template <typename A, int Q, int NT>
struct LongRowLds {
    static constexpr int kUnit = 16 / static_cast<int>(sizeof(A));
    // Columns lie an odd number of 16-byte units apart: 16 lanes' reads take
    // all banks once.
    static constexpr int kXs = NT * kLongRuns * Q + (kLongCols + Q) * kUnit;
    static constexpr int kStore = kXs + NT;
};

template <int VT, int Q, int NT>
__device__ __forceinline__ void long_row(
    typename vt<VT>::vec_t *lds, int tid, int32_t len, int64_t base, int64_t stride,
    const int32_t *__restrict__ col, const typename vt<VT>::val_t *__restrict__ val, int64_t k,
    const typename vt<VT>::vec_t *__restrict__ X, int64_t ldx,
    typename vt<VT>::vec_t *__restrict__ y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    using L = LongRowLds<A, Q, NT>;
    constexpr int R = kLongRuns, U = 8;
    // A row that was long when the list was made may be empty by now (a plan
    // used with another pattern): it has no last entry to load.
    if (len <= 0) {
        for (int64_t v = tid; v < k; v += NT) y[v] = 0;
        return;
    }
    A *const xs = lds, *const vs = lds + L::kXs;
    const auto barrier = [] {
        if constexpr (NT > kWave) {
            __syncthreads();
        } else {  // one wavefront: its LDS accesses stay in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    };
    const int32_t passes = static_cast<int32_t>((k + kLongCols - 1) / kLongCols);
    const int32_t width = static_cast<int32_t>((k + passes - 1) / passes);
    const int32_t g = (width + Q - 1) / Q;
    // Entries of a tile: whole groups of the chain, a value per thread.
    const int32_t most = NT * R / g & ~(U - 1);
    const int32_t ept = most < NT ? most : NT;
    const int32_t run = ept + L::kUnit;  // a column's place; U is even in units
    int32_t eu[R], at[R], off[R];        // this thread's entries, their LDS places, columns
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int32_t f = u * NT + tid;
        eu[u] = f / g;
        off[u] = static_cast<int32_t>(run_start<Q>(f - eu[u] * g, width));
        at[u] = eu[u] < ept ? off[u] * run + eu[u] : -1;
        if (eu[u] >= ept) eu[u] = 0;  // none: repeats a load
    }
    for (int32_t pass = 0; pass < passes; ++pass) {
        const int64_t v0 = pass * width + width <= k ? pass * width : k - width;
        int32_t c[R];
        A xr[R][Q];
        V vr;
        // Past the row's end its last entry is loaded again: under conditions
        // the loads would be waited for where their results merge.
        const auto load_columns = [&](int32_t t0) {
#pragma unroll
            for (int u = 0; u < R; ++u)
                c[u] = col[base + (t0 + eu[u] < len ? t0 + eu[u] : len - 1) * stride];
        };
        const auto gather = [&](int32_t t0) {
#pragma unroll
            for (int u = 0; u < R; ++u)
                load_cols_run<A, Q>(X + static_cast<int64_t>(c[u]) * ldx + v0 + off[u], xr[u]);
            vr = val[base + (t0 + tid < len ? t0 + tid : len - 1) * stride];
        };
        load_columns(0);
        gather(0);
        load_columns(ept);
        A acc = 0;
        for (int32_t t0 = 0; t0 < len; t0 += ept) {
            // What is past the row's end is -0 * 0, which leaves every
            // accumulator as it is, signed zeros included.
#pragma unroll
            for (int u = 0; u < R; ++u)
                if (at[u] >= 0) {
                    const bool in = t0 + eu[u] < len;
#pragma unroll
                    for (int q = 0; q < Q; ++q) xs[at[u] + q * run] = in ? xr[u][q] : A(0);
                }
            if (tid < ept) vs[tid] = t0 + tid < len ? T::widen(vr) : A(-0.0);
            barrier();
            if (t0 + ept < len) {
                gather(t0 + ept);
                load_columns(t0 + 2 * ept);
            }
            if (tid < width) {
                const A *px = xs + tid * run;
                const int32_t m = len - t0 < ept ? len - t0 : ept;
                for (int32_t e = 0; e < m; e += U) {
                    A w[U], b[U];
                    load_run<A, U>(vs + e, w);
                    load_run<A, U>(px + e, b);
#pragma unroll
                    for (int u = 0; u < U; ++u) acc = T::fma_(w[u], b[u], acc);
                }
            }
            barrier();
        }
        if (tid < width) y[v0 + tid] = acc;
    }
}

// The long rows' workgroups of a launch of 256 threads: workgroup `block` of
// rows.blocks().  row_at(i) gives the i-th long row's (length, first entry,
// output row).
template <int VT, int Q, typename RowAt>
__device__ __forceinline__ void long_rows(
    const LongRows &rows, int64_t block, const RowAt &row_at, int64_t stride,
    const int32_t *__restrict__ col, const typename vt<VT>::val_t *__restrict__ val, int64_t k,
    const typename vt<VT>::vec_t *__restrict__ X, int64_t ldx,
    typename vt<VT>::vec_t *__restrict__ Y, int64_t ldy) {
    using A = typename vt<VT>::vec_t;
    constexpr int kWhole = LongRowLds<A, Q, 256>::kStore, kPart = LongRowLds<A, Q, kWave>::kStore;
    __shared__ __align__(16) A lds[kWhole > 4 * kPart ? kWhole : 4 * kPart];
    const int tid = static_cast<int>(threadIdx.x);
    if (block < rows.whole) {
        const auto r = row_at(block);
        long_row<VT, Q, 256>(lds, tid, r.len, r.base, stride, col, val, k, X, ldx,
                             Y + r.row * ldy);
        return;
    }
    const int wave = tid / kWave;
    const int64_t i = rows.whole + (block - rows.whole) * 4 + wave;
    if (i >= rows.count) return;  // whole wavefronts
    const auto r = row_at(i);
    long_row<VT, Q, kWave>(lds + wave * kPart, tid & (kWave - 1), r.len, r.base, stride, col, val,
                           k, X, ldx, Y + r.row * ldy);
}
struct LongRowAt {
    int32_t len;
    int64_t base, row;
};

// One lane's chains over a row in groups of eight entries, the next group's
// columns and values requested before this group's X runs (LATE: after them);
// the last, shorter group is loaded at once too.  Any k >= Q.
//
// Loads return in order, so X runs requested last are also waited for until
// the next group has come: where a row's few lanes are all that is left, the
// longer wait (BF16 without a plan, 5000 rows, k = 8: 80 us, LATE 71).  Where
// long rows run elsewhere and the others are many, it keeps more requests in
// flight (FP32 with a plan, 50,000 rows, 2%), except in FP32 SELL, whose slots
// share lines (600,000 rows, k = 8: 203 and 172 us).
template <int VT, int Q, bool LATE>
__device__ __forceinline__ void run_chain(
    int64_t base, int64_t stride, int32_t len, const int32_t *__restrict__ col,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ X, int64_t ldx,
    typename vt<VT>::vec_t (&acc)[Q]) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    constexpr int U = 8;
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] = 0;
    const int32_t full = len & ~(U - 1);
    int32_t c0[U], c1[U];
    V w0[U], w1[U];
    const auto load_full = [&](int32_t j, int32_t (&c)[U], V (&w)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = col[base + (j + u) * stride];
            w[u] = val[base + (j + u) * stride];
        }
    };
    if (full > 0) load_full(0, c0, w0);
    for (int32_t j = 0; j < full; j += U) {
        // 2-byte values loaded under a condition are waited for at once; the
        // last group loads itself again (40,013 rows, k = 20: 30.4 -> 26.9 us;
        // 8-byte values 82 -> 89 us at 200,003 rows, k = 10).
        const auto load_next = [&] {
            if (sizeof(V) == 2 || j + U < full) load_full(j + U < full ? j + U : j, c1, w1);
        };
        if constexpr (!LATE) load_next();
        A xv[U][Q];
#pragma unroll
        for (int u = 0; u < U; ++u)
            load_cols_run<A, Q>(X + static_cast<int64_t>(c0[u]) * ldx, xv[u]);
        if constexpr (LATE) load_next();
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < Q; ++q) acc[q] = T::fma_(T::widen(w0[u]), xv[u][q], acc[q]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c0[u] = c1[u];
            w0[u] = w1[u];
        }
    }
    if (full < len) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (full + u < len) {
                c1[u] = col[base + (full + u) * stride];
                w1[u] = val[base + (full + u) * stride];
            }
        A xv[U][Q];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (full + u < len)
                load_cols_run<A, Q>(X + static_cast<int64_t>(c1[u]) * ldx, xv[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (full + u < len)
#pragma unroll
                for (int q = 0; q < Q; ++q) acc[q] = T::fma_(T::widen(w1[u]), xv[u][q], acc[q]);
    }
}

}  // namespace smaxhip
