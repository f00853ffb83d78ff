// Differentiation support: the SELL-C-sigma layout of A^T and the SDDMM
// value gradient on A's SELL layout.  Neither has a reference counterpart.
//
// A^T: the CRS positions j = 0..nnz-1 are already in row-major order, so a
// *stable* sort of (col[j], j) by column yields A^T's CRS with every column's
// entries in ascending original row order.  The sort is an LSD radix sort
// whose scatter ranks come from ballots and prefix sums only (no atomics
// decide an order), so the layout is deterministic.  The resulting
// CRS of A^T goes through the same GPU SELL conversion as A, with src_index
// pointing back at A's CRS nonzeros.
//
// SDDMM: dvals[src_index[e]] = sum_v G[r*k+v] * X[col[e]*k+v] for every stored
// element e of SELL row r.  The reduction tree depends only on k: with P the
// smallest power of two >= k, g = clamp(P / 4, 1, 64) lanes share an element,
// lane l sums v in [l*Q, min(k, l*Q + Q)), Q = ceil(k / g), with an fma chain
// from zero, and an xor-butterfly adds the g partial sums.  Up to k = 256 the
// lanes of a group share one row (SpMM order): the G row is read once per row
// and each element costs one coalesced X row; layouts too small for that to fill
// the chip take a group of lanes per stored element, its row from its chunk.
// Larger k take one group per stored element, with the row of each element from
// a per-element row array built on first use.  All kernels evaluate the same
// tree, so dvals do not depend on which one runs.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "convert_internal.hpp"
#include "radix.hpp"
#include "scan.hpp"

namespace smaxhip {

// ------------------------------------------------------------------ SDDMM
// elem_row[e] = original row of stored element e, -1 for padding; one lane
// per slot walks its chunk column (stores coalesced across the chunk).
__global__ __launch_bounds__(256) void k_elem_row(
    int64_t C, int64_t n_slots, int64_t n_rows, const int32_t *__restrict__ chunk_ptr,
    const int32_t *__restrict__ chunk_len, const int32_t *__restrict__ slot_len,
    const int32_t *__restrict__ slot_row, int32_t *__restrict__ elem_row) {
    const int64_t s = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (s >= n_slots) return;
    const int64_t c = s / C, i = s - c * C;
    const int64_t base = static_cast<int64_t>(chunk_ptr[c]) + i;
    const int32_t r = slot_row[s];
    const int len = r < n_rows ? slot_len[s] : 0;
    const int clen = chunk_len[c];
    for (int j = 0; j < clen; ++j) elem_row[base + static_cast<int64_t>(j) * C] = j < len ? r : -1;
}

// Lanes per element and per-lane run length of the SDDMM tree for k.
__host__ __device__ constexpr int64_t sddmm_group(int64_t k) {
    int64_t p = 1;
    while (p < k) p <<= 1;
    return p / 4 < 1 ? 1 : (p / 4 > 64 ? 64 : p / 4);
}
__host__ __device__ constexpr int64_t sddmm_run(int64_t k) {
    return (k + sddmm_group(k) - 1) / sddmm_group(k);
}

// The xor-butterfly over G lanes: every lane ends with the group's sum.
template <int G, typename A> __device__ __forceinline__ A group_sum(A acc) {
#pragma unroll
    for (int off = G / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, G);
    return acc;
}

// k > 256: one wavefront (sddmm_group(k) = 64 lanes) per stored element.
template <typename A>
__global__ __launch_bounds__(256) void scs_sddmm_kernel(
    int64_t n_elements, int64_t k, const int32_t *__restrict__ col,
    const int32_t *__restrict__ elem_row, const int32_t *__restrict__ src,
    const A *__restrict__ Gm, const A *__restrict__ X, A *__restrict__ dvals) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t e = t / kWave;
    const int lane = static_cast<int>(t % kWave);
    const bool valid = e < n_elements;
    const int32_t s = valid ? src[e] : -1;
    A acc = 0;
    if (s >= 0) {
        const int64_t r = elem_row[e];
        const int64_t c = col[e];
        const int64_t q = sddmm_run(k);
        const int64_t v1 = (lane + 1) * q < k ? (lane + 1) * q : k;
        for (int64_t v = lane * q; v < v1; ++v)
            acc = __builtin_elementwise_fma(Gm[r * k + v], X[c * k + v], acc);
    }
    acc = group_sum<kWave>(acc);
    if (s >= 0 && lane == 0) dvals[s] = acc;
}

// The same butterfly over GL >= U lanes for U elements at once: at each
// offset (GL/2 first) a lane keeps the half of its live elements that its
// lane bit selects and sends the other half to its partner, adding (own +
// partner) as group_sum does, so every element's sum is the same tree.  After
// log2(U) halving steps the remaining offsets (below GL/U) add as in
// group_sum.  Lane l returns the sum of element l / (GL / U).
// The halves are vector values, not array elements: a choice between two
// elements of one array becomes an array read at a lane-dependent index,
// which the compiler expands into a select over every element.
template <int N, int OFF, int GL, typename A>
__device__ __forceinline__ A scatter_steps(const A (&cur)[N], int l) {
    if constexpr (N == 1) {
        return cur[0];
    } else {
        constexpr int H = N / 2;
        const bool upper = (l & OFF) != 0;
        A next[H];
        if constexpr (H == 1) {
            const A keep = upper ? cur[1] : cur[0];
            const A send = upper ? cur[0] : cur[1];
            next[0] = keep + __shfl_xor(send, OFF, GL);
        } else {
            typedef A half_t __attribute__((ext_vector_type(H)));
            half_t lo, hi;
#pragma unroll
            for (int i = 0; i < H; ++i) {
                lo[i] = cur[i];
                hi[i] = cur[H + i];
            }
            const half_t keep = upper ? hi : lo;
            const half_t send = upper ? lo : hi;
#pragma unroll
            for (int i = 0; i < H; ++i) next[i] = keep[i] + __shfl_xor(send[i], OFF, GL);
        }
        return scatter_steps<H, OFF / 2, GL>(next, l);
    }
}

template <int GL, int U, typename A>
__device__ __forceinline__ A group_reduce_scatter(A (&cur)[U], int l) {
    static_assert(GL >= U, "one element per lane at most");
    A s = scatter_steps<U, GL / 2, GL>(cur, l);
#pragma unroll
    for (int off = GL / U / 2; off >= 1; off >>= 1) s += __shfl_xor(s, off, GL);
    return s;
}

// Elements per pipelined group of the row kernel, measured at N = 1M (band
// matrix, SELL-64-65536): 16 for 4 and 8 lanes (FP64 k = 16 0.61 -> 0.51 ms,
// k = 32 0.80 -> 0.69 ms; FP32 k = 32 0.403 -> 0.385 ms), 8 for 16 and more
// (FP32 k = 64 0.71 ms against 0.77 with 16) and for 1 and 2, where a lane
// holds several elements of a group and 16 would leave three or four waves per
// SIMD.
template <int GL>
constexpr int kSddmmChainGroup = GL == 4 || GL == 8 ? 16 : 8;

// What the two kernels for k <= 256 take (slots as in ScsSpmmArgs of the SpMM).
struct SddmmArgs {
    int64_t C, n_slots, n_rows, k, n_chunks, n_elements;
    FastDiv by_c;
    int64_t n_long, long_whole, long_cap;  // long slots: count, listed from the front, list size
    int32_t long_from;
    bool seq;  // src_index is consecutive within a slot
    const int32_t *long_list, *chunk_ptr, *slot_len, *order, *col, *slot_row, *src;
};

// k <= 256: GL = sddmm_group(k) lanes per slot (row), lane l with the Q =
// sddmm_run(k) entries from l * Q on of the G row in registers for the whole
// row (EXACT: GL * Q = k; otherwise the last lanes read the row's last Q
// entries and skip those before their own, and lanes past the end skip all).
// Each element costs one coalesced X row, Q fmas per lane and its share of a
// butterfly: the elements of a group go through one butterfly together
// (group_reduce_scatter) that leaves each element's sum on the lane that
// stores it, consecutive CRS positions of the row.  Column indices are
// requested a group ahead; what is left of a row goes four elements at a time
// with the surplus ones computed and not stored.
//
// The elements of a row are independent, so a long slot is shared out over
// all groups of a workgroup of its own, the first n_long ones: one group
// alone took 177 us for the longest rows of a matrix of 20,000 (k = 8, FP64).
template <typename A, int GL, int Q, bool EXACT>
__global__ __launch_bounds__(256) void scs_sddmm_rows(SddmmArgs a, const A *__restrict__ Gm,
                                                      const A *__restrict__ X,
                                                      A *__restrict__ dvals) {
    constexpr int U = kSddmmChainGroup<GL>;
    constexpr int kSlots = 256 / GL;  // groups of a workgroup
    const int l = static_cast<int>(threadIdx.x) % GL, group = static_cast<int>(threadIdx.x) / GL;
    const int64_t C = a.C;
    int64_t slot, base;
    int j = 0, end;
    if (blockIdx.x < a.n_long) {
        const int64_t i = blockIdx.x;
        slot = a.long_list[i < a.long_whole ? i : a.long_cap - 1 - (i - a.long_whole)];
        const int64_t c = slot / C;
        base = static_cast<int64_t>(a.chunk_ptr[c]) + (slot - c * C);
        const int len = a.slot_len[slot];
        const int part = (len + kSlots - 1) / kSlots;
        j = group * part;
        end = j + part < len ? j + part : len;
        if (j >= len) return;  // whole groups
    } else {
        const int64_t at = (blockIdx.x - a.n_long) * kSlots + group;
        if (at >= a.n_slots) return;
        const int32_t pos = a.by_c(static_cast<int32_t>(at));
        const int64_t chunk = a.order ? static_cast<int64_t>(a.order[pos]) : pos;
        const int64_t i = at - pos * C;
        slot = chunk * C + i;
        base = static_cast<int64_t>(a.chunk_ptr[chunk]) + i;
        end = a.slot_len[slot];
        if (end >= a.long_from || end == 0) return;
    }
    const int64_t r = a.slot_row[slot];
    if (r >= a.n_rows) return;
    const int64_t k = a.k;
    const int64_t v0 = EXACT ? l * Q : run_start<Q>(l, k);
    const int skip = EXACT ? 0 : l * Q < k ? static_cast<int>(l * Q - v0) : Q;
    const int64_t row0 = a.seq ? a.src[base] : 0;  // the row's first CRS position
    A g[Q];
    load_cols_run<A, Q>(Gm + r * k + v0, g);
    const A *xcol = X + v0;
    // m of the UU elements from position p on, with columns c
    const auto elements = [&](auto uu, int p, int m, const int32_t *c) {
        constexpr int UU = decltype(uu)::value;
        // kPer lanes hold each result, each lane holds kNpl results
        constexpr int kPer = GL >= UU ? GL / UU : 1;
        constexpr int kNpl = GL >= UU ? 1 : UU / GL;
        const int mine = l / kPer;
        int64_t to[kNpl];
#pragma unroll
        for (int n = 0; n < kNpl; ++n) {
            const int e = n * GL + mine;
            to[n] = -1;
            if (l % kPer == 0 && e < m)
                to[n] = a.seq ? row0 + p + e : a.src[base + static_cast<int64_t>(p + e) * C];
        }
        A xv[UU][Q];
#pragma unroll
        for (int u = 0; u < UU; ++u)
            load_cols_run<A, Q>(xcol + static_cast<int64_t>(c[u]) * k, xv[u]);
        A part[UU];
#pragma unroll
        for (int u = 0; u < UU; ++u) {
            A acc = 0;
#pragma unroll
            for (int t = 0; t < Q; ++t) {
                const A next = __builtin_elementwise_fma(g[t], xv[u][t], acc);
                acc = EXACT || t >= skip ? next : acc;
            }
            part[u] = acc;
        }
        if constexpr (GL == 1 && UU == U) {
            // A whole group's results are one lane's, side by side; stored one
            // by one, 1,000,000 rows, k = 1, FP32 take 379 us, this way 270.
            if (a.seq) {
                store_cols_run<A, U>(dvals + row0 + p, part);
                return;
            }
        }
        if constexpr (GL >= UU) {
            const A sum = group_reduce_scatter<GL, UU>(part, l);
            if (to[0] >= 0) dvals[to[0]] = sum;
        } else {
            // Of a whole group every lane stores all it holds.  The check of
            // each costs 1,000,000 rows, k = 8, FP32 395 us against 366; with
            // FP64 and four lanes a slot leaving it out does (k = 16: 374, 393).
            constexpr bool kAll = UU == U && (sizeof(A) == 4 || GL <= 2);
#pragma unroll
            for (int n = 0; n < kNpl; ++n) {
                A piece[GL];
#pragma unroll
                for (int i = 0; i < GL; ++i) piece[i] = part[n * GL + i];
                const A sum = group_reduce_scatter<GL, GL>(piece, l);
                if (kAll || to[n] >= 0) dvals[to[n]] = sum;
            }
        }
    };
    const int full = j + (end - j) / U * U;
    if (j < full) {
        int32_t c0[U], c1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) c0[u] = a.col[base + static_cast<int64_t>(j + u) * C];
        for (; j < full; j += U) {
            if (j + U < full)
#pragma unroll
                for (int u = 0; u < U; ++u)
                    c1[u] = a.col[base + static_cast<int64_t>(j + U + u) * C];
            elements(std::integral_constant<int, U>{}, j, U, c0);
#pragma unroll
            for (int u = 0; u < U; ++u) c0[u] = c1[u];
        }
    }
    constexpr int R = 4;
    for (; j < end; j += R) {
        int32_t c[R];
#pragma unroll
        for (int u = 0; u < R; ++u)
            c[u] = a.col[base + static_cast<int64_t>(j + u < end ? j + u : end - 1) * C];
        elements(std::integral_constant<int, R>{}, j, end - j < R ? end - j : R, c);
    }
}

// k <= 256, small layouts: a group of GL lanes per stored element (padding
// included), in the tree of the row kernel.  A wavefront finds its first
// element's chunk by search, a lane goes on from there as in the conversion's
// fill.  Bound by dependent loads: a slot's elements are independent, and here
// no lane runs more than one, where the row kernel's slots of up to 128 take
// 16 to 30 us (5000 rows of a heavy-tailed band, k = 5, FP64: 22 us by rows,
// 4.6 so; 2000 rows, k = 100: 17 and 9).
template <typename A, int GL, int Q, bool EXACT>
__global__ __launch_bounds__(256) void scs_sddmm_elements(SddmmArgs a, const A *__restrict__ Gm,
                                                          const A *__restrict__ X,
                                                          A *__restrict__ dvals) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t first = (t & ~static_cast<int64_t>(kWave - 1)) / GL, e = t / GL;
    if (first >= a.n_elements) return;  // whole wavefronts
    const int l = static_cast<int>(threadIdx.x) % GL;
    const bool valid = e < a.n_elements;
    // Loaded together, so that X does not wait for one after the other; a
    // wavefront of padding alone ends here.
    const int64_t at = valid ? e : a.n_elements - 1;
    const int32_t from = a.src[at], col = a.col[at], to = valid ? from : -1;
    if (__ballot(to >= 0) == 0) return;
    const int64_t k = a.k;
    const int64_t v0 = EXACT ? l * Q : run_start<Q>(l, k);
    const int skip = EXACT ? 0 : l * Q < k ? static_cast<int>(l * Q - v0) : Q;
    A x[Q], g[Q];
    load_cols_run<A, Q>(X + static_cast<int64_t>(col) * k + v0, x);
    int64_t c = wave_row_of(a.chunk_ptr, a.n_chunks, first);
    A acc = 0;
    if (to >= 0) {
        int32_t base = a.chunk_ptr[c], end = a.chunk_ptr[c + 1];
        for (int step = 0; e >= end && step < 8; ++step) {
            base = end;
            end = a.chunk_ptr[++c + 1];
        }
        if (e >= end) {
            c = row_of(a.chunk_ptr, c, a.n_chunks, e);
            base = a.chunk_ptr[c];
        }
        const int32_t off = static_cast<int32_t>(e) - base;
        const int64_t slot = c * a.C + (off - a.by_c(off) * a.C);
        load_cols_run<A, Q>(Gm + static_cast<int64_t>(a.slot_row[slot]) * k + v0, g);
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            const A next = __builtin_elementwise_fma(g[i], x[i], acc);
            acc = EXACT || i >= skip ? next : acc;
        }
    }
    acc = group_sum<GL>(acc);
    if (to >= 0 && l == 0) dvals[to] = acc;
}

// Whether a group an element is the faster one.  By rows a launch takes some 12
// us for its long chains and then a time per entry; by element a time per entry
// that a few lanes make the shorter one, but many a longer one (each entry reads
// its own G row), and a quarter of it per padding element.  In threads (lanes an
// entry), the difference is `more` eighths of the entries' and a quarter of the
// padding's; `fixed` is what the chains cost in that measure.  By element / by
// rows, us, heavy-tailed bands of 16 entries a row, rows in sort windows of 4096
// (2.5 elements an entry) and unsorted (17):
//   k = 3    FP64 400,000 rows 154 / 204, 700,000  334 / 309; unsorted 20,000 34 / 19
//   k = 5    FP64 120,000  56 / 70, FP32  49 / 49;            unsorted 20,000 52 / 19
//   k = 12   FP64 18,000   16 / 20, FP32  12 / 13;            unsorted 5000 16 / 17, 15 / 14
//   k = 24   FP64 9000     13 / 20, FP32  11 / 13;            unsorted 3000 12 / 15, 11 / 12
//   k = 48   FP64 5000     12 / 16, FP32  11 / 13;            unsorted 5000 41 / 17, 30 / 15
//   k = 100  FP64 4000     18 / 22, 5000  28.6 / 28.6
//   k = 200  FP64 4000     35 / 45, 5000  56 / 56;            unsorted 1000 14 / 15, 2000 39 / 22
static bool sddmm_by_element(int64_t nnz, int64_t n_elements, int64_t lanes, bool f64) {
    const int64_t more = lanes == 1 ? -3 : lanes == 2 ? -1 : lanes < 32 ? 4 : lanes == 32 ? 2 : 0;
    const int64_t fixed = lanes == 1   ? 11 << 16
                          : lanes == 2 ? (f64 ? 3 << 19 : 7 << 17)
                          : lanes < 32 ? (f64 ? 7 << 18 : 5 << 18)
                                       : 9 << 17;
    return nnz < 10'000'000 && (nnz * more + (n_elements - nnz) * 2) * lanes < fixed * 8;
}

template <typename A, int GL, int Q>
static void launch_sddmm_rows(smax_hip_ctx ctx, smax_hip_scs S, int64_t k, const void *Gm,
                              const void *X, void *dv) {
    const smax_hip_scs_info &in = S->info;
    SddmmArgs a{};
    a.C = in.C;
    a.n_chunks = in.n_chunks;
    a.n_elements = in.n_elements;
    a.n_slots = in.n_rows_padded;
    a.n_rows = in.n_rows;
    a.k = k;
    a.by_c = fast_div(in.C);
    a.n_long = S->longs.rows.count;
    a.long_whole = S->longs.rows.whole;
    a.long_cap = S->longs.cap;
    a.long_from = S->longs.from;
    a.seq = S->src_consecutive;
    a.long_list = S->longs.list;
    a.chunk_ptr = in.chunk_ptr;
    a.slot_len = in.slot_len;
    a.order = S->sched.order_lf;
    a.col = in.col;
    a.slot_row = in.slot_row;
    a.src = in.src_index;
    const dim3 grid(static_cast<unsigned>(a.n_long + ceil_div(a.n_slots, 256 / GL)));
    const auto g = static_cast<const A *>(Gm);
    const auto x = static_cast<const A *>(X);
    const auto d = static_cast<A *>(dv);
    if (sddmm_by_element(in.nnz, in.n_elements, GL, sizeof(A) == 8)) {
        const dim3 per_element = grid_for(in.n_elements * GL, 256);
        if (k == GL * Q)
            hipLaunchKernelGGL((scs_sddmm_elements<A, GL, Q, true>), per_element, dim3(256), 0,
                               ctx->stream, a, g, x, d);
        else if constexpr (GL > 1)
            hipLaunchKernelGGL((scs_sddmm_elements<A, GL, Q, false>), per_element, dim3(256), 0,
                               ctx->stream, a, g, x, d);
        return;
    }
    if (k == GL * Q)
        hipLaunchKernelGGL((scs_sddmm_rows<A, GL, Q, true>), grid, dim3(256), 0, ctx->stream, a, g,
                           x, d);
    else if constexpr (GL > 1)
        hipLaunchKernelGGL((scs_sddmm_rows<A, GL, Q, false>), grid, dim3(256), 0, ctx->stream, a,
                           g, x, d);
}

// sddmm_group(k) and sddmm_run(k) as template arguments, 1 <= k <= 256.
template <typename A>
static void sddmm_rows(smax_hip_ctx ctx, smax_hip_scs S, int64_t k, const void *Gm, const void *X,
                       void *dv) {
#define SMAX_SDDMM_ROWS(GL)                                                                \
    case GL:                                                                               \
        if (sddmm_run(k) == 3) launch_sddmm_rows<A, GL, 3>(ctx, S, k, Gm, X, dv);          \
        else launch_sddmm_rows<A, GL, 4>(ctx, S, k, Gm, X, dv);                            \
        break;
    switch (sddmm_group(k)) {
        SMAX_SDDMM_ROWS(2)
        SMAX_SDDMM_ROWS(4)
        SMAX_SDDMM_ROWS(8)
        SMAX_SDDMM_ROWS(16)
        SMAX_SDDMM_ROWS(32)
        SMAX_SDDMM_ROWS(64)
    default:  // one lane: k <= 4
        if (k == 1) launch_sddmm_rows<A, 1, 1>(ctx, S, k, Gm, X, dv);
        else if (k == 2) launch_sddmm_rows<A, 1, 2>(ctx, S, k, Gm, X, dv);
        else if (k == 3) launch_sddmm_rows<A, 1, 3>(ctx, S, k, Gm, X, dv);
        else launch_sddmm_rows<A, 1, 4>(ctx, S, k, Gm, X, dv);
        break;
    }
#undef SMAX_SDDMM_ROWS
}

}  // namespace smaxhip

using namespace smaxhip;

extern "C" {

int smax_hip_scs_transpose_from_crs(smax_hip_ctx ctx, int64_t n_rows,
                                    int64_t n_cols, int64_t nnz,
                                    const int32_t *row_ptr, const int32_t *col,
                                    const void *val, int64_t val_bytes,
                                    int64_t C, int64_t sigma,
                                    smax_hip_scs *out) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, out, "smax_hip_scs_transpose_from_crs: null output");
    *out = nullptr;
    SMAX_HIP_REQUIRE(ctx, n_rows > 0 && n_cols > 0 && nnz >= 0 &&
                              nnz <= INT32_MAX && row_ptr &&
                              (nnz == 0 || (col && val)),
                     "smax_hip_scs_transpose_from_crs: bad input");
    if (n_rows > INT32_MAX || n_cols > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "smax_hip_scs_transpose_from_crs: %lld x %lld exceeds int32",
                    (long long)n_rows, (long long)n_cols);
    const int64_t m = nnz > 0 ? nnz : 1;
    int32_t *t_row_ptr = nullptr, *t_col = nullptr;
    RadixSort sorter(ctx);
    int rc = sorter.reserve(m);
    if (!rc)
        rc = dev_alloc(ctx, reinterpret_cast<void **>(&t_row_ptr),
                       4 * (n_cols + 1), "transpose");
    if (!rc) rc = dev_alloc(ctx, reinterpret_cast<void **>(&t_col), 4 * m, "transpose");
    if (!rc) rc = sorter.sort(reinterpret_cast<const uint32_t *>(col), nnz, n_cols);
    if (!rc) rc = sorter.transposed_pattern(n_rows, n_cols, nnz, row_ptr, t_row_ptr, t_col);
    if (!rc)
        rc = build_scs(ctx, n_cols, n_rows, nnz, t_row_ptr, t_col, val,
                       val_bytes, sorter.vals(), C, sigma, out);
    (void)hipStreamSynchronize(ctx->stream);
    dev_free(t_row_ptr);
    dev_free(t_col);
    return rc;
}

int smax_hip_scs_sddmm(smax_hip_ctx ctx, int value_type, smax_hip_scs A,
                       int64_t k, const void *G, const void *X, void *dvals) {
    SMAX_HIP_CHECK_CTX(ctx);
    if (!valid_value_type(value_type))
        return fail(ctx, SMAX_HIP_ERROR_UNSUPPORTED,
                    "smax_hip_scs_sddmm: value type %d", value_type);
    SMAX_HIP_REQUIRE(ctx, A && k > 0 && G && X && dvals,
                     "smax_hip_scs_sddmm: bad arguments");
    SMAX_HIP_REQUIRE(ctx, !A->from_sell,
                     "smax_hip_scs_sddmm: the matrix was built from SELL arrays and has no CRS "
                     "positions; build it with smax_hip_scs_from_crs");
    const smax_hip_scs_info &in = A->info;
    if (!extent_ok(in.n_rows_padded, k) || !extent_ok(std::max<int64_t>(in.n_elements, 1), k))
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "smax_hip_scs_sddmm: k = %lld exceeds the launch limits", (long long)k);
    if (in.n_elements == 0) return SMAX_HIP_SUCCESS;
    if (k <= 256) {
        if (value_type == SMAX_HIP_F64) sddmm_rows<double>(ctx, A, k, G, X, dvals);
        else sddmm_rows<float>(ctx, A, k, G, X, dvals);
        SMAX_HIP_LAUNCHED(ctx, "scs_sddmm_rows");
        return SMAX_HIP_SUCCESS;
    }
    if (!A->elem_row) {
        int rc = dev_alloc(ctx, reinterpret_cast<void **>(&A->elem_row),
                           sizeof(int32_t) * in.n_elements, "sddmm element rows");
        if (rc) return rc;
        hipLaunchKernelGGL(k_elem_row, grid_for(in.n_rows_padded, 256), dim3(256), 0,
                           ctx->stream, in.C, in.n_rows_padded, in.n_rows, in.chunk_ptr,
                           in.chunk_lengths, in.slot_len, in.slot_row, A->elem_row);
        SMAX_HIP_LAUNCHED(ctx, "k_elem_row");
    }
    const dim3 grid = grid_for(in.n_elements * kWave, 256);
    if (value_type == SMAX_HIP_F64)
        hipLaunchKernelGGL(scs_sddmm_kernel<double>, grid, dim3(256), 0, ctx->stream,
                           in.n_elements, k, in.col, A->elem_row, in.src_index,
                           static_cast<const double *>(G), static_cast<const double *>(X),
                           static_cast<double *>(dvals));
    else
        hipLaunchKernelGGL(scs_sddmm_kernel<float>, grid, dim3(256), 0, ctx->stream,
                           in.n_elements, k, in.col, A->elem_row, in.src_index,
                           static_cast<const float *>(G), static_cast<const float *>(X),
                           static_cast<float *>(dvals));
    SMAX_HIP_LAUNCHED(ctx, "scs_sddmm_kernel");
    return SMAX_HIP_SUCCESS;
}

}  // extern "C"
