// SELL-C-sigma SpMV and SpMM for gfx950.
//
// Layout (src/utils/convert_formats.hpp:16-132): chunk c holds C slots; its
// element j of slot i sits at chunk_ptr[c] + j*C + i, so for C = 64 one
// wavefront reads a whole 64-slot column of a chunk with one coalesced
// load per array.  Every slot is a sequential fma chain over j, exactly the
// loop of the reference (spmv_cpu_scs_impl.hpp:27-41), so results are
// bit-identical to it; padding elements (val 0, col 0) add an exact zero.
//
// The chains are unrolled: U column indices and values are loaded
// (non-temporally, they are streamed once) before the U gathers of x and the
// U dependent fmas, so each lane keeps 2U loads in flight.
#include <algorithm>
#include <cmath>
#include <functional>
#include <utility>
#include <vector>

#include "common.hpp"
#include "convert_internal.hpp"
#include "spmm_long.hpp"

namespace smaxhip {

constexpr int kScsThreads = 256;
constexpr int kScsUnroll = 8;       // generic-C chains
// C = 64 chains, elements per group (measured on the 4M-row band matrix):
// FP64 24 (0.697 / 0.641 ms at sigma = 4096 / 65536; 16: 0.707 / 0.659, with
// 128 VGPRs against 90 -- four waves per SIMD instead of five, each with more
// gathers in flight; 28 and 32 leave two waves and lose at sigma = 4096),
// FP32 16 (24: 0.519 vs 0.493 ms), BF16 values 8 (16: 0.52 vs 0.48 ms).
template <int VT>
constexpr int kScsPipeUnroll = VT == SMAX_HIP_BF16 ? 8 : VT == SMAX_HIP_F32 ? 16 : 24;

// Layouts whose chunks are at most kShortChain long (stencils: the 512^2
// Poisson matrix has 5) run each chain as one predicated group: all of a
// lane's column/value loads, then all its gathers, then the fmas, two memory
// round trips in all.  The 512^2 Poisson SpMV after the caches are flushed:
// 7.16 -> 5.98 us kernel time; back to back 4.56 -> 4.68 us.
constexpr int kShortChain = 8;

template <int VT>
__device__ __forceinline__ typename vt<VT>::vec_t
slot_chain_short(const int32_t *__restrict__ col, const typename vt<VT>::val_t *__restrict__ val,
                 const typename vt<VT>::vec_t *__restrict__ x, int64_t base, int len) {
    using T = vt<VT>;
    int32_t c[kShortChain];
    typename T::val_t v[kShortChain];
#pragma unroll
    for (int u = 0; u < kShortChain; ++u)
        if (u < len) {
            c[u] = ld_stream(col + base + u * kWave);
            v[u] = ld_stream(val + base + u * kWave);
        }
    typename T::vec_t xv[kShortChain];
#pragma unroll
    for (int u = 0; u < kShortChain; ++u)
        if (u < len) xv[u] = x[c[u]];
    typename T::vec_t acc = 0;
#pragma unroll
    for (int u = 0; u < kShortChain; ++u)
        if (u < len) acc = T::fma_(T::widen(v[u]), xv[u], acc);
    return acc;
}

// One slot's chain in groups of U: the next group's column indices and
// values are requested before this group's x gathers (software pipelining),
// so a long chain waits about one memory round trip per group instead of
// two.  The remainder runs element by element: a predicated group for it
// costs registers and measured slower on the 4M-row band matrix.
template <int VT, int U>
__device__ __forceinline__ typename vt<VT>::vec_t
slot_chain_pipe(const int32_t *__restrict__ col,
                const typename vt<VT>::val_t *__restrict__ val,
                const typename vt<VT>::vec_t *__restrict__ x, int64_t base,
                int64_t stride, int len) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    A acc = 0;
    int j = 0;
    if (len >= U) {
        int32_t c0[U];
        V v0[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c0[u] = ld_stream(col + base + u * stride);
            v0[u] = ld_stream(val + base + u * stride);
        }
        for (; j + 2 * U <= len; j += U) {
            int32_t c1[U];
            V v1[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                c1[u] = ld_stream(col + base + (j + U + u) * stride);
                v1[u] = ld_stream(val + base + (j + U + u) * stride);
            }
            A xv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) xv[u] = x[c0[u]];
#pragma unroll
            for (int u = 0; u < U; ++u) acc = T::fma_(T::widen(v0[u]), xv[u], acc);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                c0[u] = c1[u];
                v0[u] = v1[u];
            }
        }
        A xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = x[c0[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) acc = T::fma_(T::widen(v0[u]), xv[u], acc);
        j += U;
    }
    for (; j < len; ++j) {
        const int32_t c = ld_stream(col + base + j * stride);
        const auto v = ld_stream(val + base + j * stride);
        acc = T::fma_(T::widen(v), x[c], acc);
    }
    return acc;
}

// A long chunk by a whole workgroup.  A chunk's longest rows are one lane's
// chain each: by a wavefront, the chunk takes a memory round trip for every U
// columns, with ever fewer of its lanes still at work.  Here all 256 threads
// gather a tile of kLongTile entries, request the next tile's while its first
// wavefront runs the chains out of LDS, and a tile's columns are as many as
// its lanes that are still live leave room for (64 lanes: 32 columns, 5 lanes:
// 256), each lane's entries side by side in LDS.  What is past a row's end is
// stored as -0 * 0, which leaves every accumulator as it is, signed zeros
// included.  Bound by the longest row's chain (up to some 100,000 rows) and by
// the gathers beyond; rows of up to 2000 entries in a band, before and after:
//   SELL-64-4096, FP64     20,000 rows   71 ->  36 us, 1,000,000  241 -> 169 us
//   SELL-64-4096, BF16    300,007       174 ->  66
//   SELL-64-65536, FP64   300,007       210 ->  70,    4,000,000  698 -> 680
//   SELL-64-64, FP64       20,000       210 ->  37,    4,000,000 1124 -> 1066
//   SELL-32-64, FP64      100,000       305 ->  52
// Tiles of 1024: 300,007 rows at sigma = 65536 7% slower.
constexpr int kLongTile = 2048;
// A long chunk's lanes are split between up to kLongParts workgroups, as many
// (a power of two) as leave each `share` entries or more.
constexpr int kLongParts = 8;
__host__ __device__ __forceinline__ int long_parts(int64_t entries, int64_t share) {
    int parts = 1;
    while (parts < kLongParts && 2 * parts * share <= entries) parts *= 2;
    return parts;
}

template <int VT>
struct LongChunk {
    using A = typename vt<VT>::vec_t;
    static constexpr int kAhead = 32 / static_cast<int>(sizeof(A));  // chain's LDS reads
    static constexpr int kPad = 16 / static_cast<int>(sizeof(A));    // between lanes' runs
    static constexpr int kStore = kLongTile + kWave * kPad + kAhead;
    static constexpr int64_t kBytes = 2 * static_cast<int64_t>(sizeof(A)) * kStore;
};

// Columns j0 .. j0 + cols of the chunk for the lanes whose rows reach past j0.
struct LongTile {
    int32_t j0, cols, live;  // live: how many lanes
    int32_t shift;           // cols = kLongTile >> shift
    int32_t src, left;       // this thread's lane of the chunk, its row's entries from j0 on
    int32_t row;             // the lane's place among the live ones, as a chain
};

template <int CS>
__device__ __forceinline__ LongTile long_tile(int32_t j0, int32_t len) {
    const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
    uint64_t live = __ballot(len > j0);
    if constexpr (CS < kWave) live &= (1ull << CS) - 1;
    LongTile t;
    t.j0 = j0;
    t.live = __popcll(live);
    t.shift = t.live > 1 ? 32 - __clz(t.live - 1) : 0;
    t.cols = kLongTile >> t.shift;
    t.row = __popcll(live & ((1ull << lane) - 1));
    // lane -> place, the others behind: a permutation of the wavefront
    const int to = (live >> lane) & 1 ? t.row : t.live + lane - t.row;
    const int from = __builtin_amdgcn_ds_permute(to * 4, lane);
    const int s = static_cast<int>(threadIdx.x) & ((1 << t.shift) - 1);
    t.src = __shfl(from, s);
    const int32_t n = __shfl(len, t.src);
    t.left = s < t.live ? n - j0 : 0;
    return t;
}

template <int VT, int CS>
__device__ __forceinline__ typename vt<VT>::vec_t long_chunk(
    typename vt<VT>::vec_t *__restrict__ lds, const int32_t *__restrict__ col,
    const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ x, int64_t base, int32_t len) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using L = LongChunk<VT>;
    constexpr int PER = kLongTile / kScsThreads, U = L::kAhead;
    A *const sv = lds, *const sx = lds + L::kStore;
    const int tid = static_cast<int>(threadIdx.x);
    int32_t c[PER];
    typename T::val_t v[PER];
    A xv[PER];
    const auto at = [&](const LongTile &t, int u) {
        return (tid >> t.shift) + u * (kScsThreads >> t.shift);
    };
    const auto load_columns = [&](const LongTile &t) {
        const int32_t *p = col + base + static_cast<int64_t>(t.j0) * CS + t.src;
#pragma unroll
        for (int u = 0; u < PER; ++u)
            if (at(t, u) < t.left) c[u] = ld_stream(p + at(t, u) * CS);
    };
    const auto gather = [&](const LongTile &t) {
        const typename T::val_t *p = val + base + static_cast<int64_t>(t.j0) * CS + t.src;
#pragma unroll
        for (int u = 0; u < PER; ++u)
            if (at(t, u) < t.left) {
                v[u] = ld_stream(p + at(t, u) * CS);
                xv[u] = x[c[u]];
            }
    };
    A acc = 0;
    LongTile t = long_tile<CS>(0, len);
    load_columns(t);
    gather(t);
    LongTile next = long_tile<CS>(t.j0 + t.cols, len);
    load_columns(next);
    while (t.live > 0) {
        const int run = t.cols + L::kPad;
        const int own = (tid & ((1 << t.shift) - 1)) * run;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const bool in = at(t, u) < t.left;
            sv[own + at(t, u)] = in ? T::widen(v[u]) : A(-0.0);
            sx[own + at(t, u)] = in ? xv[u] : A(0);
        }
        __syncthreads();
        const LongTile now = t;
        t = next;
        if (t.live > 0) {
            gather(t);
            next = long_tile<CS>(t.j0 + t.cols, len);
            load_columns(next);
        }
        if (tid < CS && len > now.j0) {
            const A *pv = sv + now.row * run, *px = sx + now.row * run;
            const int m = len - now.j0 < now.cols ? len - now.j0 : now.cols;
            A w0[U], b0[U], w1[U], b1[U];
            load_run<A, U>(pv, w0);
            load_run<A, U>(px, b0);
            // Up to 2U - 1 entries past the row's end are -0 * 0; the last
            // pass reads U entries more.
            for (int j = 0; j < m; j += 2 * U) {
                load_run<A, U>(pv + j + U, w1);
                load_run<A, U>(px + j + U, b1);
                __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the fmas
#pragma unroll
                for (int u = 0; u < U; ++u) acc = T::fma_(w0[u], b0[u], acc);
                load_run<A, U>(pv + j + 2 * U, w0);
                load_run<A, U>(px + j + 2 * U, b0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < U; ++u) acc = T::fma_(w1[u], b1[u], acc);
            }
        }
        __syncthreads();
    }
    return acc;
}

// The launch's long chunks (see smax_hip_scs_sched), or with tails its long
// tail waves (smax_hip_scs_tails).
struct LongChunks {
    const int32_t *list;  // kLongParts * chunk + part, -1: none
    int64_t blocks;
    int32_t from;   // chunks of this length and more, tail waves before this one
    int32_t share;  // entries that a part has at least
};

// This workgroup's part of a long chunk of CS lanes: true if there is one and
// the thread's lane of it is among them; `len` is then its row's length, 0 on
// the other lanes.  Every thread of the workgroup comes here.
template <int CS>
__device__ __forceinline__ bool long_part(int32_t part, int32_t share, int32_t &len, bool &any) {
    const int lane = static_cast<int>(threadIdx.x) & (CS - 1);
    int64_t entries = len;
#pragma unroll
    for (int d = 1; d < CS; d *= 2) entries += __shfl_xor(entries, d);
    const int parts = long_parts(entries, share);
    any = part < parts;
    const bool mine = any && lane * parts / CS == part;
    if (!mine) len = 0;
    return mine;
}

// What the SpMV kernels take, in one or two arguments: a launch costs the host
// time for every argument it copies (small matrices back to back: 3.95 us a
// product with 17 arguments, 3.70 with these).
template <int VT>
struct ScsSpmv {
    int64_t n_chunks, n_rows;
    const int32_t *chunk_ptr, *chunk_len, *slot_len, *order, *col;
    const typename vt<VT>::val_t *val;
    const int32_t *slot_row;
    const typename vt<VT>::vec_t *x;
    typename vt<VT>::vec_t *y;
};

// Tail waves (t_slot null: none) and long chunks; layouts of short chunks
// have neither.
template <int VT, bool SHORT>
struct ScsParts {
    const int32_t *t_head, *t_slot;
    const int64_t *t_ptr;
    const int32_t *t_col;
    const typename vt<VT>::val_t *t_val;
    int64_t t_blocks;
    LongChunks longs;
};
template <int VT>
struct ScsParts<VT, true> {
    static constexpr const int32_t *t_head = nullptr, *t_slot = nullptr, *t_col = nullptr;
    static constexpr const int64_t *t_ptr = nullptr;
    static constexpr const typename vt<VT>::val_t *t_val = nullptr;
    static constexpr int64_t t_blocks = 0;
};

// C == 64: one wavefront per chunk, one lane per slot.
//   REMAP: XCD-contiguous workgroup order (see xcd_block).
//   order: optional execution order, wave position -> chunk (-1: idle).
//   LEN:   each lane stops at its row's last stored element (slot_len); a
//          lane with padding then applies the reference's padding term
//          fma(0, x[0], acc) once, which equals applying it any number of
//          times (f(a) = fma(0, x0, a) satisfies f(f(a)) = f(a) for every a,
//          signed zeros and non-finite x0 included), so results stay
//          bit-identical to the full-chunk chain.
//   SHORT: every chunk is at most kShortChain long (single-group chains;
//          no tail waves).
//   tails (LEN only; t_slot null: none): the first t_blocks workgroups run
//          the handle's tail waves (smax_hip_scs_tails), the rest the chunks,
//          whose lanes longer than t_head[chunk] then leave at once.  Both
//          kinds of wave run the same chain code on their own arrays;
//          t_blocks is a multiple of 8, so the chunks' workgroups keep their
//          XCD alignment.
//   LONG (LEN only): the first longs.blocks workgroups (again a multiple of
//          8) run the long chunks or, with tails, the long tail waves; the
//          wavefronts leave those out.
//   FOUR: held to 128 registers, 4 wavefronts per SIMD.  FP64 takes 136 by
//   itself, which leaves three, 768 workgroups on the chip: larger grids then
//   run in two rounds (the 27-point stencil of 64^3, 1024 workgroups, 44 -> 30
//   us, SELL-64-64 of 4,000,000 rows 1.16 -> 1.08 ms), smaller ones are slower
//   held to 128 (24^3 13.1 -> 13.7 us).
template <int VT, bool UNPERM, bool REMAP, bool LEN, bool SHORT, bool LONG, bool FOUR>
__global__ __launch_bounds__(kScsThreads, FOUR ? 4 : 1) void scs_spmv_w64(
    ScsSpmv<VT> a, ScsParts<VT, SHORT> p) {
    using T = vt<VT>;
    // All of a short layout's arguments at once: fetched as they come up, the
    // later ones each add a wait (the 512^2 Laplacian, FP64: 4.37 us, not 4.57).
    if constexpr (SHORT)
        asm volatile("" ::"s"(a.x), "s"(a.y), "s"(a.slot_row), "s"(a.col), "s"(a.val),
                     "s"(a.order), "s"(a.chunk_ptr), "s"(a.chunk_len), "s"(a.slot_len));
    const int lane = threadIdx.x & (kWave - 1);
    if constexpr (LONG) {
        if (static_cast<int64_t>(blockIdx.x) < p.longs.blocks) {
            extern __shared__ __align__(16) char long_lds[];
            const int32_t id = p.longs.list[blockIdx.x];
            if (id < 0) return;
            const int64_t at = id / kLongParts;
            const bool tail = p.t_slot != nullptr;
            const int64_t slot = tail ? p.t_slot[at * kWave + lane] : at * kWave + lane;
            const int32_t full = slot >= 0 ? a.slot_len[slot] : 0;
            int32_t len = full;
            bool any;
            const bool mine = long_part<kWave>(id % kLongParts, p.longs.share, len, any);
            if (!any) return;
            typename T::vec_t acc = long_chunk<VT, kWave>(
                reinterpret_cast<typename T::vec_t *>(long_lds), tail ? p.t_col : a.col,
                tail ? p.t_val : a.val, a.x, tail ? p.t_ptr[at] : a.chunk_ptr[at], len);
            if (!mine || slot < 0 || threadIdx.x >= kWave) return;
            if (full < a.chunk_len[slot / kWave])
                acc = T::fma_(T::widen(typename T::val_t(0)), a.x[0], acc);
            if (!UNPERM) {
                a.y[slot] = acc;
            } else if (a.slot_row[slot] < a.n_rows) {
                a.y[a.slot_row[slot]] = acc;
            }
            return;
        }
    }
    const bool tails = !SHORT && LEN && p.t_slot != nullptr;
    int64_t block = blockIdx.x, blocks = gridDim.x, from = 0;
    if constexpr (LONG) {
        block -= p.longs.blocks;
        blocks -= p.longs.blocks;
        from = p.longs.from;
    }
    int64_t slot, base;
    int clen, len;
    const int32_t *cp;
    const typename T::val_t *vp;
    if (tails && block < p.t_blocks) {
        const int64_t w = block * (kScsThreads / kWave) + threadIdx.x / kWave;
        if (LONG && w < from) return;
        const int32_t ts = p.t_slot[w * kWave + lane];
        if (ts < 0) return;
        slot = ts;
        base = p.t_ptr[w] + lane;
        clen = a.chunk_len[ts / kWave];
        len = a.slot_len[ts];
        cp = p.t_col;
        vp = p.t_val;
    } else {
        const int64_t hb = tails ? block - p.t_blocks : block;
        const int64_t hn = tails ? blocks - p.t_blocks : blocks;
        const int64_t blk = REMAP ? xcd_block(hb, hn) : hb;
        const int64_t pos = blk * (kScsThreads / kWave) + (threadIdx.x / kWave);
        const int64_t chunk = a.order ? static_cast<int64_t>(a.order[pos]) : pos;
        if (chunk < 0 || chunk >= a.n_chunks) return;
        slot = chunk * kWave + lane;
        base = static_cast<int64_t>(a.chunk_ptr[chunk]) + lane;
        clen = a.chunk_len[chunk];
        if (LONG && !tails && clen >= from) return;
        len = LEN ? a.slot_len[slot] : clen;
        if (tails && len > p.t_head[chunk]) return;
        cp = a.col;
        vp = a.val;
    }
    typename T::vec_t acc = 0;
    if constexpr (SHORT) {
        acc = slot_chain_short<VT>(cp, vp, a.x, base, len);
    } else {
        acc = slot_chain_pipe<VT, kScsPipeUnroll<VT>>(cp, vp, a.x, base, kWave, len);
    }
    if (LEN && len < clen) acc = T::fma_(T::widen(typename T::val_t(0)), a.x[0], acc);
    if (UNPERM) {
        const int32_t r = a.slot_row[slot];
        if (r < a.n_rows) a.y[r] = acc;
    } else {
        a.y[slot] = acc;
    }
}

// Any C: one lane per slot, 256 / C chunks per workgroup (C <= 256) or one
// chunk over several workgroups; chunks in the optional execution `order`;
// LEN and the tail waves (C <= 256 only; their arrays are a SELL-64 whatever
// C is) as in scs_spmv_w64.
//   CS > 0: C fixed at compile time (layouts without tail waves): the chain
//   then addresses its elements with constant offsets and runs the C = 64
//   kernel's group size (4M-row band matrix, C = 32, FP64: sigma = 65536
//   0.692 -> 0.660 ms, 0.640 with the occupancy cap; sigma = N 1.093 ->
//   1.061 ms; BF16 values, sigma = 65536: 0.495 -> 0.477 ms).  FP64 is held to
//   128 registers as above except in this form without long chunks (27-point
//   stencil of 24^3 14.5 us held, 13.9 not, of 128^3 225 and 222).
template <int VT, bool UNPERM, bool LEN, bool REMAP, int CS, bool LONG>
__global__ __launch_bounds__(kScsThreads, VT == SMAX_HIP_F64 && (LONG || CS == 0) ? 4 : 1) void scs_spmv_generic(
    int64_t C, int64_t cpb, int64_t bpc, ScsSpmv<VT> a, ScsParts<VT, false> p) {
    using T = vt<VT>;
    if constexpr (CS > 0) C = CS;
    if constexpr (LONG) {
        if (static_cast<int64_t>(blockIdx.x) < p.longs.blocks) {
            extern __shared__ __align__(16) char long_lds[];
            // C = 32 chunks, or tail waves of any C
            constexpr int LC = CS > 0 ? CS : kWave;
            const int32_t id = p.longs.list[blockIdx.x];
            if (id < 0) return;
            const int64_t at = id / kLongParts;
            const int lane = static_cast<int>(threadIdx.x) % LC;
            const int64_t slot = CS == 0 ? p.t_slot[at * LC + lane] : at * LC + lane;
            const int32_t full = slot >= 0 ? a.slot_len[slot] : 0;
            int32_t len = full;
            bool any;
            const bool mine = long_part<LC>(id % kLongParts, p.longs.share, len, any);
            if (!any) return;
            typename T::vec_t acc = long_chunk<VT, LC>(
                reinterpret_cast<typename T::vec_t *>(long_lds), CS == 0 ? p.t_col : a.col,
                CS == 0 ? p.t_val : a.val, a.x, CS == 0 ? p.t_ptr[at] : a.chunk_ptr[at], len);
            if (!mine || slot < 0 || static_cast<int>(threadIdx.x) >= LC) return;
            if (full < a.chunk_len[slot / C])
                acc = T::fma_(T::widen(typename T::val_t(0)), a.x[0], acc);
            if (!UNPERM) {
                a.y[slot] = acc;
            } else if (a.slot_row[slot] < a.n_rows) {
                a.y[a.slot_row[slot]] = acc;
            }
            return;
        }
    }
    const bool tails = CS == 0 && LEN && p.t_slot != nullptr;
    int64_t slot, base, stride;
    int clen, len;
    const int32_t *cp;
    const typename T::val_t *vp;
    const int64_t block = LONG ? blockIdx.x - p.longs.blocks : blockIdx.x;
    const int64_t blocks = LONG ? gridDim.x - p.longs.blocks : gridDim.x;
    if (tails && block < p.t_blocks) {
        const int lane = threadIdx.x & (kWave - 1);
        const int64_t w = block * (kScsThreads / kWave) + threadIdx.x / kWave;
        if (LONG && w < p.longs.from) return;
        const int32_t ts = p.t_slot[w * kWave + lane];
        if (ts < 0) return;
        slot = ts;
        base = p.t_ptr[w] + lane;
        stride = kWave;
        clen = a.chunk_len[ts / C];
        len = a.slot_len[ts];
        cp = p.t_col;
        vp = p.t_val;
    } else {
        int64_t pos, i;
        if (cpb > 0) {
            const int64_t hb = tails ? block - p.t_blocks : block;
            const int64_t hn = tails ? blocks - p.t_blocks : blocks;
            const int64_t blk = REMAP ? xcd_block(hb, hn) : hb;
            pos = blk * cpb + threadIdx.x / C;
            i = threadIdx.x % C;
            if (threadIdx.x >= cpb * C) return;
        } else {
            pos = blockIdx.x / bpc;
            i = (blockIdx.x % bpc) * kScsThreads + threadIdx.x;
            if (i >= C) return;
        }
        if (pos >= a.n_chunks) return;
        const int64_t chunk = a.order ? static_cast<int64_t>(a.order[pos]) : pos;
        if (chunk < 0) return;
        slot = chunk * C + i;
        base = static_cast<int64_t>(a.chunk_ptr[chunk]) + i;
        stride = C;
        clen = a.chunk_len[chunk];
        if (LONG && !tails && clen >= p.longs.from) return;
        len = LEN ? a.slot_len[slot] : clen;
        if (tails && len > p.t_head[chunk]) return;
        cp = a.col;
        vp = a.val;
    }
    typename T::vec_t acc;
    if constexpr (CS > 0)
        acc = slot_chain_pipe<VT, kScsPipeUnroll<VT>>(cp, vp, a.x, base, CS, len);
    else
        acc = slot_chain_pipe<VT, kScsUnroll>(cp, vp, a.x, base, stride, len);
    if (LEN && len < clen) acc = T::fma_(T::widen(typename T::val_t(0)), a.x[0], acc);
    if (UNPERM) {
        const int32_t r = a.slot_row[slot];
        if (r < a.n_rows) a.y[r] = acc;
    } else {
        a.y[slot] = acc;
    }
}

// The i-th long slot of a handle: the whole-workgroup ones are listed from
// the front, the others from the back.
struct ListedSlot {
    const int32_t *__restrict__ list;
    int64_t cap, whole;
    int64_t C;
    const int32_t *__restrict__ chunk_ptr, *__restrict__ slot_len, *__restrict__ slot_row;
    __device__ __forceinline__ LongRowAt operator()(int64_t i) const {
        const int64_t s = list[i < whole ? i : cap - 1 - (i - whole)];
        const int64_t c = s / C;
        return {slot_len[s], static_cast<int64_t>(chunk_ptr[c]) + (s - c * C), slot_row[s]};
    }
};

// Long slots that are neighbours, whose columns and values share lines, on one
// XCD: 1,000,000 rows, k = 32: 0.367 -> 0.359 ms, 200,003: 0.087 -> 0.082.
__device__ __forceinline__ int64_t long_block(const LongRows &r, int64_t b) {
    return b < r.whole ? xcd_block(b, r.whole)
                       : r.whole + xcd_block(b - r.whole, r.blocks() - r.whole);
}

// What the two SpMM kernels take.  The launch's first longs.blocks()
// workgroups run the long slots, the others `per` slots each, in the execution
// order of their chunks, `lanes` threads a slot (or one slot in `parts`).
struct ScsSpmmArgs {
    int64_t C, n_slots, n_rows, k, lanes, per, parts;
    FastDiv by_lanes, by_c;
    LongRows longs;
    int32_t long_from;        // slots of this length and more are long (LONG)
    const int32_t *long_list;
    int64_t long_cap;
    const int32_t *chunk_ptr, *chunk_len, *slot_len, *order, *col, *slot_row;

    __device__ __forceinline__ ListedSlot listed() const {
        return {long_list, long_cap, longs.whole, C, chunk_ptr, slot_len, slot_row};
    }
    // This thread's chunk, slot of the chunk and lane of the slot; false: none.
    __device__ __forceinline__ bool place(int64_t block, int64_t &chunk, int64_t &i,
                                          int64_t &l) const {
        int64_t at;
        if (per > 0) {
            const int32_t t = by_lanes(static_cast<int32_t>(threadIdx.x));
            if (t >= per) return false;
            at = block * per + t;
            l = static_cast<int64_t>(threadIdx.x) - t * lanes;
        } else {
            at = block / parts;
            l = (block - at * parts) * kScsThreads + threadIdx.x;
        }
        if (at >= n_slots || l >= lanes) return false;
        const int32_t pos = by_c(static_cast<int32_t>(at));
        chunk = order ? static_cast<int64_t>(order[pos]) : pos;
        i = at - pos * C;
        return true;
    }
};

// SpMM, X and Y row-major with any k columns, in the lanes and runs of
// crs_spmm_run; Y in original row order.  LEN: each slot stops at its row's
// length and no padding term is applied, so Y equals the CRS SpMM bit for
// bit; without it the chain runs over the padded chunk (padding adds
// 0 * X[0, v]).  LONG (with LEN): long slots run in workgroups and wavefronts
// of their own, in runs of LQ columns.  One column per lane, four bytes an
// access, and no such path took 128 us for 40,013 rows, k = 20, BF16 values.
template <int VT, bool LEN, int Q, int LQ, bool LONG>
__global__ __launch_bounds__(kScsThreads) void scs_spmm_run(
    ScsSpmmArgs a, const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ X, typename vt<VT>::vec_t *__restrict__ Y) {
    using A = typename vt<VT>::vec_t;
    if constexpr (LONG) {
        if (blockIdx.x < a.longs.blocks()) {
            long_rows<VT, LQ>(a.longs, long_block(a.longs, blockIdx.x), a.listed(), a.C, a.col,
                             val, a.k, X, a.k, Y, a.k);
            return;
        }
    }
    int64_t chunk, i, l;
    if (!a.place(blockIdx.x - (LONG ? a.longs.blocks() : 0), chunk, i, l)) return;
    const int64_t slot = chunk * a.C + i;
    const int32_t r = a.slot_row[slot];
    if (r >= a.n_rows) return;
    const int len = LEN ? a.slot_len[slot] : a.chunk_len[chunk];
    if (LONG && len >= a.long_from) return;
    const int64_t v = run_start<Q>(l, a.k);
    A acc[Q];
    run_chain<VT, Q, VT == SMAX_HIP_F32>(static_cast<int64_t>(a.chunk_ptr[chunk]) + i, a.C, len, a.col, val, X + v,
                     a.k, acc);
    store_cols_run<A, Q>(Y + static_cast<int64_t>(r) * a.k + v, acc);
}

// As scs_spmm_run for k = K a power of two with 16-byte aligned X and Y:
// a lane owns Q = 16 / sizeof(vec) consecutive columns v (K / Q lanes per
// slot), reads its part of each X row with one 16-byte load and keeps Q fma
// chains, each the same sequential chain as in scs_spmm_run.
template <int VT, bool LEN, int K, bool LONG>
__global__ __launch_bounds__(kScsThreads) void scs_spmm_vec(
    ScsSpmmArgs a, const typename vt<VT>::val_t *__restrict__ val,
    const typename vt<VT>::vec_t *__restrict__ X, typename vt<VT>::vec_t *__restrict__ Y) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    using V = typename T::val_t;
    constexpr int Q = 16 / sizeof(A);
    constexpr int GL = K / Q;
    constexpr int U = 8;
    static_assert(GL * Q == K, "K must be a multiple of the run length");
    if constexpr (LONG) {
        if (blockIdx.x < a.longs.blocks()) {
            long_rows<VT, Q>(a.longs, long_block(a.longs, blockIdx.x), a.listed(), a.C, a.col,
                             val, K, X, K, Y, K);
            return;
        }
    }
    int64_t chunk, i, l64;
    if (!a.place(blockIdx.x - (LONG ? a.longs.blocks() : 0), chunk, i, l64)) return;
    const int l = static_cast<int>(l64);
    const int64_t C = a.C;
    const int64_t slot = chunk * C + i;
    const int32_t r = a.slot_row[slot];
    if (r >= a.n_rows) return;
    const int64_t base = static_cast<int64_t>(a.chunk_ptr[chunk]) + i;
    const int len = LEN ? a.slot_len[slot] : a.chunk_len[chunk];
    if (LONG && len >= a.long_from) return;
    const int32_t *__restrict__ col = a.col;
    A acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] = 0;
    int j = 0;
    if constexpr ((GL == U || GL == 2 * U) && sizeof(V) <= 4) {
        // K / Q = 8 or 16 lanes per slot (k = 32 or 64 with 4-byte X
        // entries): every lane would load the same column index and value of
        // each element, a third of the bytes the slot requests.  Instead lane
        // l loads element l % 8 of each group of 8 and a swizzle within the 8
        // lanes (a DPP row broadcast within the 16) hands every lane all of
        // them; the next group's are requested before this group's X rows
        // (lomax band N = 1M, k = 32: FP32 values 0.378 -> 0.371 ms, A^T
        // 0.213 -> 0.200 ms; BF16 values 0.389 -> 0.372 ms).
        if (len >= U) {
            const int le = l % U;  // the element of each group this lane loads
            int cm = col[base + static_cast<int64_t>(le) * C];
            int wm = val_bits<V>(val[base + static_cast<int64_t>(le) * C]);
            for (;;) {
                const bool more = j + 2 * U <= len;
                int cn = 0, wn = 0;
                if (more) {
                    const int64_t o = base + static_cast<int64_t>(j + U + le) * C;
                    cn = col[o];
                    wn = val_bits<V>(val[o]);
                }
                int cs[U], ws[U];
                if constexpr (GL == U)
                    grp8_bcast8(cm, wm, cs, ws, std::make_integer_sequence<int, U>{});
                else
                    row16_bcast8(cm, wm, cs, ws, std::make_integer_sequence<int, U>{});
                A xv[U][Q];
#pragma unroll
                for (int u = 0; u < U; ++u)
                    load_run<A, Q>(X + static_cast<int64_t>(cs[u]) * K + l * Q, xv[u]);
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
    } else if (len >= U) {
        int32_t c0[U];
        V w0[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c0[u] = col[base + u * C];
            w0[u] = val[base + u * C];
        }
        for (;;) {
            const bool more = j + 2 * U <= len;
            int32_t c1[U];
            V w1[U];
            if (more) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    c1[u] = col[base + static_cast<int64_t>(j + U + u) * C];
                    w1[u] = val[base + static_cast<int64_t>(j + U + u) * C];
                }
            }
            A xv[U][Q];
#pragma unroll
            for (int u = 0; u < U; ++u)
                load_run<A, Q>(X + static_cast<int64_t>(c0[u]) * K + l * Q, xv[u]);
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
    for (; j < len; ++j) {
        const int64_t o = base + static_cast<int64_t>(j) * C;
        A xv[Q];
        load_run<A, Q>(X + static_cast<int64_t>(col[o]) * K + l * Q, xv);
        const A w = T::widen(val[o]);
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[q] = T::fma_(w, xv[q], acc[q]);
    }
    store_run<A, Q>(Y + static_cast<int64_t>(r) * K + l * Q, acc);
}

template <int VT, int K>
static void launch_scs_spmm_vec(smax_hip_ctx ctx, const ScsSpmmArgs &a, dim3 grid,
                                const typename vt<VT>::val_t *val,
                                const typename vt<VT>::vec_t *X, typename vt<VT>::vec_t *Y) {
#define SMAX_SCS_VEC(LEN, LONG)                                                               \
    hipLaunchKernelGGL((scs_spmm_vec<VT, LEN, K, LONG>), grid, dim3(kScsThreads), 0, ctx->stream, \
                       a, val, X, Y)
    if (a.longs.count > 0) SMAX_SCS_VEC(true, true);
    else if (a.slot_len) SMAX_SCS_VEC(true, false);
    else SMAX_SCS_VEC(false, false);
#undef SMAX_SCS_VEC
}

template <int VT, int Q, int LQ>
static void launch_scs_spmm_run(smax_hip_ctx ctx, const ScsSpmmArgs &a, dim3 grid,
                                const typename vt<VT>::val_t *val,
                                const typename vt<VT>::vec_t *X, typename vt<VT>::vec_t *Y) {
#define SMAX_SCS_RUN(LEN, LONG)                                                               \
    hipLaunchKernelGGL((scs_spmm_run<VT, LEN, Q, LONG ? LQ : Q, LONG>), grid, dim3(kScsThreads), 0, ctx->stream, \
                       a, val, X, Y)
    if (a.longs.count > 0) SMAX_SCS_RUN(true, true);
    else if (a.slot_len) SMAX_SCS_RUN(true, false);
    else SMAX_SCS_RUN(false, false);
#undef SMAX_SCS_RUN
}

// longs: the handle's long slots (nullptr: none; needs slot_len).
template <int VT>
static int launch_scs_spmm(smax_hip_ctx ctx, int64_t C, int64_t n_chunks, int64_t n_rows,
                           int64_t k, const int32_t *chunk_ptr, const int32_t *chunk_len,
                           const int32_t *slot_len, const int32_t *order,
                           const int32_t *col, const void *val, const int32_t *slot_row,
                           const void *X, void *Y, const smax_hip_scs_longs *longs = nullptr) {
    using T = vt<VT>;
    using A = typename T::vec_t;
    constexpr int64_t Q = 16 / sizeof(A);
    // k a power of two in [4Q, 64] with 16-byte aligned operands: Q columns
    // per lane, at least 4 lanes per slot
    const bool vec = k >= 4 * Q && k <= 64 && (k & (k - 1)) == 0 && aligned16(X, Y);
    // Columns per lane: 16 bytes where that leaves three lanes a slot or more.
    // A wavefront lasts as long as its longest slot, and with one or two lanes
    // a slot it holds many (1,000,000 rows, SELL-64-4096, FP32, k = 4: 292 us
    // with four columns a lane, 228 with two, 207 with one; k = 8: 266 and 257,
    // k = 12: 346 and 407; FP64, k = 4: 301 and 287 with one).
    const int64_t q = vec || k >= 3 * Q ? Q : k > 4 ? 2 : 1;
    const int64_t lanes = run_lanes(k, q);
    ScsSpmmArgs a{};
    a.C = C;
    a.n_slots = n_chunks * C;
    a.n_rows = n_rows;
    a.k = k;
    a.lanes = lanes;
    a.per = kScsThreads / lanes;
    // Slots are sorted in windows of a power of two; 42, 18 or 14 of them a
    // workgroup fall in step with those, one less does not (600,000 rows,
    // SELL-64-4096, k = 24, FP32, 42 slots 362 us, 41: 263; FP64, k = 28, 18
    // and 17: 503 and 465; SELL-64-65536: 240 and 239).
    if (a.per % 4 == 2 && a.per > 2) --a.per;
    a.parts = a.per > 0 ? 1 : ceil_div(lanes, kScsThreads);
    a.by_lanes = fast_div(a.per > 0 ? lanes : 1);
    a.by_c = fast_div(C);
    if (longs && slot_len) {
        a.longs = longs->rows;
        a.long_from = longs->from;
        a.long_list = longs->list;
        a.long_cap = longs->cap;
    }
    a.chunk_ptr = chunk_ptr;
    a.chunk_len = chunk_len;
    a.slot_len = slot_len;
    a.order = order;
    a.col = col;
    a.slot_row = slot_row;
    const int64_t blocks =
        a.longs.blocks() + (a.per > 0 ? ceil_div(a.n_slots, a.per) : a.n_slots * a.parts);
    SMAX_HIP_REQUIRE(ctx, blocks <= INT32_MAX, "scs spmm: grid too large");
    const dim3 grid(static_cast<unsigned>(blocks));
    auto v = static_cast<const typename T::val_t *>(val);
    auto xv = static_cast<const typename T::vec_t *>(X);
    auto yv = static_cast<typename T::vec_t *>(Y);
    if (vec) {
        switch (k) {
#define SMAX_SCS_SPMM_VEC(KK)                                                                \
    case KK:                                                                                  \
        if constexpr (KK >= 4 * Q) launch_scs_spmm_vec<VT, KK>(ctx, a, grid, v, xv, yv);      \
        break;
            SMAX_SCS_SPMM_VEC(8)
            SMAX_SCS_SPMM_VEC(16)
            SMAX_SCS_SPMM_VEC(32)
            SMAX_SCS_SPMM_VEC(64)
#undef SMAX_SCS_SPMM_VEC
        }
        SMAX_HIP_LAUNCHED(ctx, "scs_spmm_vec");
        return SMAX_HIP_SUCCESS;
    }
    if (q == Q) launch_scs_spmm_run<VT, Q, Q>(ctx, a, grid, v, xv, yv);
    else if (q == 2) launch_scs_spmm_run<VT, 2, Q>(ctx, a, grid, v, xv, yv);
    else if (k >= Q) launch_scs_spmm_run<VT, 1, Q>(ctx, a, grid, v, xv, yv);
    else if (k >= 2) launch_scs_spmm_run<VT, 1, 2>(ctx, a, grid, v, xv, yv);
    else launch_scs_spmm_run<VT, 1, 1>(ctx, a, grid, v, xv, yv);
    SMAX_HIP_LAUNCHED(ctx, "scs_spmm_run");
    return SMAX_HIP_SUCCESS;
}

template <int VT>
struct ScsLaunch {
    unsigned lds_bytes;  // dynamic LDS per workgroup (long chunks, occupancy cap)
    ScsSpmv<VT> a;
    ScsParts<VT, false> p;
};

template <int VT, bool UNPERM, bool REMAP, bool LEN, bool SHORT, bool LONG>
static void launch_w64(smax_hip_ctx ctx, const ScsLaunch<VT> &l) {
    const int64_t blocks =
        ceil_div(l.a.n_chunks, kScsThreads / kWave) + l.p.t_blocks + l.p.longs.blocks;
    const dim3 grid(static_cast<unsigned>(blocks));
    constexpr bool kFour = VT == SMAX_HIP_F64;
    constexpr int64_t kCus = 256;
    if constexpr (SHORT) {
        hipLaunchKernelGGL((scs_spmv_w64<VT, UNPERM, REMAP, LEN, true, false, false>), grid,
                           dim3(kScsThreads), l.lds_bytes, ctx->stream, l.a,
                           ScsParts<VT, true>{});
    } else if (kFour && !LONG && blocks <= 3 * kCus) {
        hipLaunchKernelGGL((scs_spmv_w64<VT, UNPERM, REMAP, LEN, false, false, false>), grid,
                           dim3(kScsThreads), l.lds_bytes, ctx->stream, l.a, l.p);
    } else {
        hipLaunchKernelGGL((scs_spmv_w64<VT, UNPERM, REMAP, LEN, false, LONG, kFour>), grid,
                           dim3(kScsThreads), l.lds_bytes, ctx->stream, l.a, l.p);
    }
}

template <int VT, bool UNPERM, bool SHORT>
static void launch_w64_len(smax_hip_ctx ctx, bool remap, const ScsLaunch<VT> &l) {
    const bool len = l.a.slot_len != nullptr;
    if constexpr (!SHORT) {
        if (l.p.longs.blocks > 0) {
            if (remap)
                launch_w64<VT, UNPERM, true, true, false, true>(ctx, l);
            else
                launch_w64<VT, UNPERM, false, true, false, true>(ctx, l);
            return;
        }
    }
    if (remap && len)
        launch_w64<VT, UNPERM, true, true, SHORT, false>(ctx, l);
    else if (remap)
        launch_w64<VT, UNPERM, true, false, SHORT, false>(ctx, l);
    else if (len)
        launch_w64<VT, UNPERM, false, true, SHORT, false>(ctx, l);
    else
        launch_w64<VT, UNPERM, false, false, SHORT, false>(ctx, l);
}

// remap: XCD-contiguous order (right when sigma-windows keep rows local);
// slot_len: optional per-slot lengths (nullptr: full chunk chains);
// sched: the layout's schedule (nullptr: chunk order);
// tails: the handle's tail waves (C = 64 with slot_len; nullptr: none).
template <int VT>
int launch_scs_spmv(smax_hip_ctx ctx, int64_t C, int64_t n_chunks,
                    int64_t n_rows, const int32_t *chunk_ptr,
                    const int32_t *chunk_len, const int32_t *col,
                    const void *val, const int32_t *slot_row, const void *x,
                    void *y, bool unperm, const smax_hip_scs_sched *sched = nullptr,
                    const int32_t *slot_len = nullptr,
                    const smax_hip_scs_tails *tails = nullptr) {
    const bool remap = sched ? sched->remap : true;
    ScsLaunch<VT> l{};
    l.a = {n_chunks, n_rows, chunk_ptr, chunk_len, slot_len,
           !sched ? nullptr : C <= kScsThreads ? sched->order : sched->order_lf, col,
           static_cast<const typename vt<VT>::val_t *>(val), slot_row,
           static_cast<const typename vt<VT>::vec_t *>(x),
           static_cast<typename vt<VT>::vec_t *>(y)};
    l.lds_bytes = sched ? static_cast<unsigned>(sched->lds_cap_bytes) : 0u;
    const bool has_tails = slot_len && C <= kScsThreads && tails && tails->n_blocks > 0;
    if (has_tails) {
        l.p.t_head = tails->head;
        l.p.t_slot = tails->slot;
        l.p.t_ptr = tails->ptr;
        l.p.t_col = tails->col;
        l.p.t_val = static_cast<const typename vt<VT>::val_t *>(tails->val);
        l.p.t_blocks = tails->n_blocks;
        l.p.longs = {tails->wide, tails->wide_blocks, tails->n_wide, tails->share};
    } else if (sched && slot_len && sched->long_blocks > 0) {
        l.p.longs = {sched->long_chunks, sched->long_blocks, sched->long_from,
                     sched->long_share};
    }
    if (l.p.longs.blocks > 0)
        l.lds_bytes = std::max(l.lds_bytes, static_cast<unsigned>(LongChunk<VT>::kBytes));
    if (C == kWave) {
        // Short chains only without tail waves (a layout with them is padded
        // more than 6x, and its chunks then run their heads only).
        const bool short_chains = sched && !has_tails && sched->max_chunk_len >= 0 &&
                                  sched->max_chunk_len <= kShortChain;
        if (unperm && short_chains)
            launch_w64_len<VT, true, true>(ctx, remap, l);
        else if (unperm)
            launch_w64_len<VT, true, false>(ctx, remap, l);
        else if (short_chains)
            launch_w64_len<VT, false, true>(ctx, remap, l);
        else
            launch_w64_len<VT, false, false>(ctx, remap, l);
        SMAX_HIP_LAUNCHED(ctx, "scs_spmv_w64");
        return SMAX_HIP_SUCCESS;
    }
    const int64_t cpb = C <= kScsThreads ? kScsThreads / C : 0;
    const int64_t bpc = C <= kScsThreads ? 1 : ceil_div(C, kScsThreads);
    const int64_t blocks = (cpb > 0 ? ceil_div(n_chunks, cpb) : n_chunks * bpc) +
                           l.p.t_blocks + l.p.longs.blocks;
    SMAX_HIP_REQUIRE(ctx, blocks <= INT32_MAX, "scs spmv: grid too large");
    const dim3 grid(static_cast<unsigned>(blocks));
    const bool rm = remap && cpb > 0;
    // C = 32 without tail waves: the compile-time chunk width, and the
    // schedule's occupancy cap
    const bool c32 = C == 32 && !has_tails;
    const unsigned lds = c32 || l.p.longs.blocks > 0 ? l.lds_bytes : 0u;
#define SMAX_SCS_GENERIC_CS(U, L, R, CS, LONG)                                                \
    hipLaunchKernelGGL((scs_spmv_generic<VT, U, L, R, CS, LONG>), grid, dim3(kScsThreads), lds, \
                       ctx->stream, C, cpb, bpc, l.a, l.p)
#define SMAX_SCS_GENERIC(U, L, R)                                                        \
    if (c32) SMAX_SCS_GENERIC_CS(U, L, R, 32, false); else SMAX_SCS_GENERIC_CS(U, L, R, 0, false)
#define SMAX_SCS_GENERIC_LONG(U, R)                                                      \
    if (c32) SMAX_SCS_GENERIC_CS(U, true, R, 32, true); else SMAX_SCS_GENERIC_CS(U, true, R, 0, true)
    if (l.p.longs.blocks > 0) {
        if (unperm) {
            if (rm) SMAX_SCS_GENERIC_LONG(true, true); else SMAX_SCS_GENERIC_LONG(true, false);
        } else {
            if (rm) SMAX_SCS_GENERIC_LONG(false, true); else SMAX_SCS_GENERIC_LONG(false, false);
        }
    } else if (unperm && slot_len) {
        if (rm) SMAX_SCS_GENERIC(true, true, true); else SMAX_SCS_GENERIC(true, true, false);
    } else if (unperm) {
        if (rm) SMAX_SCS_GENERIC(true, false, true); else SMAX_SCS_GENERIC(true, false, false);
    } else if (slot_len) {
        if (rm) SMAX_SCS_GENERIC(false, true, true); else SMAX_SCS_GENERIC(false, true, false);
    } else {
        if (rm) SMAX_SCS_GENERIC(false, false, true); else SMAX_SCS_GENERIC(false, false, false);
    }
#undef SMAX_SCS_GENERIC
#undef SMAX_SCS_GENERIC_LONG
#undef SMAX_SCS_GENERIC_CS
    SMAX_HIP_LAUNCHED(ctx, "scs_spmv_generic");
    return SMAX_HIP_SUCCESS;
}

// Execution schedule of the C = 64 kernel on a converted matrix.
//
// Block order: windows much shorter than an XCD's share keep rows (and their
// x bands) local, so each XCD gets a contiguous range of chunks (remap).  A
// near-global sort puts the longest chunks first, where a contiguous split
// would leave one XCD with all of them, and runs each length's rows across
// the whole matrix at once (every XCD then gathers from all of x).  When the
// rows of the slots are known (a converted matrix), such layouts run their
// chunks sorted by their first slot's row instead: the XCDs get contiguous
// ranges of that sequence, so each holds one stretch of rows with its share
// of every length, and rows in flight stay local as with short windows.
// Without the rows, the hardware's round-robin order is kept.
//
// Chunk order: one wave runs a chunk's 64 rows; the longest chunks (rows of
// up to thousands of entries) then set the kernel's critical path, and in
// chunk order the last window's long chunks start late.  Within each range
// (each XCD's, or the whole grid) chunks of at least kLongChunk entries per
// slot (and 8x the mean) start first, longest first, one per workgroup where
// the range has room (each on its own CU, with its own miss queue); the rest
// follow in chunk order.  Results do not depend on the order.
//
// Where the slots' lengths are at hand, chunks of at least kWideChunk entries
// per slot (and 4x the mean) leave this order and are run by whole workgroups
// (long_chunk).  With 128 and 8x instead: 1,000,000 rows, C = 32, sigma =
// 65536, FP32 133 us against 127, 4,000,000 rows, C = 32, sigma = 4096, FP64
// 803 against 760.  Against the order alone, 4,000,000 rows, FP32: C = 64, sigma
// = 1024 609 us and 644, C = 32, sigma = 65536 489 and 504, but C = 64, sigma =
// 4096 534 and 528, sigma = 65536 479 and 471 (BF16 458 and 457; 2,000,000 rows
// 227 and 235).
constexpr int kLongChunk = 128;
constexpr int kWideChunk = 64;
constexpr int64_t kLdsPerCu = 160 * 1024;

static int upload_order(smax_hip_ctx ctx, const std::vector<int32_t> &ord, int32_t **out) {
    int rc = dev_alloc(ctx, reinterpret_cast<void **>(out), sizeof(int32_t) * ord.size(),
                       "scs execution order");
    if (rc) return rc;
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(*out, ord.data(), sizeof(int32_t) * ord.size(),
                                      hipMemcpyHostToDevice, ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    return SMAX_HIP_SUCCESS;
}

// Entries per workgroup of a long chunk: enough workgroups for the chip while
// the matrix is small, whole chunks once there are many of them (1 / 2048 of the
// entries: 1,000,000 rows, C = 32, sigma = 65536, FP32 142 us against 127).
static int32_t long_share(int64_t nnz) {
    return static_cast<int32_t>(std::max<int64_t>(2048, nnz / 1024));
}

// Appends the eight lists entry by entry, the i-th of list r at 8i + r, with
// -1 behind the shorter ones; returns the number of entries.
static size_t append_by_xcd(std::vector<int32_t> &out,
                            const std::vector<std::vector<int32_t>> &lists) {
    size_t most = 0;
    for (const auto &l : lists) most = std::max(most, l.size());
    const size_t at = out.size();
    out.resize(at + 8 * most, -1);
    for (size_t r = 0; r < lists.size(); ++r)
        for (size_t i = 0; i < lists[r].size(); ++i) out[at + 8 * i + r] = lists[r][i];
    return 8 * most;
}

void free_schedule(smax_hip_scs_sched &s) {
    dev_free(s.order);
    dev_free(s.order_lf);
    s.order = s.order_lf = nullptr;
    s.long_chunks = nullptr;
    s.long_blocks = 0;
}

// Row of each chunk's first slot, packed for one copy to the host (a strided
// copy of 7,813 such entries took 52 ms).
__global__ void k_first_rows(int64_t n_chunks, int64_t C, const int32_t *__restrict__ slot_row,
                             int32_t *__restrict__ out) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c < n_chunks) out[c] = slot_row[c * C];
}

int build_schedule(smax_hip_ctx ctx, int64_t C, int64_t sigma, int64_t n_rows_padded,
                   int64_t n_chunks, int64_t n_elements, int64_t nnz,
                   const int32_t *chunk_lengths, smax_hip_scs_sched *out,
                   const int32_t *slot_row) {
    *out = smax_hip_scs_sched{};
    const bool local = sigma * 16 <= n_rows_padded;
    const bool by_row = !local && slot_row != nullptr && C <= kScsThreads;
    out->remap = local || by_row;
    // Occupancy: with little padding every lane of a wave has gathers in
    // flight, and five waves per SIMD congest the path from L2 to the MALL;
    // reserving LDS for four workgroups per CU (four waves per SIMD) runs
    // faster (0.70 -> 0.63 ms on the 4M-row Lomax matrix at sigma = 65536;
    // C = 32: 0.660 -> 0.640 ms).  Padded layouts (fill > 1.5) keep lanes
    // idle and want every wave (C = 32, sigma = 4096, fill 1.7: 0.745 ->
    // 0.824 ms with the cap).
    if ((C == kWave || C == 32) && nnz > 0 && 2 * n_elements <= 3 * nnz)
        out->lds_cap_bytes = kLdsPerCu / 4;
    const int64_t n = n_chunks;
    if (n <= 0) return SMAX_HIP_SUCCESS;
    std::vector<int32_t> cl(static_cast<size_t>(n));
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(cl.data(), chunk_lengths, sizeof(int32_t) * n,
                                      hipMemcpyDeviceToHost, ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    out->max_chunk_len = *std::max_element(cl.begin(), cl.end());
    const double mean =
        static_cast<double>(n_elements) / static_cast<double>(n * C);
    const int64_t thr =
        std::max<int64_t>(kLongChunk, static_cast<int64_t>(std::ceil(8 * mean)));
    const int64_t n_long =
        std::count_if(cl.begin(), cl.end(), [&](int32_t l) { return l >= thr; });
    if (n_long == 0 && !by_row) return SMAX_HIP_SUCCESS;
    // by_row: the chunks sorted by the row of their first slot (stable)
    std::vector<int32_t> seq;
    if (by_row) {
        std::vector<int32_t> first(static_cast<size_t>(n));
        int32_t *packed = nullptr;
        int rc = dev_alloc(ctx, reinterpret_cast<void **>(&packed), sizeof(int32_t) * n,
                           "scs execution order");
        if (rc) return rc;
        hipLaunchKernelGGL(k_first_rows, grid_for(n, 256), dim3(256), 0, ctx->stream, n, C,
                           slot_row, packed);
        rc = check_launch(ctx, "k_first_rows");
        if (!rc)
            rc = smax_hip_memcpy_d2h(ctx, first.data(), packed, sizeof(int32_t) * n);
        dev_free(packed);
        if (rc) return rc;
        seq.resize(static_cast<size_t>(n));
        for (int64_t c = 0; c < n; ++c) seq[c] = static_cast<int32_t>(c);
        std::stable_sort(seq.begin(), seq.end(),
                         [&](int32_t p, int32_t q) { return first[p] < first[q]; });
    }
    // positions [a, b) of `ord` receive the chunks at [a, min(b, n)) of the
    // chunk sequence (`sq`, or chunk order when null): long chunks first
    // (longest first) at every `spread`-th position when they fit, then the
    // rest in sequence order
    auto fill = [&](std::vector<int32_t> &ord, int64_t a, int64_t b, int64_t spread,
                    const std::vector<int32_t> *sq) {
        const int64_t e = std::min(b, n);
        if (e <= a) return;
        std::vector<int32_t> lg, rest;
        for (int64_t i = a; i < e; ++i) {
            const int32_t c = sq ? (*sq)[i] : static_cast<int32_t>(i);
            (cl[c] >= thr ? lg : rest).push_back(c);
        }
        std::stable_sort(lg.begin(), lg.end(),
                         [&](int32_t p, int32_t q) { return cl[p] > cl[q]; });
        const int64_t m = static_cast<int64_t>(lg.size());
        const int64_t step = m > 0 && (m - 1) * spread < e - a ? spread : 1;
        std::vector<char> taken(static_cast<size_t>(e - a), 0);
        for (int64_t i = 0; i < m; ++i) {
            ord[a + i * step] = lg[i];
            taken[i * step] = 1;
        }
        int64_t r = 0;
        for (int64_t p = a; p < e; ++p)
            if (!taken[p - a]) ord[p] = rest[r++];
    };
    if (n_long > 0) {
        std::vector<int32_t> lf(static_cast<size_t>(n), -1);
        fill(lf, 0, n, 1, nullptr);
        const int rc = upload_order(ctx, lf, &out->order_lf);
        if (rc) return rc;
    }
    if (C > kScsThreads) return SMAX_HIP_SUCCESS;
    const std::vector<int32_t> *sq = by_row ? &seq : nullptr;
    const int64_t per_block = kScsThreads / C;  // chunks per workgroup
    const int64_t nb = ceil_div(n, per_block);
    std::vector<int32_t> ord(static_cast<size_t>(nb * per_block), -1);
    // The long chunks of each range, longest first.
    std::vector<std::vector<int32_t>> longs;
    const int64_t wide = std::max<int64_t>(kWideChunk, static_cast<int64_t>(std::ceil(4 * mean)));
    auto list_longs = [&](int64_t a, int64_t b) {
        std::vector<int32_t> l;
        for (int64_t i = a; i < std::min(b, n); ++i) {
            const int32_t c = sq ? (*sq)[i] : static_cast<int32_t>(i);
            if (cl[c] >= wide) l.push_back(c);
        }
        std::stable_sort(l.begin(), l.end(),
                         [&](int32_t p, int32_t q) { return cl[p] > cl[q]; });
        longs.push_back(std::move(l));
    };
    if (out->remap) {
        constexpr int64_t kXcd = 8;
        const int64_t q = nb / kXcd, rem = nb % kXcd;
        for (int64_t k = 0; k < kXcd; ++k) {
            const int64_t s = k < rem ? k * (q + 1) : rem * (q + 1) + (k - rem) * q;
            const int64_t len = k < rem ? q + 1 : q;
            fill(ord, s * per_block, (s + len) * per_block, per_block, sq);
            list_longs(s * per_block, (s + len) * per_block);
        }
    } else {
        fill(ord, 0, nb * per_block, per_block, sq);
        list_longs(0, nb * per_block);
    }
    if ((C == kWave || C == 32) && n_long > 0) {
        // one range: dealt out in turn; eight: one range per XCD.  A chunk
        // gets the workgroups that it needs if no lane of it is padded.  First
        // parts come first: they hold the longest rows, and the hardware hands
        // an XCD's workgroups to its CUs in turn (parts of a chunk side by side,
        // 1,000,000 rows, sigma = 4096, FP64: 0.286 ms against 0.168).
        const int32_t share = long_share(nnz);
        std::vector<std::vector<int32_t>> parts(8);
        for (int p = 0; p < kLongParts; ++p)
            for (size_t r = 0; r < longs.size(); ++r)
                for (size_t i = 0; i < longs[r].size(); ++i) {
                    const int32_t c = longs[r][i];
                    if (p < long_parts(C * cl[c], share))
                        parts[longs.size() == 1 ? i % 8 : r].push_back(c * kLongParts + p);
                }
        const size_t at = ord.size();
        const size_t blocks = append_by_xcd(ord, parts);
        const int rc = upload_order(ctx, ord, &out->order);
        if (rc) return rc;
        out->long_chunks = out->order + at;
        out->long_blocks = static_cast<int64_t>(blocks);
        out->long_from = static_cast<int32_t>(std::min<int64_t>(wide, INT32_MAX));
        out->long_share = share;
        return SMAX_HIP_SUCCESS;
    }
    return upload_order(ctx, ord, &out->order);
}

// ------------------------------------------------------------ tail waves
// Layouts whose padding exceeds 5x their stored entries get tail waves (see
// smax_hip_scs_tails).  Measured on the 4M-row band matrix (FP64): SELL-64-1
// 2.32 -> 1.14 ms, SELL-64-64 2.09 -> 1.04 ms, SELL-32-1 2.14 -> 1.17 ms,
// SELL-32-64 1.91 -> 1.05 ms, SELL-128-1 2.20 -> 1.13 ms.  Sorted windows
// leave only the matrix's longest rows skewed: their waves then carry the
// kernel's longest chains together and finish last (SELL-64-4096, fill 2.5:
// 0.76 ms against 0.70; SELL-128-4096, fill 4.0: 0.82 against 0.75).  A
// skewed chunk keeps its slots up to its (C/8)-th longest one (the 8th for
// C = 64: 1.10 ms for SELL-64-1, against 1.23 ms up to the 4th);
// a tail wave takes at most kTailWaveWork elements (32768: 1.10 ms, 16384:
// 1.11 ms, unbounded 1.39 ms).
constexpr int64_t kTailWaveWork = 32768;

// Copies the elements of every tail slot into its wave's arrays: element j of
// the slot (chunk c, lane i) at chunk_ptr[c] + j*C + i goes to
// t_ptr[w] + j*64 + l for its tail-wave lane l of wave w.  One thread per
// tail-wave lane; t_col null: values only.
template <typename E>
__global__ void k_tail_fill(int64_t n_lanes, int64_t C, const int32_t *__restrict__ t_slot,
                            const int64_t *__restrict__ t_ptr,
                            const int32_t *__restrict__ slot_len,
                            const int32_t *__restrict__ chunk_ptr,
                            const int32_t *__restrict__ col, const E *__restrict__ val,
                            int32_t *__restrict__ t_col, E *__restrict__ t_val) {
    const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= n_lanes) return;
    const int32_t ts = t_slot[p];
    if (ts < 0) return;
    const int64_t src = static_cast<int64_t>(chunk_ptr[ts / C]) + ts % C;
    const int64_t dst = t_ptr[p / kWave] + p % kWave;
    const int len = slot_len[ts];
    for (int j = 0; j < len; ++j) {
        const int64_t s = static_cast<int64_t>(j) * C, d = static_cast<int64_t>(j) * kWave;
        if (t_col) t_col[dst + d] = col[src + s];
        t_val[dst + d] = val[src + s];
    }
}

static int tail_fill(smax_hip_ctx ctx, smax_hip_scs A, bool with_col) {
    const smax_hip_scs_info &in = A->info;
    const smax_hip_scs_tails &t = A->tails;
    const int64_t lanes = t.n_blocks * kScsThreads;
    int32_t *tc = with_col ? t.col : nullptr;
#define SMAX_TAIL_FILL(E)                                                                 \
    hipLaunchKernelGGL((k_tail_fill<E>), grid_for(lanes, kScsThreads), dim3(kScsThreads), \
                       0, ctx->stream, lanes, in.C, t.slot, t.ptr, in.slot_len,           \
                       in.chunk_ptr,                                                      \
                       in.col, static_cast<const E *>(in.val), tc, static_cast<E *>(t.val))
    switch (in.val_bytes) {
    case 8: SMAX_TAIL_FILL(uint64_t); break;
    case 4: SMAX_TAIL_FILL(uint32_t); break;
    default: SMAX_TAIL_FILL(uint16_t); break;
    }
#undef SMAX_TAIL_FILL
    SMAX_HIP_LAUNCHED(ctx, "k_tail_fill");
    return SMAX_HIP_SUCCESS;
}

void free_tails(smax_hip_scs_tails &t) {
    dev_free(t.head);
    dev_free(t.slot);
    dev_free(t.ptr);
    dev_free(t.col);
    dev_free(t.val);
    t = smax_hip_scs_tails{};
}

int build_tails(smax_hip_ctx ctx, smax_hip_scs A) {
    const smax_hip_scs_info &in = A->info;
    const int64_t C = in.C;
    if (C < 16 || C > kScsThreads || C % 8 != 0 || in.nnz <= 0 || in.n_elements <= 6 * in.nnz)
        return SMAX_HIP_SUCCESS;
    const int64_t rank = C / 8;
    const int64_t nc = in.n_chunks;
    std::vector<int32_t> sl(static_cast<size_t>(nc * C)), cl(static_cast<size_t>(nc));
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(sl.data(), in.slot_len, sizeof(int32_t) * sl.size(),
                                      hipMemcpyDeviceToHost, ctx->stream));
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(cl.data(), in.chunk_lengths, sizeof(int32_t) * nc,
                                      hipMemcpyDeviceToHost, ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    // per chunk: the head length, and the slots beyond it
    std::vector<int32_t> head(static_cast<size_t>(nc));
    std::vector<std::pair<int32_t, int32_t>> tail;  // (length, slot)
    std::vector<int32_t> lens(static_cast<size_t>(C));
    for (int64_t c = 0; c < nc; ++c) {
        const int32_t *l = sl.data() + c * C;
        std::copy(l, l + C, lens.begin());
        std::nth_element(lens.begin(), lens.begin() + (rank - 1), lens.end(),
                         std::greater<int32_t>());
        const int32_t h = lens[rank - 1];
        head[c] = 2 * static_cast<int64_t>(h) < cl[c] ? h : cl[c];
        for (int64_t i = 0; i < C; ++i)
            if (l[i] > head[c]) tail.emplace_back(l[i], static_cast<int32_t>(c * C + i));
    }
    if (tail.empty()) return SMAX_HIP_SUCCESS;
    // longest first (ties in slot order), packed greedily into waves
    std::sort(tail.begin(), tail.end(), [](const auto &a, const auto &b) {
        return a.first != b.first ? a.first > b.first : a.second < b.second;
    });
    std::vector<int64_t> wave_len;  // each wave's longest slot (its first)
    std::vector<int64_t> pos(tail.size());
    int64_t cnt = kWave, work = 0;
    for (size_t t = 0; t < tail.size(); ++t) {
        const int64_t l = tail[t].first;
        if (cnt == kWave || work + l > kTailWaveWork) {
            wave_len.push_back(l);
            cnt = work = 0;
        }
        pos[t] = static_cast<int64_t>(wave_len.size() - 1) * kWave + cnt;
        ++cnt;
        work += l;
    }
    const int64_t n_waves = static_cast<int64_t>(wave_len.size());
    const int64_t per_block = kScsThreads / kWave;
    const int64_t n_blocks = ceil_div(ceil_div(n_waves, per_block), 8) * 8;
    std::vector<int32_t> tslot(static_cast<size_t>(n_blocks * kScsThreads), -1);
    for (size_t t = 0; t < tail.size(); ++t) tslot[pos[t]] = tail[t].second;
    std::vector<int64_t> tptr(static_cast<size_t>(n_blocks * per_block), 0);
    int64_t store = 0;
    for (int64_t w = 0; w < n_waves; ++w) {
        tptr[w] = store;
        store += wave_len[w] * kWave;
    }
    // The waves of kWideChunk columns and more, by whole workgroups.
    const int32_t share = long_share(in.nnz);
    std::vector<std::vector<int32_t>> parts(8);
    int64_t wide = 0;
    while (wide < n_waves && wave_len[wide] >= kWideChunk) ++wide;
    for (int p = 0; p < kLongParts; ++p)
        for (int64_t w = 0; w < wide; ++w)
            if (p < long_parts(kWave * wave_len[w], share))
                parts[w % 8].push_back(static_cast<int32_t>(w * kLongParts + p));
    const size_t listed = tslot.size();
    const int64_t wide_blocks = static_cast<int64_t>(append_by_xcd(tslot, parts));
    smax_hip_scs_tails t;
    t.n_elements = store;
    t.n_slots = static_cast<int64_t>(tail.size());
    t.n_waves = n_waves;
    int rc = 0;
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&t.head), sizeof(int32_t) * nc, "scs tails");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&t.slot), sizeof(int32_t) * tslot.size(),
                    "scs tails");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&t.ptr), sizeof(int64_t) * tptr.size(),
                    "scs tails");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&t.col), sizeof(int32_t) * store, "scs tails");
    rc |= dev_alloc(ctx, &t.val, static_cast<size_t>(in.val_bytes) * store, "scs tails");
    if (rc) {
        free_tails(t);
        return SMAX_HIP_ERROR_OUT_OF_MEMORY;
    }
    // elements past a lane's length are never read; zero them all the same
    rc = smax_hip_zero(ctx, t.col, sizeof(int32_t) * store);
    if (!rc) rc = smax_hip_zero(ctx, t.val, static_cast<size_t>(in.val_bytes) * store);
    if (rc) {
        free_tails(t);
        return rc;
    }
    const hipError_t e1 = hipMemcpyAsync(t.head, head.data(), sizeof(int32_t) * nc,
                                         hipMemcpyHostToDevice, ctx->stream);
    const hipError_t e2 = hipMemcpyAsync(t.slot, tslot.data(), sizeof(int32_t) * tslot.size(),
                                         hipMemcpyHostToDevice, ctx->stream);
    const hipError_t e3 = hipMemcpyAsync(t.ptr, tptr.data(), sizeof(int64_t) * tptr.size(),
                                         hipMemcpyHostToDevice, ctx->stream);
    const hipError_t e4 = hipStreamSynchronize(ctx->stream);
    for (hipError_t e : {e1, e2, e3, e4})
        if (e != hipSuccess) {
            free_tails(t);
            return hip_fail(ctx, e, "scs tails");
        }
    t.n_blocks = n_blocks;
    t.wide = t.slot + listed;
    t.wide_blocks = wide_blocks;
    t.n_wide = static_cast<int32_t>(wide);
    t.share = share;
    A->tails = t;  // freed with the handle from here on
    rc = tail_fill(ctx, A, true);
    if (rc) return rc;
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    return SMAX_HIP_SUCCESS;
}

int refresh_tail_values(smax_hip_ctx ctx, smax_hip_scs A) {
    return A->tails.n_blocks > 0 ? tail_fill(ctx, A, false) : SMAX_HIP_SUCCESS;
}

static int check_scs_args(smax_hip_ctx ctx, const char *fn, int value_type,
                          int64_t C, int64_t n_chunks, const void *chunk_ptr,
                          const void *chunk_len, const void *col,
                          const void *val, const void *x, const void *y) {
    if (!valid_value_type(value_type))
        return fail(ctx, SMAX_HIP_ERROR_UNSUPPORTED, "%s: value type %d", fn,
                    value_type);
    SMAX_HIP_REQUIRE(ctx, C > 0 && n_chunks > 0, "%s: bad C/n_chunks", fn);
    SMAX_HIP_REQUIRE(ctx, C <= INT32_MAX && n_chunks <= INT32_MAX / C, "%s: too many slots", fn);
    SMAX_HIP_REQUIRE(ctx, chunk_ptr && chunk_len && col && val && x && y,
                     "%s: null pointer", fn);
    return SMAX_HIP_SUCCESS;
}

}  // namespace smaxhip

using namespace smaxhip;

extern "C" {

int smax_hip_scs_spmv(smax_hip_ctx ctx, int value_type, int64_t C,
                      int64_t n_chunks, const int32_t *chunk_ptr,
                      const int32_t *chunk_lengths, const int32_t *col,
                      const void *val, const void *x, void *y) {
    SMAX_HIP_CHECK_CTX(ctx);
    int rc = check_scs_args(ctx, "smax_hip_scs_spmv", value_type, C, n_chunks,
                            chunk_ptr, chunk_lengths, col, val, x, y);
    if (rc) return rc;
    SMAX_HIP_DISPATCH_VT(value_type,
                         return launch_scs_spmv<VT>(ctx, C, n_chunks,
                                                    n_chunks * C, chunk_ptr,
                                                    chunk_lengths, col, val,
                                                    nullptr, x, y, false));
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_scs_spmv_unpermuted(smax_hip_ctx ctx, int value_type, int64_t C,
                                 int64_t n_chunks, int64_t n_rows,
                                 const int32_t *chunk_ptr,
                                 const int32_t *chunk_lengths,
                                 const int32_t *col, const void *val,
                                 const int32_t *slot_row, const void *x,
                                 void *y) {
    SMAX_HIP_CHECK_CTX(ctx);
    int rc = check_scs_args(ctx, "smax_hip_scs_spmv_unpermuted", value_type, C,
                            n_chunks, chunk_ptr, chunk_lengths, col, val, x, y);
    if (rc) return rc;
    SMAX_HIP_REQUIRE(ctx, slot_row && n_rows > 0 && n_rows <= n_chunks * C,
                     "smax_hip_scs_spmv_unpermuted: bad slot_row / n_rows");
    SMAX_HIP_DISPATCH_VT(value_type,
                         return launch_scs_spmv<VT>(ctx, C, n_chunks, n_rows,
                                                    chunk_ptr, chunk_lengths,
                                                    col, val, slot_row, x, y,
                                                    true));
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_scs_plan_create(smax_hip_ctx ctx, int64_t C, int64_t sigma,
                             int64_t n_rows_padded, int64_t n_chunks,
                             int64_t n_elements, int64_t nnz,
                             const int32_t *chunk_lengths, smax_hip_scs_plan *out) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, out, "smax_hip_scs_plan_create: null output");
    *out = nullptr;
    SMAX_HIP_REQUIRE(ctx, C > 0 && sigma > 0 && n_chunks > 0 && n_elements >= 0 &&
                              nnz >= 0 && nnz <= n_elements && C <= INT32_MAX &&
                              n_chunks <= INT32_MAX / C && n_rows_padded == n_chunks * C &&
                              chunk_lengths,
                     "smax_hip_scs_plan_create: bad arguments");
    auto *plan = new smax_hip_scs_plan_s();
    plan->C = C;
    plan->n_chunks = n_chunks;
    int rc = build_schedule(ctx, C, sigma, n_rows_padded, n_chunks, n_elements, nnz,
                            chunk_lengths, &plan->sched);
    if (rc) {
        free_schedule(plan->sched);
        delete plan;
        return rc;
    }
    *out = plan;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_scs_plan_destroy(smax_hip_ctx ctx, smax_hip_scs_plan plan) {
    if (!plan) return SMAX_HIP_SUCCESS;
    if (ctx) {
        (void)bind(ctx);
        (void)hipStreamSynchronize(ctx->stream);
    }
    free_schedule(plan->sched);
    delete plan;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_scs_spmv_plan(smax_hip_ctx ctx, int value_type, smax_hip_scs_plan plan,
                           const int32_t *chunk_ptr, const int32_t *chunk_lengths,
                           const int32_t *col, const void *val, const void *x,
                           void *y) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, plan, "smax_hip_scs_spmv_plan: null plan");
    int rc = check_scs_args(ctx, "smax_hip_scs_spmv_plan", value_type, plan->C,
                            plan->n_chunks, chunk_ptr, chunk_lengths, col, val, x, y);
    if (rc) return rc;
    const int64_t npad = plan->n_chunks * plan->C;
    SMAX_HIP_DISPATCH_VT(value_type,
                         return launch_scs_spmv<VT>(ctx, plan->C, plan->n_chunks, npad,
                                                    chunk_ptr, chunk_lengths, col, val,
                                                    nullptr, x, y, false, &plan->sched));
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_scs_apply(smax_hip_ctx ctx, int value_type, smax_hip_scs A,
                       const void *x, void *y, int unpermuted) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, A, "smax_hip_scs_apply: null matrix");
    const smax_hip_scs_info &in = A->info;
    int rc = check_scs_args(ctx, "smax_hip_scs_apply", value_type, in.C, in.n_chunks,
                            in.chunk_ptr, in.chunk_lengths, in.col, in.val, x, y);
    if (rc) return rc;
    if (vt_val_bytes(value_type) != in.val_bytes)
        return fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                    "smax_hip_scs_apply: value type %d does not match %lld-byte values",
                    value_type, (long long)in.val_bytes);
    SMAX_HIP_DISPATCH_VT(value_type,
                         return launch_scs_spmv<VT>(ctx, in.C, in.n_chunks, in.n_rows,
                                                    in.chunk_ptr, in.chunk_lengths,
                                                    in.col, in.val, in.slot_row, x, y,
                                                    unpermuted != 0, &A->sched,
                                                    in.slot_len, &A->tails));
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_scs_get_tails(smax_hip_scs A, int64_t *n_slots, int64_t *n_waves,
                           int64_t *n_entries) {
    if (!A || !n_slots || !n_waves || !n_entries)
        return fail(nullptr, SMAX_HIP_ERROR_INVALID_VALUE, "smax_hip_scs_get_tails: null");
    *n_slots = A->tails.n_slots;
    *n_waves = A->tails.n_waves;
    *n_entries = A->tails.n_elements;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_scs_spmm(smax_hip_ctx ctx, int value_type, int64_t C,
                      int64_t n_chunks, int64_t n_rows,
                      const int32_t *chunk_ptr, const int32_t *chunk_lengths,
                      const int32_t *col, const void *val,
                      const int32_t *slot_row, int64_t k, const void *X,
                      void *Y) {
    SMAX_HIP_CHECK_CTX(ctx);
    int rc = check_scs_args(ctx, "smax_hip_scs_spmm", value_type, C, n_chunks,
                            chunk_ptr, chunk_lengths, col, val, X, Y);
    if (rc) return rc;
    SMAX_HIP_REQUIRE(ctx, slot_row && k > 0 && n_rows > 0 &&
                              n_rows <= n_chunks * C,
                     "smax_hip_scs_spmm: bad slot_row / n_rows / k");
    if (!extent_ok(n_chunks * C, k))
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "smax_hip_scs_spmm: k = %lld exceeds the launch limits", (long long)k);
    SMAX_HIP_DISPATCH_VT(value_type,
                         return launch_scs_spmm<VT>(ctx, C, n_chunks, n_rows, k, chunk_ptr,
                                                    chunk_lengths, nullptr, nullptr, col,
                                                    val, slot_row, X, Y));
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

int smax_hip_scs_apply_spmm(smax_hip_ctx ctx, int value_type, smax_hip_scs A,
                            int64_t k, const void *X, void *Y) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, A, "smax_hip_scs_apply_spmm: null matrix");
    SMAX_HIP_REQUIRE(ctx, !A->from_sell,
                     "smax_hip_scs_apply_spmm: the matrix was built from SELL arrays, whose slot "
                     "lengths may drop stored +0 entries; build it with smax_hip_scs_from_crs");
    const smax_hip_scs_info &in = A->info;
    int rc = check_scs_args(ctx, "smax_hip_scs_apply_spmm", value_type, in.C,
                            in.n_chunks, in.chunk_ptr, in.chunk_lengths, in.col, in.val,
                            X, Y);
    if (rc) return rc;
    SMAX_HIP_REQUIRE(ctx, k > 0, "smax_hip_scs_apply_spmm: k must be positive");
    if (!extent_ok(in.n_rows_padded, k))
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "smax_hip_scs_apply_spmm: k = %lld exceeds the launch limits", (long long)k);
    if (vt_val_bytes(value_type) != in.val_bytes)
        return fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                    "smax_hip_scs_apply_spmm: value type %d does not match %lld-byte "
                    "values", value_type, (long long)in.val_bytes);
    SMAX_HIP_DISPATCH_VT(value_type,
                         return launch_scs_spmm<VT>(ctx, in.C, in.n_chunks, in.n_rows, k,
                                                    in.chunk_ptr, in.chunk_lengths,
                                                    in.slot_len, A->sched.order_lf, in.col,
                                                    in.val, in.slot_row, X, Y, &A->longs));
    return SMAX_HIP_ERROR_UNSUPPORTED;
}

}  // extern "C"
