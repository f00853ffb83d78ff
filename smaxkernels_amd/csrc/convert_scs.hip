// CRS -> SELL-C-sigma on the GPU, bit-identical to
// SMAX::Utils::convert_crs_to_scs (src/utils/convert_formats.hpp:16-132).
//
// The only non-trivial step is the per-sigma-window std::sort of
// (index, count) pairs by count descending (convert_formats.hpp:46-55).
// std::sort is unstable, so tied rows end up in the order libstdc++'s
// introsort leaves them; that order is reproduced exactly here by running the
// introsort recursion level-synchronously over every segment at once (windows
// and segments of up to a few thousand rows inside LDS, k_sort_tiles; longer
// ones level by level over global memory until they are that short):
//
//  * a segment [h, e) with e - h > 16 and depth > 0 is partitioned exactly as
//    __unguarded_partition_pivot does (bits/stl_algo.h:1878-1907): the
//    median of (h+1, h+(e-h)/2, e-1) is swapped to h, then the Hoare scan
//    swaps the k-th "left stopper" (count <= pivot, scanning up from h+1)
//    with the k-th "right stopper" (count >= pivot, scanning down from e-1)
//    for every k with l_k < r_k.  With L(q) / R(q) the number of left / right
//    stoppers in (h, q] / [q, e), the swap count is s = max_q min(L(q),
//    R(q+1)) and the returned cut is min(l_{s+1}, r_s) — both read off
//    prefix sums, so every element's destination is known in parallel;
//  * both halves inherit depth - 1 (bits/stl_algo.h:1925-1941);
//  * a segment still longer than 16 at depth 0 is heap-sorted sequentially
//    (make_heap + sort_heap, bits/stl_heap.h);
//  * the closing __final_insertion_sort never moves an element across a
//    partition boundary (left parts hold counts >= pivot, right parts
//    <= pivot, and insertion only passes strictly smaller counts), so it is
//    a stable insertion sort of every segment of <= 16 elements.
//
// Everything else (chunk lengths, chunk_ptr, perm, zero-padded col/val and
// the CRS-order scatter) is data-parallel.
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "convert_internal.hpp"
#include "scan.hpp"

namespace smaxhip {

// SEG_PARKED: short enough for k_sort_tiles, which runs the rest of it.
enum : int32_t { SEG_ACTIVE = 0, SEG_LEAF = 1, SEG_HEAP = 2, SEG_NONE = 3, SEG_PARKED = 4 };
constexpr int kThreshold = 16;  // _S_threshold, bits/stl_algo.h:1855
constexpr int kThreads = 256;

// k_sort_tiles: positions of a workgroup's tile, and the longest segment that
// the level-by-level phase leaves to it (segments that start in the same
// kParked positions end within 2 * kParked - 1 of the first, one tile).
constexpr int kTile = 4096;
constexpr int kTileThreads = 1024;
constexpr int kTileItems = kTile / kTileThreads;
constexpr int kParked = kTile / 2;

__device__ __forceinline__ int32_t lg2(int64_t n) {
    return 63 - __clzll(static_cast<unsigned long long>(n));
}

// ------------------------------------------------------------ init
// Windows longer than a tile: their segments and (index, count) pairs.
__global__ void k_init(int64_t n, int64_t n_rows, int64_t sigma,
                       const int32_t *__restrict__ row_ptr,
                       int32_t *__restrict__ idx, int32_t *__restrict__ cnt,
                       int32_t *__restrict__ head, int32_t *__restrict__ end,
                       int32_t *__restrict__ depth, int32_t *__restrict__ state,
                       int32_t *__restrict__ list, int64_t *__restrict__ nlist) {
    int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= n) return;
    idx[q] = static_cast<int32_t>(q);
    cnt[q] = q < n_rows ? row_ptr[q + 1] - row_ptr[q] : 0;
    int64_t h = (q / sigma) * sigma;
    head[q] = static_cast<int32_t>(h);
    if (h == q) {
        int64_t e = h + sigma < n ? h + sigma : n;
        int64_t len = e - h;
        end[q] = static_cast<int32_t>(e);
        depth[q] = 2 * lg2(len);  // std::__lg(last - first) * 2
        if (len > kParked) {
            state[q] = SEG_ACTIVE;
            list[atomicAdd(reinterpret_cast<unsigned long long *>(nlist), 1ull)] =
                static_cast<int32_t>(q);
        } else {
            state[q] = SEG_PARKED;
        }
    } else {
        state[q] = SEG_NONE;
    }
}

// ------------------------------------------------------------ level kernels
__device__ __forceinline__ void swap_pair(int32_t *idx, int32_t *cnt,
                                          int64_t a, int64_t b) {
    int32_t ti = idx[a], tc = cnt[a];
    idx[a] = idx[b];
    cnt[a] = cnt[b];
    idx[b] = ti;
    cnt[b] = tc;
}

// __move_median_to_first (bits/stl_algo.h:79-97) with comp(a,b) = a > b.
__global__ void k_pivot(int64_t nl, const int32_t *__restrict__ list,
                        const int32_t *__restrict__ end,
                        const int32_t *__restrict__ depth,
                        int32_t *__restrict__ state, int32_t *__restrict__ idx,
                        int32_t *__restrict__ cnt, int32_t *__restrict__ pv,
                        int32_t *__restrict__ sw) {
    int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= nl) return;
    const int64_t h = list[t];
    if (depth[h] == 0) {  // __partial_sort fallback, bits/stl_algo.h:1931-1935
        state[h] = SEG_HEAP;
        return;
    }
    const int64_t e = end[h];
    const int64_t a = h + 1, b = h + (e - h) / 2, c = e - 1;
    const int32_t ca = cnt[a], cb = cnt[b], cc = cnt[c];
    int64_t m;
    if (ca > cb) {
        if (cb > cc) m = b;
        else if (ca > cc) m = c;
        else m = a;
    } else if (ca > cc) m = a;
    else if (cb > cc) m = c;
    else m = b;
    swap_pair(idx, cnt, h, m);
    pv[h] = cnt[h];
    sw[h] = 0;
}

// Left / right stopper flags of every element inside an active segment.
__global__ void k_flags(int64_t n, const int32_t *__restrict__ head,
                        const int32_t *__restrict__ state,
                        const int32_t *__restrict__ cnt,
                        const int32_t *__restrict__ pv,
                        int32_t *__restrict__ lf, int32_t *__restrict__ rf) {
    int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int64_t h = head[q];
    int32_t l = 0, r = 0;
    if (state[h] == SEG_ACTIVE && q > h) {
        const int32_t c = cnt[q], p = pv[h];
        l = c <= p;  // !comp(*first, *pivot): left scan stops
        r = c >= p;  // !comp(*pivot, *last):  right scan stops
    }
    lf[q] = l;
    rf[q] = r;
}

__device__ __forceinline__ int32_t suffix_at(const int32_t *SR, int64_t q,
                                             int64_t n) {
    return q < n ? SR[q] : 0;
}

// Stopper ranks, position lists and the swap count s of every segment.
// s is a maximum over the segment's positions: a wavefront whose lanes all
// lie in one segment takes its maximum first and issues one atomic (one
// per element would serialise millions of atomics on one address when a
// sigma window is one large segment).
__global__ __launch_bounds__(256) void k_rank(
    int64_t n, const int32_t *__restrict__ head, const int32_t *__restrict__ state,
    const int32_t *__restrict__ end, const int32_t *__restrict__ cnt,
    const int32_t *__restrict__ pv, const int32_t *__restrict__ PL,
    const int32_t *__restrict__ SR, int32_t *__restrict__ posL,
    int32_t *__restrict__ posR, int32_t *__restrict__ sw) {
    const int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    int64_t h = -1;
    int32_t cand = 0;
    if (q < n) {
        h = head[q];
        if (state[h] == SEG_ACTIVE) {
            const int64_t e = end[h];
            const int32_t se = suffix_at(SR, e, n);
            const int32_t Lq = PL[q] - PL[h];
            if (q > h) {
                const int32_t c = cnt[q], p = pv[h];
                if (c <= p) posL[h + Lq] = static_cast<int32_t>(q);
                if (c >= p) posR[h + (SR[q] - se)] = static_cast<int32_t>(q);
            }
            const int32_t Rq1 = q + 1 < e ? SR[q + 1] - se : 0;
            cand = Lq < Rq1 ? Lq : Rq1;
        }
    }
    // every lane of the wavefront reaches this point
    if (__all(h == __shfl(h, 0))) {
        int32_t m = cand;
#pragma unroll
        for (int off = kWave / 2; off >= 1; off >>= 1) m = max(m, __shfl_xor(m, off));
        if ((threadIdx.x & (kWave - 1)) == 0 && m > 0) atomicMax(sw + h, m);
    } else if (cand > 0) {
        atomicMax(sw + h, cand);
    }
}

__global__ void k_cut(int64_t nl, const int32_t *__restrict__ list,
                      const int32_t *__restrict__ state,
                      const int32_t *__restrict__ end,
                      const int32_t *__restrict__ PL,
                      const int32_t *__restrict__ posL,
                      const int32_t *__restrict__ posR,
                      const int32_t *__restrict__ sw, int32_t *__restrict__ cut,
                      int64_t *__restrict__ errflag) {
    int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= nl) return;
    const int64_t h = list[t];
    if (state[h] != SEG_ACTIVE) return;
    const int64_t e = end[h];
    const int32_t s = sw[h];
    const int32_t ltot = PL[e - 1] - PL[h];
    const int64_t big = e;  // never returned: one of the two always exists
    const int64_t lnext = s + 1 <= ltot ? posL[h + s + 1] : big;
    const int64_t rs = s >= 1 ? posR[h + s] : big;
    int64_t c = lnext < rs ? lnext : rs;
    if (c <= h || c >= e) {  // cannot happen for a valid partition
        atomicAdd(reinterpret_cast<unsigned long long *>(errflag), 1ull);
        c = h + 1;
    }
    cut[h] = static_cast<int32_t>(c);
}

__global__ void k_move(int64_t n, const int32_t *__restrict__ head,
                       const int32_t *__restrict__ state,
                       const int32_t *__restrict__ end,
                       const int32_t *__restrict__ pv,
                       const int32_t *__restrict__ sw,
                       const int32_t *__restrict__ PL,
                       const int32_t *__restrict__ SR,
                       const int32_t *__restrict__ posL,
                       const int32_t *__restrict__ posR,
                       const int32_t *__restrict__ idx,
                       const int32_t *__restrict__ cnt,
                       int32_t *__restrict__ idx2, int32_t *__restrict__ cnt2) {
    int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int64_t h = head[q];
    int64_t dest = q;
    const int32_t c = cnt[q];
    if (state[h] == SEG_ACTIVE && q > h) {
        const int32_t p = pv[h], s = sw[h];
        if (c <= p) {
            const int32_t Lq = PL[q] - PL[h];
            if (Lq <= s) dest = posR[h + Lq];
        }
        if (dest == q && c >= p) {
            const int32_t Rq = SR[q] - suffix_at(SR, end[h], n);
            if (Rq <= s) dest = posL[h + Rq];
        }
    }
    idx2[dest] = idx[q];
    cnt2[dest] = c;
}

__global__ void k_split(int64_t n, int32_t *__restrict__ head,
                        const int32_t *__restrict__ state,
                        const int32_t *__restrict__ cut) {
    int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int64_t h = head[q];
    if (state[h] == SEG_ACTIVE && q >= cut[h]) head[q] = cut[h];
}

__global__ void k_newsegs(int64_t nl, const int32_t *__restrict__ list,
                          int32_t *__restrict__ state, int32_t *__restrict__ end,
                          int32_t *__restrict__ depth,
                          const int32_t *__restrict__ cut,
                          int32_t *__restrict__ next,
                          int64_t *__restrict__ nnext) {
    int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= nl) return;
    const int32_t h = list[t];
    if (state[h] != SEG_ACTIVE) return;
    const int32_t e = end[h], c = cut[h], d = depth[h] - 1;
    end[c] = e;
    depth[c] = d;
    end[h] = c;
    depth[h] = d;
    const bool right = e - c > kParked, left = c - h > kParked;
    state[c] = right ? SEG_ACTIVE : SEG_PARKED;
    state[h] = left ? SEG_ACTIVE : SEG_PARKED;
    unsigned long long *cntp = reinterpret_cast<unsigned long long *>(nnext);
    if (right) next[atomicAdd(cntp, 1ull)] = c;
    if (left) next[atomicAdd(cntp, 1ull)] = h;
}

// ------------------------------------------------------------ heap fallback
// make_heap + sort_heap of bits/stl_heap.h on (idx, cnt) pairs,
// comp(a, b) = a.count > b.count.
template <typename Index>
__device__ void push_heap_d(Index *I, int32_t *K, int64_t hole, int64_t top,
                            Index vi, int32_t vk) {
    int64_t parent = (hole - 1) / 2;
    while (hole > top && K[parent] > vk) {
        I[hole] = I[parent];
        K[hole] = K[parent];
        hole = parent;
        parent = (hole - 1) / 2;
    }
    I[hole] = vi;
    K[hole] = vk;
}

template <typename Index>
__device__ void adjust_heap_d(Index *I, int32_t *K, int64_t hole,
                              int64_t len, Index vi, int32_t vk) {
    const int64_t top = hole;
    int64_t second = hole;
    while (second < (len - 1) / 2) {
        second = 2 * (second + 1);
        if (K[second] > K[second - 1]) second--;
        I[hole] = I[second];
        K[hole] = K[second];
        hole = second;
    }
    if ((len & 1) == 0 && second == (len - 2) / 2) {
        second = 2 * (second + 1);
        I[hole] = I[second - 1];
        K[hole] = K[second - 1];
        hole = second - 1;
    }
    push_heap_d(I, K, hole, top, vi, vk);
}

template <typename Index>
__device__ void heap_sort_d(Index *I, int32_t *K, int64_t len) {
    if (len >= 2) {  // __make_heap
        int64_t parent = (len - 2) / 2;
        for (;;) {
            adjust_heap_d(I, K, parent, len, I[parent], K[parent]);
            if (parent == 0) break;
            parent--;
        }
    }
    for (int64_t last = len; last > 1;) {  // __sort_heap / __pop_heap
        --last;
        const Index vi = I[last];
        const int32_t vk = K[last];
        I[last] = I[0];
        K[last] = K[0];
        adjust_heap_d(I, K, 0, last, vi, vk);
    }
}

// Where position p's pair ends up: slot p holds row `row` of `count` entries.
__device__ __forceinline__ void emit_slot(int64_t p, int32_t row, int32_t count, int64_t n_rows,
                                          int32_t *__restrict__ slot_row,
                                          int32_t *__restrict__ slot_len,
                                          int32_t *__restrict__ perm) {
    slot_row[p] = row;
    slot_len[p] = count;
    if (row < n_rows) perm[row] = static_cast<int32_t>(p);
}

// Segments that ran out of depth while still too long for a tile.
__global__ void k_heapsort(int64_t n, int64_t n_rows, const int32_t *__restrict__ head,
                           const int32_t *__restrict__ state,
                           const int32_t *__restrict__ end, int32_t *idx, int32_t *cnt,
                           int32_t *__restrict__ slot_row, int32_t *__restrict__ slot_len,
                           int32_t *__restrict__ perm) {
    int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= n || head[q] != q || state[q] != SEG_HEAP) return;
    heap_sort_d(idx + q, cnt + q, end[q] - q);
    for (int64_t p = q; p < end[q]; ++p) emit_slot(p, idx[p], cnt[p], n_rows, slot_row, slot_len, perm);
}

// ------------------------------------------------------------ tiles in LDS
// The same recursion for every segment of one tile of up to kTile positions,
// all levels in one launch, and the leaves; the result goes straight to
// slot_row, slot_len and perm.
//   WINDOWS: tile t holds the whole windows [t * span, t * span + span), span
//     a multiple of sigma; counts come from row_ptr.
//   otherwise: the parked segments that start in the t-th kParked positions,
//     with their pairs in idx / cnt (segments longer than kParked are done by
//     k_heapsort).
//
// A thread owns kTileItems neighbouring positions and keeps their segment
// heads in registers.  Per level: pivots; stopper flags, both kinds in one
// packed 16 + 16 bit prefix sum; stopper positions by rank, and the swap count
// s, which the position where L(q) = min(L, R) ends writes (L(q) never falls
// and R(q + 1) never rises, so max_q min(L(q), R(q + 1)) lies there); moves;
// new segments.
//
// What bounds it: LDS latency between some six barriers a level, 72 KB a
// workgroup, two workgroups a CU.  Level by level over global memory, ten
// launches each, a conversion of 2,000,003 rows at sigma = 4096 spent 2.6 ms
// here.
template <bool WINDOWS>
__global__ __launch_bounds__(kTileThreads, 8) void k_sort_tiles(
    int64_t n, int64_t n_rows, int64_t sigma, int64_t span, const int32_t *__restrict__ row_ptr,
    const int32_t *__restrict__ idx_in, const int32_t *__restrict__ cnt_in,
    const int32_t *__restrict__ g_head, const int32_t *__restrict__ g_end,
    const int32_t *__restrict__ g_depth, int32_t *__restrict__ slot_row,
    int32_t *__restrict__ slot_len, int32_t *__restrict__ perm, int64_t *__restrict__ errflag) {
    __shared__ __align__(16) int32_t cnt[kTile];
    __shared__ __align__(16) uint32_t pre[kTile];  // inclusive prefix: left (low), right (high)
    __shared__ uint16_t idx[kTile];
    __shared__ uint16_t pos_l[kTile + 1], pos_r[kTile + 1];  // entry h: swap count, cut
    __shared__ uint16_t seg_end[kTile];
    __shared__ uint8_t seg_depth[kTile], seg_state[kTile];
    __shared__ uint32_t wave_sum[kTileThreads / kWave];
    const int tid = static_cast<int>(threadIdx.x);
    const int q0 = tid * kTileItems;
    int64_t base;
    int w;  // positions of this tile
    if (WINDOWS) {
        base = static_cast<int64_t>(blockIdx.x) * span;
        w = static_cast<int>(n - base < span ? n - base : span);
    } else {
        const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kParked;
        const int64_t t1 = (t0 + kParked < n ? t0 + kParked : n) - 1;
        const int64_t h0 = g_head[t0], h1 = g_head[t1];
        base = h0 == t0 ? t0 : g_end[h0];
        const int64_t stop = g_end[h1] - h1 > kParked ? h1 : g_end[h1];
        if (stop <= base) return;
        w = static_cast<int>(stop - base);
    }
    int head[kTileItems];
#pragma unroll
    for (int u = 0; u < kTileItems; ++u) {
        const int q = q0 + u;
        head[u] = -1;
        if (q < w) {
            const int64_t g = base + q;
            int e, depth;
            if (WINDOWS) {
                cnt[q] = g < n_rows ? row_ptr[g + 1] - row_ptr[g] : 0;
                head[u] = q - q % static_cast<int>(sigma);
                e = head[u] + static_cast<int>(sigma) < w ? head[u] + static_cast<int>(sigma) : w;
                depth = 2 * lg2(e - head[u]);
            } else {
                cnt[q] = cnt_in[g];
                const int64_t h = g_head[g];
                head[u] = static_cast<int>(h - base);
                e = static_cast<int>(g_end[h] - base);
                depth = g_depth[h];
            }
            idx[q] = static_cast<uint16_t>(q);
            if (head[u] == q) {
                seg_end[q] = static_cast<uint16_t>(e);
                seg_depth[q] = static_cast<uint8_t>(depth);
                seg_state[q] = e - q > kThreshold ? SEG_ACTIVE : SEG_LEAF;
            }
        }
    }
    __syncthreads();
    for (;;) {
        bool any = false;
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            const int h = q0 + u;
            if (head[u] != h || seg_state[h] != SEG_ACTIVE) continue;
            if (seg_depth[h] == 0) {  // __partial_sort fallback
                seg_state[h] = SEG_HEAP;
                continue;
            }
            any = true;
            const int e = seg_end[h];
            const int a = h + 1, b = h + (e - h) / 2, c = e - 1;
            const int32_t ca = cnt[a], cb = cnt[b], cc = cnt[c];
            int m;  // __move_median_to_first, comp(a, b) = a > b
            if (ca > cb) m = cb > cc ? b : ca > cc ? c : a;
            else m = ca > cc ? a : cb > cc ? c : b;
            const int32_t tc = cnt[h];
            const uint16_t ti = idx[h];
            cnt[h] = cnt[m];
            idx[h] = idx[m];
            cnt[m] = tc;
            idx[m] = ti;
        }
        if (!__syncthreads_or(any)) break;
        uint32_t mine[kTileItems];  // flags, then inclusive prefix
        bool active[kTileItems];
        uint32_t sum = 0;
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            const int q = q0 + u, h = head[u];
            active[u] = h >= 0 && seg_state[h] == SEG_ACTIVE;
            uint32_t f = 0;
            if (active[u] && q > h) {
                const int32_t c = cnt[q], p = cnt[h];
                f = (c <= p ? 1u : 0u) | (c >= p ? 0x10000u : 0u);
            }
            sum += f;
            mine[u] = sum;
        }
        const uint32_t incl = wave_incl_scan(sum);
        if ((tid & (kWave - 1)) == kWave - 1) wave_sum[tid / kWave] = incl;
        __syncthreads();
        uint32_t before = incl - sum;
        for (int v = 0; v < tid / kWave; ++v) before += wave_sum[v];
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            mine[u] += before;
            pre[q0 + u] = mine[u];
        }
        __syncthreads();
        // stopper ranks: L(q) of (h, q], R(q) of [q, e)
        int lq[kTileItems], rq1[kTileItems];
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            const int q = q0 + u, h = head[u];
            if (!active[u]) continue;
            const int e = seg_end[h];
            const uint32_t ph = pre[h], pe = pre[e - 1];
            lq[u] = static_cast<int>((mine[u] & 0xffffu) - (ph & 0xffffu));
            rq1[u] = static_cast<int>((pe >> 16) - (mine[u] >> 16));
            if (q > h) {
                const int32_t c = cnt[q], p = cnt[h];
                if (c <= p) pos_l[h + lq[u]] = static_cast<uint16_t>(q);
                if (c >= p) pos_r[h + rq1[u] + 1] = static_cast<uint16_t>(q);
            }
            if (lq[u] <= rq1[u]) {
                int ln = INT32_MAX, rn = 0;
                if (q + 1 < e) {
                    const uint32_t pn = pre[q + 1];
                    ln = static_cast<int>((pn & 0xffffu) - (ph & 0xffffu));
                    rn = static_cast<int>((pe >> 16) - (pn >> 16));
                }
                if (ln > rn) pos_l[h] = static_cast<uint16_t>(lq[u] > rn ? lq[u] : rn);
            }
        }
        __syncthreads();
        int dest[kTileItems];
        int32_t mc[kTileItems];
        uint16_t mi[kTileItems];
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            const int q = q0 + u, h = head[u];
            dest[u] = q;
            if (!active[u]) continue;
            const int s = pos_l[h];
            if (q == h) {
                const int e = seg_end[h];
                const int ltot = static_cast<int>((pre[e - 1] & 0xffffu) - (pre[h] & 0xffffu));
                const int lnext = s + 1 <= ltot ? pos_l[h + s + 1] : e;
                const int rs = s >= 1 ? pos_r[h + s] : e;
                int cut = lnext < rs ? lnext : rs;
                if (cut <= h || cut >= e) {  // cannot happen for a valid partition
                    atomicAdd(reinterpret_cast<unsigned long long *>(errflag), 1ull);
                    cut = h + 1;
                }
                pos_r[h] = static_cast<uint16_t>(cut);
                continue;
            }
            mc[u] = cnt[q];
            mi[u] = idx[q];
            const int32_t p = cnt[h];
            if (mc[u] <= p && lq[u] <= s) dest[u] = pos_r[h + lq[u]];
            if (dest[u] == q && mc[u] >= p && rq1[u] + 1 <= s) dest[u] = pos_l[h + rq1[u] + 1];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kTileItems; ++u) {
            const int q = q0 + u, h = head[u];
            if (!active[u]) continue;
            if (dest[u] != q) {
                cnt[dest[u]] = mc[u];
                idx[dest[u]] = mi[u];
            }
            const int cut = pos_r[h];
            if (q == h) {
                const int e = seg_end[h];
                const uint8_t d = static_cast<uint8_t>(seg_depth[h] - 1);
                seg_end[cut] = static_cast<uint16_t>(e);
                seg_depth[cut] = d;
                seg_state[cut] = e - cut > kThreshold ? SEG_ACTIVE : SEG_LEAF;
                seg_end[h] = static_cast<uint16_t>(cut);
                seg_depth[h] = d;
                seg_state[h] = cut - h > kThreshold ? SEG_ACTIVE : SEG_LEAF;
            } else if (q >= cut) {
                head[u] = cut;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < kTileItems; ++u) {
        const int h = q0 + u;
        if (head[u] == h && seg_state[h] == SEG_HEAP) heap_sort_d(idx + h, cnt + h, seg_end[h] - h);
    }
    __syncthreads();
    // leaves: the stable order by count descending, each position counting
    // the elements of its segment (at most 16) that come before it
#pragma unroll
    for (int u = 0; u < kTileItems; ++u) {
        const int q = q0 + u, h = head[u];
        if (h < 0) continue;
        const int32_t c = cnt[q];
        int p = q;
        if (seg_state[h] == SEG_LEAF) {
            p = h;
            const int e = seg_end[h];
            for (int t = h; t < e; ++t) p += cnt[t] > c || (cnt[t] == c && t < q);
        }
        const int64_t g = base + idx[q];
        emit_slot(base + p, WINDOWS ? static_cast<int32_t>(g) : idx_in[g], c, n_rows, slot_row,
                  slot_len, perm);
    }
}

// ------------------------------------------------------------ chunk layout
__global__ void k_chunk_len(int64_t n_chunks, int64_t C,
                            const int32_t *__restrict__ cnt,
                            int32_t *__restrict__ chunk_len,
                            int64_t *__restrict__ chunk_elems) {
    int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= n_chunks) return;
    int32_t m = cnt[c * C];
    for (int64_t i = 1; i < C; ++i) m = max(m, cnt[c * C + i]);
    chunk_len[c] = m;
    chunk_elems[c] = static_cast<int64_t>(m) * C;
}

// chunk_ptr from the inclusive sums; the number of elements also to *total.
__global__ void k_chunk_ptr(int64_t n_chunks,
                            const int64_t *__restrict__ incl,
                            int32_t *__restrict__ chunk_ptr, int64_t *__restrict__ total) {
    int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c > n_chunks) return;
    chunk_ptr[c] = c == 0 ? 0 : static_cast<int32_t>(incl[c - 1]);
    if (c == n_chunks) *total = incl[c - 1];
}

// Lists the slots of `from` entries and more (smax_hip_scs_longs); counts[0]
// and [1] (zero on entry): whole-workgroup ones and the others.  Their order
// is that of the atomics; only which workgroup runs which depends on it.
__global__ void k_long_slots(int64_t n, int32_t from, const int32_t *__restrict__ slot_len,
                             int32_t *__restrict__ list, int64_t cap,
                             int64_t *__restrict__ counts) {
    const int64_t s = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= n || slot_len[s] < from) return;
    const bool whole = slot_len[s] >= kLongestRow;
    const int64_t i = static_cast<int64_t>(
        atomicAdd(reinterpret_cast<unsigned long long *>(counts + (whole ? 0 : 1)), 1ull));
    list[whole ? i : cap - 1 - i] = static_cast<int32_t>(s);
}

__global__ void k_fill_i32(int64_t n, int32_t v, int32_t *__restrict__ p) {
    int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// The SELL arrays (convert_formats.hpp:101-128), element by element: element
// j of slot i of chunk c, at chunk_ptr[c] + j*C + i, is entry j of the slot's
// row, or padding (column 0, value 0, no source) past the row's end.
//
// What bounds it: the stores of the padded arrays, 8 bytes and the value each
// (contiguous; 225 us for the 80 M elements of 2,000,003 rows at sigma = 4096
// in FP64), and, not overlapped with them, the reads along 64 rows at once
// (260 us).  A wavefront takes kFillItems x 64 consecutive elements wherever
// they lie, so rows of thousands of entries are shared out too, and a lane
// that keeps its slot reads kFillItems entries of one row while their lines
// are in L1; the outputs pass the caches by.  0.65 ms with 4 elements at a time
// and 256 apart, 0.56 this way.  Scattering in CRS order instead (a 21-step
// search of each entry's row, scattered 4- and 8-byte stores) after three
// passes that cleared the arrays took 1.15 + 0.24 ms.
constexpr int kFillItems = 16;

template <typename V>
__global__ __launch_bounds__(256) void k_fill(
    int64_t n_elements, int64_t n_chunks, int64_t n_rows, int32_t C, FastDiv by_c,
    const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
    const V *__restrict__ val, const int32_t *__restrict__ src_map,
    const int32_t *__restrict__ chunk_ptr, const int32_t *__restrict__ slot_row,
    const int32_t *__restrict__ slot_len, int32_t *__restrict__ out_col, V *__restrict__ out_val,
    int32_t *__restrict__ out_src) {
    // neighbouring workgroups, whose rows share lines, on one XCD
    const int64_t w0 = (xcd_block(blockIdx.x, gridDim.x) * 256 + (threadIdx.x & ~(kWave - 1))) *
                       kFillItems;
    if (w0 >= n_elements) return;  // whole wavefronts
    const int64_t e0 = w0 + (threadIdx.x & (kWave - 1));
    int64_t c = wave_row_of(chunk_ptr, n_chunks, w0);
    int32_t begin = chunk_ptr[c], end = chunk_ptr[c + 1];
    int64_t at = -1;  // the slot whose row start and length are held
    int32_t start = 0, len = 0;
    int32_t from[kFillItems];  // each element's CRS position, -1 for padding
#pragma unroll
    for (int u = 0; u < kFillItems; ++u) {
        const int64_t e = e0 + u * kWave;
        from[u] = -1;
        if (e >= n_elements) continue;
        if (e >= end) {
            // the next chunks in turn; past a run of empty ones by search
            for (int step = 0; e >= end && step < 8; ++step) end = chunk_ptr[++c + 1];
            if (e >= end) {
                c = row_of(chunk_ptr, c, n_chunks, e);
                end = chunk_ptr[c + 1];
            }
            begin = chunk_ptr[c];
        }
        const int32_t off = static_cast<int32_t>(e - begin);
        const int32_t j = by_c(off);
        const int64_t slot = c * C + (off - j * C);
        if (slot != at) {
            at = slot;
            len = slot_len[slot];
            const int32_t r = slot_row[slot];
            start = r < n_rows ? row_ptr[r] : 0;
        }
        if (j < len) from[u] = start + j;
    }
    int32_t vc[kFillItems], vs[kFillItems];
    V vv[kFillItems];
#pragma unroll
    for (int u = 0; u < kFillItems; ++u) {
        vc[u] = 0;
        vs[u] = from[u];
        if (from[u] >= 0) {
            vc[u] = col[from[u]];
            if (src_map) vs[u] = src_map[from[u]];
        }
    }
#pragma unroll
    for (int u = 0; u < kFillItems; ++u) vv[u] = vs[u] >= 0 ? val[vs[u]] : V(0);
#pragma unroll
    for (int u = 0; u < kFillItems; ++u) {
        const int64_t e = e0 + u * kWave;
        if (e >= n_elements) continue;
        __builtin_nontemporal_store(vc[u], out_col + e);
        __builtin_nontemporal_store(vv[u], out_val + e);
        __builtin_nontemporal_store(vs[u], out_src + e);
    }
}

// val[e] = crs_val[src[e]].  What bounds it: the reads along 64 rows at once,
// which for a transposed layout are scattered.  A lane takes ITEMS elements of
// its slot, whose values share lines while they are in L1 (and as many reads
// are in flight), and the stores pass the caches by.  Layouts, FP32, 1 -> 8
// items: 100,000 rows 14.1 -> 9.8 us, 1,000,000 82 -> 55, transposed 188 ->
// 182; 200,000 rows, FP64, transposed 33 -> 24.  Below kRefreshWide elements
// that leaves CUs idle (transposed, 40,013 rows: 4.3 us with one item, 4.9).
// STREAM: not where the tail waves' copy reads the values next, whose lanes
// follow one slot each and wait for every entry: 50,000 rows, SELL-32-1, FP64
// 1043 us for that copy after streaming stores, 609 otherwise.
constexpr int64_t kRefreshWide = 1 << 20;

template <typename V, int ITEMS, bool STREAM>
__global__ __launch_bounds__(256) void k_refresh(int64_t n_elem, const int32_t *__restrict__ src,
                                                 const V *__restrict__ crs_val,
                                                 V *__restrict__ val) {
    const int64_t block = ITEMS > 1 ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t e0 = (block * 256 + (threadIdx.x & ~(kWave - 1))) * ITEMS +
                       (threadIdx.x & (kWave - 1));
    int32_t s[ITEMS];
    V v[ITEMS];
#pragma unroll
    for (int u = 0; u < ITEMS; ++u)
        s[u] = e0 + u * kWave < n_elem ? src[e0 + u * kWave] : -1;
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) v[u] = s[u] >= 0 ? crs_val[s[u]] : V(0);
#pragma unroll
    for (int u = 0; u < ITEMS; ++u)
        if (e0 + u * kWave < n_elem) {
            if constexpr (STREAM) __builtin_nontemporal_store(v[u], val + e0 + u * kWave);
            else val[e0 + u * kWave] = v[u];
        }
}

template <typename V>
static int launch_refresh(smax_hip_ctx ctx, int64_t m, const int32_t *src, const void *crs_val,
                          void *val, bool stream) {
    const auto launch = [&](auto kernel, int items) {
        hipLaunchKernelGGL(kernel, grid_for(m, 256 * items), dim3(256), 0, ctx->stream, m, src,
                           static_cast<const V *>(crs_val), static_cast<V *>(val));
    };
    if (m < kRefreshWide) launch(k_refresh<V, 1, false>, 1);
    else if (stream) launch(k_refresh<V, 8, true>, 8);
    else launch(k_refresh<V, 8, false>, 8);
    SMAX_HIP_LAUNCHED(ctx, "k_refresh");
    return SMAX_HIP_SUCCESS;
}

// ------------------------------------------------------- caller SELL arrays
// Structure checks of SELL arrays handed in by a caller: every chunk's range
// is C * chunk_lengths[c] entries from chunk_ptr[c] (chunk_ptr[0] = 0,
// chunk_ptr[n_chunks] = n_elements) and every column lies in [0, n_cols).
// Any failure sets *bad (every writer stores the same 1).
__global__ void k_check_sell_chunks(int64_t n_chunks, int64_t C, int64_t n_elements,
                                    const int32_t *__restrict__ chunk_ptr,
                                    const int32_t *__restrict__ chunk_len,
                                    int32_t *__restrict__ bad) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c > n_chunks) return;
    if (c == 0 && chunk_ptr[0] != 0) *bad = 1;
    if (c == n_chunks) {
        if (chunk_ptr[c] != n_elements) *bad = 1;
        return;
    }
    const int64_t len = chunk_len[c];
    if (len < 0 || static_cast<int64_t>(chunk_ptr[c + 1]) - chunk_ptr[c] != C * len) *bad = 1;
}

__global__ void k_check_sell_cols(int64_t n_elements, int64_t n_cols,
                                  const int32_t *__restrict__ col, int32_t *__restrict__ bad) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e < n_elements && (col[e] < 0 || col[e] >= n_cols)) *bad = 1;
}

// slot_row[perm[r]] = r (slot_row prefilled with n_rows, which marks padding);
// perm entries outside [0, n_slots) set *bad and are skipped.
__global__ void k_slot_row_from_perm(int64_t n_rows, int64_t n_slots,
                                     const int32_t *__restrict__ perm,
                                     int32_t *__restrict__ slot_row, int32_t *__restrict__ bad) {
    const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= n_rows) return;
    const int32_t s = perm[r];
    if (s < 0 || s >= n_slots) {
        *bad = 1;
        return;
    }
    slot_row[s] = static_cast<int32_t>(r);
}

// After the scatter: a perm that maps two rows to one slot leaves one of them
// unmatched.
__global__ void k_check_perm(int64_t n_rows, const int32_t *__restrict__ perm,
                             const int32_t *__restrict__ slot_row, int32_t *__restrict__ bad) {
    const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r < n_rows && slot_row[perm[r]] != r) *bad = 1;
}

// Stored length of each slot of caller SELL arrays: the slot's elements up to
// its last one that is not +0.0 (all value bits zero) at column 0.  Trailing
// +0.0 entries at column 0 are exactly the reference's padding elements: each
// adds fma(+0, x[0], acc), the padding term, which a lane that stops early
// applies once (it is idempotent), so the product is unchanged bit for bit.
// A trailing -0.0 stays: fma(-0, x, -0) = -0 where fma(+0, x, -0) = +0.
template <typename E>
__global__ void k_sell_slot_len(int64_t n_slots, int64_t C,
                                const int32_t *__restrict__ chunk_ptr,
                                const int32_t *__restrict__ chunk_len,
                                const int32_t *__restrict__ col, const E *__restrict__ val,
                                int32_t *__restrict__ slot_len) {
    const int64_t s = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= n_slots) return;
    const int64_t c = s / C, base = static_cast<int64_t>(chunk_ptr[c]) + s % C;
    int j = chunk_len[c];
    while (j > 0) {
        const int64_t e = base + static_cast<int64_t>(j - 1) * C;
        if (val[e] != E(0) || col[e] != 0) break;
        --j;
    }
    slot_len[s] = j;
}

// ------------------------------------------------------------ host side
// Temporary device buffers, released (after the stream drains) on scope exit.
struct Scratch {
    smax_hip_ctx ctx;
    std::vector<void *> ptrs;
    explicit Scratch(smax_hip_ctx c) : ctx(c) {}
    ~Scratch() {
        if (!ptrs.empty()) (void)hipStreamSynchronize(ctx->stream);
        for (void *p : ptrs) dev_free(p);
    }
    template <typename T>
    int get(smax_hip_ctx ctx, T **p, int64_t n, const char *what) {
        void *q = nullptr;
        int rc = dev_alloc(ctx, &q, sizeof(T) * static_cast<size_t>(n > 0 ? n : 1),
                           what);
        if (rc) return rc;
        ptrs.push_back(q);
        *p = static_cast<T *>(q);
        return SMAX_HIP_SUCCESS;
    }
};

void scs_free_arrays(smax_hip_scs_info &in) {
    dev_free(in.chunk_ptr);
    dev_free(in.chunk_lengths);
    dev_free(in.col);
    dev_free(in.val);
    dev_free(in.perm);
    dev_free(in.slot_row);
    dev_free(in.src_index);
    dev_free(in.slot_len);
    in.chunk_ptr = in.chunk_lengths = in.col = in.perm = in.slot_row =
        in.src_index = in.slot_len = nullptr;
    in.val = nullptr;
}

#define LAUNCH(kernel, n, ...)                                                \
    do {                                                                      \
        hipLaunchKernelGGL(kernel, grid_for((n), kThreads), dim3(kThreads), 0, \
                           ctx->stream, __VA_ARGS__);                         \
        SMAX_HIP_LAUNCHED(ctx, #kernel);                                      \
    } while (0)

// Slots of every sigma window in std::sort's order: slot_row, slot_len and
// perm.  A failed partition is counted in *errors (device, zero on entry).
int sell_sort_windows(smax_hip_ctx ctx, int64_t n, int64_t n_rows, int64_t sigma,
                      const int32_t *row_ptr, int32_t *slot_row, int32_t *slot_len,
                      int32_t *perm, int64_t *errors, Scratch &S) {
    if (sigma <= kTile) {
        const int64_t span = kTile / sigma * sigma;
        hipLaunchKernelGGL(k_sort_tiles<true>, grid_for(n, static_cast<int>(span)),
                           dim3(kTileThreads), 0, ctx->stream, n, n_rows, sigma, span, row_ptr,
                           nullptr, nullptr, nullptr, nullptr, nullptr, slot_row, slot_len, perm,
                           errors);
        SMAX_HIP_LAUNCHED(ctx, "k_sort_tiles");
        return SMAX_HIP_SUCCESS;
    }
    int32_t *idx, *cnt, *idx2, *cnt2, *head, *end, *depth, *state;
    int32_t *pv, *sw, *cut, *PL, *SR, *posL, *posR, *listA, *listB, *tmp;
    int64_t *nlist;
    const int64_t nlist_cap = n / (kParked + 1) + 2;
    int rc = 0;
    rc |= S.get(ctx, &idx, n, "sell sort");
    rc |= S.get(ctx, &cnt, n, "sell sort");
    rc |= S.get(ctx, &idx2, n, "sell sort");
    rc |= S.get(ctx, &cnt2, n, "sell sort");
    rc |= S.get(ctx, &head, n, "sell sort");
    rc |= S.get(ctx, &end, n, "sell sort");
    rc |= S.get(ctx, &depth, n, "sell sort");
    rc |= S.get(ctx, &state, n, "sell sort");
    rc |= S.get(ctx, &listA, nlist_cap, "sell sort");
    rc |= S.get(ctx, &listB, nlist_cap, "sell sort");
    rc |= S.get(ctx, &nlist, 1, "sell sort");
    if (rc) return SMAX_HIP_ERROR_OUT_OF_MEMORY;
    rc = smax_hip_zero(ctx, nlist, sizeof(int64_t));
    if (rc) return rc;
    const int64_t sig = sigma < n ? sigma : n;
    LAUNCH(k_init, n, n, n_rows, sig, row_ptr, idx, cnt, head, end, depth,
           state, listA, nlist);
    int64_t nl = 0;
    rc = read_i64(ctx, nlist, &nl);
    if (rc) return rc;
    if (nl > 0) {
        rc |= S.get(ctx, &pv, n, "sell sort");
        rc |= S.get(ctx, &sw, n, "sell sort");
        rc |= S.get(ctx, &cut, n, "sell sort");
        rc |= S.get(ctx, &PL, n, "sell sort");
        rc |= S.get(ctx, &SR, n, "sell sort");
        rc |= S.get(ctx, &posL, n, "sell sort");
        rc |= S.get(ctx, &posR, n, "sell sort");
        rc |= S.get(ctx, &tmp, scan_tmp_elems(n), "sell sort");
        if (rc) return SMAX_HIP_ERROR_OUT_OF_MEMORY;
    }
    int level = 0;
    while (nl > 0) {
        if (++level > 200)
            return fail(ctx, SMAX_HIP_ERROR_RUNTIME,
                        "sell sort: recursion did not terminate");
        LAUNCH(k_pivot, nl, nl, listA, end, depth, state, idx, cnt, pv, sw);
        LAUNCH(k_flags, n, n, head, state, cnt, pv, PL, SR);
        rc = scan_inclusive<int32_t, false>(ctx, PL, PL, n, tmp);
        if (rc) return rc;
        rc = scan_inclusive<int32_t, true>(ctx, SR, SR, n, tmp);
        if (rc) return rc;
        LAUNCH(k_rank, n, n, head, state, end, cnt, pv, PL, SR, posL, posR, sw);
        LAUNCH(k_cut, nl, nl, listA, state, end, PL, posL, posR, sw, cut, errors);
        LAUNCH(k_move, n, n, head, state, end, pv, sw, PL, SR, posL, posR, idx,
               cnt, idx2, cnt2);
        std::swap(idx, idx2);
        std::swap(cnt, cnt2);
        LAUNCH(k_split, n, n, head, state, cut);
        rc = smax_hip_zero(ctx, nlist, sizeof(int64_t));
        if (rc) return rc;
        LAUNCH(k_newsegs, nl, nl, listA, state, end, depth, cut, listB, nlist);
        rc = read_i64(ctx, nlist, &nl);
        if (rc) return rc;
        std::swap(listA, listB);
    }
    LAUNCH(k_heapsort, n, n, n_rows, head, state, end, idx, cnt, slot_row, slot_len, perm);
    hipLaunchKernelGGL(k_sort_tiles<false>, grid_for(n, kParked), dim3(kTileThreads), 0,
                       ctx->stream, n, n_rows, sig, 0, nullptr, idx, cnt, head, end, depth,
                       slot_row, slot_len, perm, errors);
    SMAX_HIP_LAUNCHED(ctx, "k_sort_tiles");
    return SMAX_HIP_SUCCESS;
}

int build_scs(smax_hip_ctx ctx, int64_t n_rows, int64_t n_cols, int64_t nnz,
              const int32_t *row_ptr, const int32_t *col, const void *val,
              int64_t val_bytes, const int32_t *src_map, int64_t C,
              int64_t sigma, smax_hip_scs *out) {
    SMAX_HIP_REQUIRE(ctx, out, "scs conversion: null output");
    *out = nullptr;
    SMAX_HIP_REQUIRE(ctx, n_rows > 0 && n_cols > 0 && nnz >= 0,
                     "scs conversion: bad shape (%lld x %lld, nnz %lld)",
                     (long long)n_rows, (long long)n_cols, (long long)nnz);
    SMAX_HIP_REQUIRE(ctx, C > 0 && sigma > 0,
                     "scs conversion: C and sigma must be positive");
    SMAX_HIP_REQUIRE(ctx, val_bytes == 2 || val_bytes == 4 || val_bytes == 8,
                     "scs conversion: val_bytes must be 2, 4 or 8");
    SMAX_HIP_REQUIRE(ctx, row_ptr && (nnz == 0 || (col && val)),
                     "scs conversion: null input array");
    if (n_rows > INT32_MAX || n_cols > INT32_MAX || C > INT32_MAX || nnz > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "scs conversion: %lld x %lld, C = %lld or %lld entries exceed int32",
                    (long long)n_rows, (long long)n_cols, (long long)C, (long long)nnz);
    const int64_t n_chunks = ceil_div(n_rows, C);
    const int64_t n = n_chunks * C;
    if (n > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "scs conversion: %lld padded rows exceed int32",
                    (long long)n);
    Scratch S(ctx);
    int rc = 0;
    smax_hip_scs_info info{};
    info.C = C;
    info.sigma = sigma;
    info.n_rows = n_rows;
    info.n_rows_padded = n;
    info.n_cols = n_cols;
    info.n_chunks = n_chunks;
    info.nnz = nnz;
    info.val_bytes = val_bytes;
    struct Guard {
        smax_hip_ctx ctx;
        smax_hip_scs_info *p;
        bool keep = false;
        smax_hip_scs_longs *longs;
        ~Guard() {
            if (keep) return;
            (void)hipStreamSynchronize(ctx->stream);
            scs_free_arrays(*p);
            dev_free(longs->list);
        }
    };
    smax_hip_scs_longs longs;
    const int64_t from = long_slot_from(nnz, n_rows);
    longs.from = static_cast<int32_t>(from <= INT32_MAX ? from : INT32_MAX);
    longs.cap = nnz / longs.from + 1;
    Guard guard{ctx, &info, false, &longs};

    // words: sort errors, SELL elements, long slots (two counts)
    int64_t *elems, *incl, *tmp64, *words;
    rc |= S.get(ctx, &words, 4, "scs conversion");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&longs.list), sizeof(int32_t) * longs.cap,
                    "scs long slots");
    rc |= S.get(ctx, &elems, n_chunks, "scs conversion");
    rc |= S.get(ctx, &incl, n_chunks, "scs conversion");
    rc |= S.get(ctx, &tmp64, scan_tmp_elems(n_chunks), "scs conversion");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.chunk_lengths),
                    sizeof(int32_t) * n_chunks, "scs chunk_lengths");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.chunk_ptr),
                    sizeof(int32_t) * (n_chunks + 1), "scs chunk_ptr");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.perm),
                    sizeof(int32_t) * n_rows, "scs perm");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.slot_row),
                    sizeof(int32_t) * n, "scs slot_row");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.slot_len),
                    sizeof(int32_t) * n, "scs slot_len");
    if (rc) return SMAX_HIP_ERROR_OUT_OF_MEMORY;

    rc = smax_hip_zero(ctx, words, 4 * sizeof(int64_t));
    if (!rc)
        rc = sell_sort_windows(ctx, n, n_rows, sigma, row_ptr, info.slot_row, info.slot_len,
                               info.perm, words, S);
    if (rc) return rc;
    LAUNCH(k_chunk_len, n_chunks, n_chunks, C, info.slot_len, info.chunk_lengths, elems);
    rc = scan_inclusive<int64_t, false>(ctx, elems, incl, n_chunks, tmp64);
    if (rc) return rc;
    LAUNCH(k_chunk_ptr, n_chunks + 1, n_chunks, incl, info.chunk_ptr, words + 1);
    LAUNCH(k_long_slots, n, n, longs.from, info.slot_len, longs.list, longs.cap, words + 2);
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(ctx->host_word, words, 4 * sizeof(int64_t),
                                      hipMemcpyDeviceToHost, ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    if (ctx->host_word[0])
        return fail(ctx, SMAX_HIP_ERROR_RUNTIME,
                    "sell sort: %lld partitions produced an invalid cut",
                    static_cast<long long>(ctx->host_word[0]));
    const int64_t n_elements = ctx->host_word[1];
    longs.rows.whole = ctx->host_word[2];
    longs.rows.count = longs.rows.whole + ctx->host_word[3];
    if (n_elements > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW,
                    "scs conversion: %lld SELL elements exceed int32 chunk_ptr",
                    (long long)n_elements);
    info.n_elements = n_elements;

    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.col),
                    sizeof(int32_t) * n_elements, "scs col");
    rc |= dev_alloc(ctx, &info.val, val_bytes * n_elements, "scs val");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.src_index),
                    sizeof(int32_t) * n_elements, "scs src_index");
    if (rc) return SMAX_HIP_ERROR_OUT_OF_MEMORY;
    if (n_elements > 0) {
#define SMAX_FILL(V)                                                                        \
    hipLaunchKernelGGL(k_fill<V>, grid_for(n_elements, 256 * kFillItems), dim3(256), 0,     \
                       ctx->stream, n_elements, n_chunks, n_rows, static_cast<int32_t>(C),  \
                       fast_div(C), row_ptr, col, static_cast<const V *>(val), src_map,     \
                       info.chunk_ptr, info.slot_row, info.slot_len, info.col,              \
                       static_cast<V *>(info.val), info.src_index)
        switch (val_bytes) {
        case 8: SMAX_FILL(uint64_t); break;
        case 4: SMAX_FILL(uint32_t); break;
        default: SMAX_FILL(uint16_t); break;
        }
#undef SMAX_FILL
        SMAX_HIP_LAUNCHED(ctx, "k_fill");
    }
    // Scratch is released on return; wait so it is not freed under the GPU.
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    smax_hip_scs scs = new smax_hip_scs_s();
    scs->info = info;
    scs->longs = longs;
    scs->src_consecutive = src_map == nullptr;
    guard.keep = true;
    rc = build_schedule(ctx, C, sigma, n, n_chunks, n_elements, nnz, info.chunk_lengths,
                        &scs->sched, info.slot_row);
    if (!rc) rc = build_tails(ctx, scs);
    if (rc) {
        smax_hip_scs_destroy(ctx, scs);
        return rc;
    }
    *out = scs;
    return SMAX_HIP_SUCCESS;
}

int build_scs_from_sell(smax_hip_ctx ctx, int64_t C, int64_t sigma, int64_t n_rows,
                        int64_t n_rows_padded, int64_t n_cols, int64_t n_chunks,
                        int64_t n_elements, int64_t nnz, const int32_t *chunk_ptr,
                        const int32_t *chunk_lengths, const int32_t *col, const void *val,
                        int64_t val_bytes, const int32_t *perm, smax_hip_scs *out) {
    SMAX_HIP_REQUIRE(ctx, out, "smax_hip_scs_from_sell: null output");
    *out = nullptr;
    // n_rows_padded == n_chunks * C, tested without forming the product
    SMAX_HIP_REQUIRE(ctx, C > 0 && sigma > 0 && n_chunks > 0 && n_rows_padded % C == 0 &&
                              n_rows_padded / C == n_chunks && n_rows > 0 &&
                              n_rows <= n_rows_padded && n_cols > 0 && n_elements >= 0 &&
                              nnz >= 0 && nnz <= n_elements,
                     "smax_hip_scs_from_sell: inconsistent sizes");
    SMAX_HIP_REQUIRE(ctx, val_bytes == 2 || val_bytes == 4 || val_bytes == 8,
                     "smax_hip_scs_from_sell: val_bytes must be 2, 4 or 8");
    SMAX_HIP_REQUIRE(ctx, chunk_ptr && chunk_lengths && perm && (n_elements == 0 || (col && val)),
                     "smax_hip_scs_from_sell: null array");
    if (n_rows_padded > INT32_MAX || n_elements > INT32_MAX)
        return fail(ctx, SMAX_HIP_ERROR_OVERFLOW, "smax_hip_scs_from_sell: sizes exceed int32");
    smax_hip_scs_info info{};
    info.C = C;
    info.sigma = sigma;
    info.n_rows = n_rows;
    info.n_rows_padded = n_rows_padded;
    info.n_cols = n_cols;
    info.n_chunks = n_chunks;
    info.n_elements = n_elements;
    info.nnz = nnz;
    info.val_bytes = val_bytes;
    struct Guard {
        smax_hip_ctx ctx;
        smax_hip_scs_info *p;
        bool keep = false;
        ~Guard() {
            if (keep) return;
            (void)hipStreamSynchronize(ctx->stream);
            scs_free_arrays(*p);
        }
    } guard{ctx, &info};
    Scratch S(ctx);
    int32_t *bad = nullptr;
    int rc = S.get(ctx, &bad, 1, "scs adoption");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.chunk_ptr),
                    sizeof(int32_t) * (n_chunks + 1), "scs chunk_ptr");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.chunk_lengths),
                    sizeof(int32_t) * n_chunks, "scs chunk_lengths");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.col),
                    sizeof(int32_t) * (n_elements > 0 ? n_elements : 1), "scs col");
    rc |= dev_alloc(ctx, &info.val, val_bytes * (n_elements > 0 ? n_elements : 1), "scs val");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.perm), sizeof(int32_t) * n_rows,
                    "scs perm");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.slot_row),
                    sizeof(int32_t) * n_rows_padded, "scs slot_row");
    rc |= dev_alloc(ctx, reinterpret_cast<void **>(&info.slot_len),
                    sizeof(int32_t) * n_rows_padded, "scs slot_len");
    if (rc) return SMAX_HIP_ERROR_OUT_OF_MEMORY;
    const auto d2d = [&](void *dst, const void *src, size_t bytes) {
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream);
    };
    SMAX_HIP_CALL(ctx, d2d(info.chunk_ptr, chunk_ptr, sizeof(int32_t) * (n_chunks + 1)));
    SMAX_HIP_CALL(ctx, d2d(info.chunk_lengths, chunk_lengths, sizeof(int32_t) * n_chunks));
    if (n_elements > 0) {
        SMAX_HIP_CALL(ctx, d2d(info.col, col, sizeof(int32_t) * n_elements));
        SMAX_HIP_CALL(ctx, d2d(info.val, val, val_bytes * n_elements));
    }
    SMAX_HIP_CALL(ctx, d2d(info.perm, perm, sizeof(int32_t) * n_rows));
    LAUNCH(k_fill_i32, 1, 1, 0, bad);
    LAUNCH(k_check_sell_chunks, n_chunks + 1, n_chunks, C, n_elements, info.chunk_ptr,
           info.chunk_lengths, bad);
    int32_t h_bad = 0;
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(&h_bad, bad, sizeof(int32_t), hipMemcpyDeviceToHost,
                                      ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    if (h_bad)
        return fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                    "smax_hip_scs_from_sell: chunk_ptr does not match C * chunk_lengths "
                    "(or chunk_ptr[n_chunks] != n_elements)");
    if (n_elements > 0)
        LAUNCH(k_check_sell_cols, n_elements, n_elements, n_cols, info.col, bad);
    LAUNCH(k_fill_i32, n_rows_padded, n_rows_padded, static_cast<int32_t>(n_rows),
           info.slot_row);
    LAUNCH(k_slot_row_from_perm, n_rows, n_rows, n_rows_padded, info.perm, info.slot_row, bad);
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(&h_bad, bad, sizeof(int32_t), hipMemcpyDeviceToHost,
                                      ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    if (h_bad)
        return fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                    "smax_hip_scs_from_sell: a column index lies outside [0, n_cols) or a perm "
                    "entry outside [0, n_rows_padded)");
    LAUNCH(k_check_perm, n_rows, n_rows, info.perm, info.slot_row, bad);
    switch (val_bytes) {
    case 8:
        LAUNCH(k_sell_slot_len<uint64_t>, n_rows_padded, n_rows_padded, C, info.chunk_ptr,
               info.chunk_lengths, info.col, static_cast<const uint64_t *>(info.val),
               info.slot_len);
        break;
    case 4:
        LAUNCH(k_sell_slot_len<uint32_t>, n_rows_padded, n_rows_padded, C, info.chunk_ptr,
               info.chunk_lengths, info.col, static_cast<const uint32_t *>(info.val),
               info.slot_len);
        break;
    default:
        LAUNCH(k_sell_slot_len<uint16_t>, n_rows_padded, n_rows_padded, C, info.chunk_ptr,
               info.chunk_lengths, info.col, static_cast<const uint16_t *>(info.val),
               info.slot_len);
        break;
    }
    SMAX_HIP_CALL(ctx, hipMemcpyAsync(&h_bad, bad, sizeof(int32_t), hipMemcpyDeviceToHost,
                                      ctx->stream));
    SMAX_HIP_CALL(ctx, hipStreamSynchronize(ctx->stream));
    if (h_bad)
        return fail(ctx, SMAX_HIP_ERROR_INVALID_VALUE,
                    "smax_hip_scs_from_sell: perm maps two rows to one slot");
    smax_hip_scs scs = new smax_hip_scs_s();
    scs->info = info;
    scs->from_sell = true;
    guard.keep = true;
    rc = build_schedule(ctx, C, sigma, n_rows_padded, n_chunks, n_elements, nnz,
                        info.chunk_lengths, &scs->sched, info.slot_row);
    if (!rc) rc = build_tails(ctx, scs);
    if (rc) {
        smax_hip_scs_destroy(ctx, scs);
        return rc;
    }
    *out = scs;
    return SMAX_HIP_SUCCESS;
}

}  // namespace smaxhip

using namespace smaxhip;

extern "C" {

int smax_hip_scs_from_sell(smax_hip_ctx ctx, int64_t C, int64_t sigma, int64_t n_rows,
                           int64_t n_rows_padded, int64_t n_cols, int64_t n_chunks,
                           int64_t n_elements, int64_t nnz, const int32_t *chunk_ptr,
                           const int32_t *chunk_lengths, const int32_t *col, const void *val,
                           int64_t val_bytes, const int32_t *perm, smax_hip_scs *out) {
    SMAX_HIP_CHECK_CTX(ctx);
    return build_scs_from_sell(ctx, C, sigma, n_rows, n_rows_padded, n_cols, n_chunks,
                               n_elements, nnz, chunk_ptr, chunk_lengths, col, val, val_bytes,
                               perm, out);
}

int smax_hip_scs_from_crs(smax_hip_ctx ctx, int64_t n_rows, int64_t n_cols,
                          int64_t nnz, const int32_t *row_ptr,
                          const int32_t *col, const void *val,
                          int64_t val_bytes, int64_t C, int64_t sigma,
                          smax_hip_scs *out) {
    SMAX_HIP_CHECK_CTX(ctx);
    return build_scs(ctx, n_rows, n_cols, nnz, row_ptr, col, val, val_bytes,
                     nullptr, C, sigma, out);
}

int smax_hip_scs_get_info(smax_hip_scs scs, smax_hip_scs_info *info) {
    if (!scs || !info)
        return fail(nullptr, SMAX_HIP_ERROR_INVALID_VALUE,
                    "smax_hip_scs_get_info: null argument");
    *info = scs->info;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_scs_destroy(smax_hip_ctx ctx, smax_hip_scs scs) {
    if (!scs) return SMAX_HIP_SUCCESS;
    if (ctx) {
        (void)bind(ctx);
        (void)hipStreamSynchronize(ctx->stream);
    }
    scs_free_arrays(scs->info);
    dev_free(scs->col_slot);
    dev_free(scs->col_rel);
    dev_free(scs->col_idx);
    dev_free(scs->col_idx_row);
    dev_free(scs->col_tab);
    dev_free(scs->val_f32);
    dev_free(scs->val_bf16);
    dev_free(scs->diag_f32);
    free_schedule(scs->sched);
    free_tails(scs->tails);
    dev_free(scs->longs.list);
    dev_free(scs->elem_row);
    delete scs;
    return SMAX_HIP_SUCCESS;
}

int smax_hip_scs_refresh_values(smax_hip_ctx ctx, smax_hip_scs scs,
                                const void *crs_val) {
    SMAX_HIP_CHECK_CTX(ctx);
    SMAX_HIP_REQUIRE(ctx, scs && crs_val, "smax_hip_scs_refresh_values: null");
    SMAX_HIP_REQUIRE(ctx, !scs->from_sell,
                     "smax_hip_scs_refresh_values: the handle was built from SELL arrays and "
                     "has no CRS positions; build it with smax_hip_scs_from_crs");
    const smax_hip_scs_info &in = scs->info;
    const int64_t m = in.n_elements;
    // the solvers' rounded copies follow the old values: drop them (rebuilt
    // on the next solve); without copies the refresh stays asynchronous
    if (scs->val_f32 || scs->val_bf16 || scs->diag_f32) {
        (void)hipStreamSynchronize(ctx->stream);
        for (void **p : {reinterpret_cast<void **>(&scs->val_f32),
                         reinterpret_cast<void **>(&scs->val_bf16),
                         reinterpret_cast<void **>(&scs->diag_f32)}) {
            dev_free(*p);
            *p = nullptr;
        }
        scs->bf16_split = -1;
    }
    if (m == 0) return SMAX_HIP_SUCCESS;
    const bool stream = scs->tails.n_blocks == 0;
    int rc;
    switch (in.val_bytes) {
    case 8: rc = launch_refresh<uint64_t>(ctx, m, in.src_index, crs_val, in.val, stream); break;
    case 4: rc = launch_refresh<uint32_t>(ctx, m, in.src_index, crs_val, in.val, stream); break;
    default: rc = launch_refresh<uint16_t>(ctx, m, in.src_index, crs_val, in.val, stream); break;
    }
    if (rc) return rc;
    // the tail waves hold copies of their slots' values
    return refresh_tail_values(ctx, scs);
}

}  // extern "C"
