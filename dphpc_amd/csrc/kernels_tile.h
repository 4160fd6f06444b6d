// Dense-tile path: 16-row strips of S whose 16x16 tiles are well filled are
// computed on the matrix cores, one MFMA accumulator per tile, instead of one
// gathered B row per stored entry.
//
//   * a strip is rows [16*ti, 16*ti+16); a tile is the strip's entries whose
//     column lies in [16*tj, 16*tj+16);
//   * the classifier (k_own_rows / k_strip_tiles / k_tile_rows, plan phase,
//     device only) finds the non-empty tiles of every strip and emits one TileDesc
//     per tile: for every row the CSR position of its first entry inside the tile
//     and a 16-bit mask of the columns present;
//   * a strip goes to this path as a whole (then every one of its entries is
//     computed here, sparse tiles included) or not at all, so the gather kernels
//     and this one never share a row;
//   * k_tile computes the full 16x16 product A[strip rows] * B[tile cols]^T with
//     fp32 accumulation (bf16 / fp16: v_mfma_f32_16x16x32_bf16 / _f16, fp32: v_mfma_f32_16x16x4_f32,
//     both exact products of the stored inputs), multiplies by the S values and
//     writes only the positions the masks name -- P keeps S's order.
//
// The B tile costs 16 rows per tile whatever its fill, a gathered entry costs one
// row each: the tile path moves fewer bytes once a tile holds more than 16
// entries, and far fewer at the 25-100 % fill it is used for.
#pragma once
#include "device_utils.h"
#include "kernels_gather.h"
#include "kernels_plan.h"

namespace sddmm {

struct alignas(16) TileDesc {
    int32_t strip;      // 16-row strip index
    int32_t tj;         // tile column: columns [16*tj, 16*tj+16)
    int32_t pad[2];
    int32_t off[16];    // per row: CSR position of the row's first entry in the tile
    uint16_t mask[16];  // per row: bit c set <=> column 16*tj+c is stored
};
static_assert(sizeof(TileDesc) == 112, "TileDesc layout");

// Walks the tiles of one strip in increasing tile column.  All 16 lanes of the
// strip call on_tile(tj, first, mask) together; `first` / `mask` are this lane's
// row's first position and column mask in the tile (mask 0: row absent).  The walk
// stops early when on_tile returns false (it must return the same in all 16 lanes).
// Returns false in a lane whose row is not strictly increasing in column.
template <class F>
__device__ __forceinline__ bool walk_strip(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M,
                                           int64_t strip, int sub, F &&on_tile) {
    const int64_t row = strip * 16 + sub;
    int p = 0, end = 0;
    if (row < M) { p = rowptr[row]; end = rowptr[row + 1]; }
    bool sorted = true;
    int prev = -1;
    // The row is read 8 column indices at a time (two 16-byte loads, clamped to the
    // row's last entry), so the walk is not one dependent load per entry.
    int buf[8];
    int buf_at = p;                       // buf[i] = col[min(buf_at + i, end - 1)]
    auto refill = [&](int at) {
        buf_at = at;
        if (at < end) {
            const int last = end - 1;
            if (at + 7 <= last) {
                const I4u lo = *reinterpret_cast<const I4u *>(col + at);
                const I4u hi = *reinterpret_cast<const I4u *>(col + at + 4);
                buf[0] = lo.x; buf[1] = lo.y; buf[2] = lo.z; buf[3] = lo.w;
                buf[4] = hi.x; buf[5] = hi.y; buf[6] = hi.z; buf[7] = hi.w;
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) buf[i] = col[at + i < last ? at + i : last];
            }
        }
    };
    auto peek = [&](int at) {             // col[at] for buf_at <= at < buf_at + 8
        const int i = at - buf_at;
        int v = buf[0];
#pragma unroll
        for (int k = 1; k < 8; ++k) v = i == k ? buf[k] : v;
        return v;
    };
    refill(p);
    int c = p < end ? peek(p) : -1;
    while (true) {
        const int mine = p < end ? (c >> 4) : INT32_MAX;
        const int t = min16(mine);
        if (t == INT32_MAX) break;
        const int first = p;
        unsigned int mask = 0;
        while (p < end && (c >> 4) == t) {
            if (c <= prev) sorted = false;
            prev = c;
            mask |= 1u << (c & 15);
            ++p;
            if (p - buf_at >= 8) refill(p);
            c = p < end ? peek(p) : -1;
        }
        if (!on_tile(t, first, mask)) break;
    }
    return sorted;
}

// Every tile lists its 16 B rows (tile_cols, 16 per descriptor, ascending; INT32_MAX
// where a union tile has fewer): consecutive columns for the aligned tiles.
__device__ __forceinline__ void write_aligned_cols(int32_t *__restrict__ tile_cols, int64_t at, int tj) {
    int4 *dst = reinterpret_cast<int4 *>(tile_cols + at * 16);
    const int c0 = tj * 16;
    dst[0] = make_int4(c0, c0 + 1, c0 + 2, c0 + 3);
    dst[1] = make_int4(c0 + 4, c0 + 5, c0 + 6, c0 + 7);
    dst[2] = make_int4(c0 + 8, c0 + 9, c0 + 10, c0 + 11);
    dst[3] = make_int4(c0 + 12, c0 + 13, c0 + 14, c0 + 15);
}

// ---- parallel strip classifier ---------------------------------------------------
// One wavefront per strip, four strips per workgroup.  The strip's entries are
// contiguous in the CSR arrays, so the wave streams them 64 per load, several
// loads in flight, instead of merging 16 sorted lists entry by entry:
//
//   * walking the entries in storage order, the tile column changes at least once
//     per (row, tile) pair minus the 15 row boundaries, and a strip has at least
//     (pairs / 16) tiles: the number of changes bounds the tile count from below
//     without any merging, and the scan stops as soon as that bound exceeds what
//     the fill threshold allows (a strip of scattered entries is given up after
//     its first few hundred);
//   * the same scan marks the tile column after every change in a bitmap in LDS
//     that covers the strip's column span -- every tile present is marked at least
//     once; the number of set bits is the number of tiles, the rank of a bit the
//     position of its tile in the strip's (column-ordered) descriptor range;
//   * rows are strictly increasing iff the only places where a column does not
//     exceed its predecessor are row boundaries: the scan counts all such places,
//     the 16 row starts are checked apart;
//   * a strip whose span does not fit the bitmap is scanned without it and, if it
//     passes, merged by the walk above in its first 16 lanes.
//
// The bitmap is private to its wave: LDS operations of one wave execute in program
// order, so clearing, marking and counting need no workgroup barrier, only that
// the compiler keeps their order (wave_lds_order).
constexpr int STRIP_BM_WORDS = 1024;          // 32768 tile columns: a span of 524288 columns
constexpr int STRIP_UNROLL = 4;               // loads of 256 entries per batch, two batches in flight
constexpr int STRIPS_PER_BLOCK = 4;

// N * 256 entries from base on, four per lane and load; past e1 the last one, or anything in whole loads past it.
constexpr int PER_LOAD = WAVE * 4;
template <int N>
__device__ __forceinline__ void load_entries(const int32_t *__restrict__ col, int base, int e1, I4u (&c)[N]) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int b = base + u * PER_LOAD, i0 = b + 4 * lane_id(), last = e1 - 1;
        if (b + PER_LOAD <= e1) {                                 // wave-uniform: every lane's four entries exist
            c[u] = *reinterpret_cast<const I4u *>(col + i0);
        } else if (b < e1 || u == 0) {                            // the last load: clamped, entry by entry
            c[u].x = col[i0 < last ? i0 : last];
            c[u].y = col[i0 + 1 < last ? i0 + 1 : last];
            c[u].z = col[i0 + 2 < last ? i0 + 2 : last];
            c[u].w = col[i0 + 3 < last ? i0 + 3 : last];
        } else {
            c[u] = I4u{0, 0, 0, 0};
        }
    }
}

// Streams entries [e0, e1).  Returns the number of tile-column changes, or -1 as
// soon as it exceeds `budget`; *descents receives the number of entries whose
// column does not exceed the column stored before them.  BITS == 1: also sets bit
// (col>>4) - lo in bm after every change (tile columns); BITS == 2: sets bit col - lo
// for every entry (columns).
// A lane takes four consecutive entries per load (16 bytes; the column array is only
// 4-byte aligned at a strip's start, which global loads allow), a load instruction 256
// entries, a batch STRIP_UNROLL of them with the next batch in flight: a strip of 8 000
// entries is eight dependent round trips.
template <int BITS>
__device__ __forceinline__ int64_t strip_scan(const int32_t *__restrict__ col, int e0, int e1, int64_t budget,
                                              int lo, int span, unsigned int *bm, int64_t *descents) {
    const int lane = lane_id();
    constexpr int BATCH = PER_LOAD * STRIP_UNROLL;
    int64_t changes = 0, desc = 0;
    int carry = -1;                           // column before the batch; -1: entry e0 counts as a change
    auto mark = [&](bool on, int column) {
        if constexpr (BITS == 1) {
            const int t = (column >> 4) - lo;
            if (on && (unsigned int)t < (unsigned int)span) atomicOr(&bm[t >> 5], 1u << (t & 31));
        } else if constexpr (BITS == 2) {
            const int t = column - lo;
            if (on && (unsigned int)t < (unsigned int)span) atomicOr(&bm[t >> 5], 1u << (t & 31));
        }
    };
    I4u cur[STRIP_UNROLL], nxt[STRIP_UNROLL];
    load_entries(col, e0, e1, cur);
    for (int base = e0; base < e1; base += BATCH) {
        load_entries(col, base + BATCH, e1, nxt);
        int my_changes = 0, my_desc = 0;
#pragma unroll
        for (int u = 0; u < STRIP_UNROLL; ++u) {
            const int cbase = base + u * PER_LOAD;
            if (cbase >= e1) break;                               // wave-uniform
            const int i0 = cbase + 4 * lane;
            const I4u c = cur[u];
            // column of the entry before this lane's first: the last of lane - 1 (wave_shr:1), lane 0 takes the carry
            const int prev = __builtin_amdgcn_update_dpp(carry, c.w, 0x138, 0xF, 0xF, false);
            carry = __builtin_amdgcn_readlane(c.w, WAVE - 1);
            const bool v0 = i0 < e1, v1 = i0 + 1 < e1, v2 = i0 + 2 < e1, v3 = i0 + 3 < e1;
            const bool c0 = v0 && (c.x >> 4) != (prev >> 4), c1 = v1 && (c.y >> 4) != (c.x >> 4);
            const bool c2 = v2 && (c.z >> 4) != (c.y >> 4), c3 = v3 && (c.w >> 4) != (c.z >> 4);
            if constexpr (BITS == 1) { mark(c0, c.x); mark(c1, c.y); mark(c2, c.z); mark(c3, c.w); }
            if constexpr (BITS == 2) { mark(v0, c.x); mark(v1, c.y); mark(v2, c.z); mark(v3, c.w); }
            my_changes += (int)c0 + (int)c1 + (int)c2 + (int)c3;
            my_desc += (int)(v0 && c.x <= prev) + (int)(v1 && c.y <= c.x) + (int)(v2 && c.z <= c.y) + (int)(v3 && c.w <= c.z);
        }
        changes += wave_sum_i32(my_changes);
        desc += wave_sum_i32(my_desc);
        if (changes > budget) return -1;
#pragma unroll
        for (int u = 0; u < STRIP_UNROLL; ++u) cur[u] = nxt[u];
    }
    *descents = desc;
    return changes;
}

// From the first and last entry of each of the 16 rows (lane i < 16: row i, whose
// rowptr is lane_rp): the strip's column span in tile columns (SHIFT 4) or columns
// (SHIFT 0), [lo, lo + span)
// (exact when the rows are sorted; span <= 0 when they are not or no row has an
// entry), and the number of row starts whose column does not exceed the column
// stored before them -- the descents a sorted strip is allowed.
template <int SHIFT = 4>
__device__ __forceinline__ void strip_bounds(const int32_t *__restrict__ col, int lane_rp, int e0, int *lo, int *span,
                                             int *boundary_descents) {
    const int lane = lane_id();
    const int nxt = __shfl_down(lane_rp, 1, WAVE);
    const bool has = lane < 16 && nxt > lane_rp;
    const int first_col = has ? col[lane_rp] : INT32_MAX;
    const int last_col = has ? col[nxt - 1] : -1;
    const int before = has && lane_rp > e0 ? col[lane_rp - 1] : -1;
    const int l = __builtin_amdgcn_readfirstlane(min16(has ? first_col >> SHIFT : INT32_MAX));
    const int hneg = __builtin_amdgcn_readfirstlane(min16(has ? -(last_col >> SHIFT) : 1));
    *lo = l;
    *span = l == INT32_MAX ? 0 : -hneg - l + 1;
    *boundary_descents = __popcll(__ballot(has && first_col <= before));
}

// Number of tiles of a strip that goes to the tile path (sorted rows, at least min_fill entries per tile on average), else 0.
// bm: STRIP_BM_WORDS words of the wave's own.
__device__ __forceinline__ int strip_tiles_of(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M,
                                              int64_t strip, int lane_rp, int e0, int e1, int min_fill, unsigned int *bm) {
    const int lane = lane_id();
    const int64_t entries = (int64_t)e1 - (int64_t)e0;
    const int64_t max_tiles = entries / min_fill;
    // changes >= (row, tile) pairs - 15 and tiles >= pairs / 16
    const int64_t budget = 16 * max_tiles;
    int64_t tiles = 0, descents = 0;
    bool take = false;
    // most strips of a scattered matrix are given up on their first 512 entries,
    // before anything else is read
    constexpr int FIRST = 512;
    if (max_tiles > 0 &&
        strip_scan<0>(col, e0, e1 - e0 > FIRST ? e0 + FIRST : e1, budget, 0, 0, nullptr, &descents) >= 0) {
        int lo, span, allowed;
        strip_bounds(col, lane_rp, e0, &lo, &span, &allowed);
        if (span > STRIP_BM_WORDS * 32) {
            // too wide for the bitmap: scan without it, then merge the 16 rows in the first
            // 16 lanes if the strip is still a candidate
            const int64_t ch = strip_scan<0>(col, e0, e1, budget, 0, 0, nullptr, &descents);
            if (ch >= 0 && descents == allowed) {
                int t = 0;
                if (lane < 16) {
                    (void)walk_strip(rowptr, col, M, strip, lane, [&](int, int, unsigned int) {
                        ++t;
                        return (int64_t)t <= max_tiles;
                    });
                }
                tiles = __builtin_amdgcn_readfirstlane(t);
            }
        } else if (span > 0) {
            const int words = (span + 31) >> 5;
            for (int w = lane; w < words; w += WAVE) bm[w] = 0u;
            wave_lds_order();
            // Rows 0 and 8 first: their tile columns alone often exceed what the strip may have
            // (two 8-row blocks with different column lists), and the other 14 rows are then
            // never read.  The bits stay: the scan of the whole strip sets them again.
            int64_t ch = 0;
            if (entries > 4 * FIRST) {
                int64_t unused;
                const int a0 = e0, a1 = __builtin_amdgcn_readlane(lane_rp, 1);
                const int b0 = __builtin_amdgcn_readlane(lane_rp, 8), b1 = __builtin_amdgcn_readlane(lane_rp, 9);
                if (a1 > a0) (void)strip_scan<1>(col, a0, a1, INT64_MAX, lo, span, bm, &unused);
                if (b1 > b0) (void)strip_scan<1>(col, b0, b1, INT64_MAX, lo, span, bm, &unused);
                wave_lds_order();
                int t = 0;
                for (int w = lane; w < words; w += WAVE) t += __builtin_popcount(bm[w]);
                if (wave_sum_i32(t) > max_tiles) ch = -1;
            }
            if (ch >= 0) ch = strip_scan<1>(col, e0, e1, budget, lo, span, bm, &descents);
            wave_lds_order();
            if (ch >= 0 && descents == allowed) {
                int t = 0;
                for (int w = lane; w < words; w += WAVE) t += __builtin_popcount(bm[w]);
                tiles = wave_sum_i32(t);
            }
        }
        take = tiles > 0 && tiles <= max_tiles && entries >= (int64_t)min_fill * tiles;
    }
    return take ? (int)tiles : 0;
}

// The same by a workgroup of 16 wavefronts, a row each (every wavefront must call it; each answers for the whole strip).
// bm and flags (0, 0) are the workgroup's.
constexpr int WIDE_BLOCK = 16 * WAVE;
__device__ __forceinline__ int strip_tiles_of_wide(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M,
                                                   int64_t strip, int lane_rp, int e0, int e1, int min_fill, unsigned int *bm,
                                                   int *flags) {
    const int lane = lane_id(), wv = wave_in_block();
    const int64_t entries = (int64_t)e1 - (int64_t)e0, max_tiles = entries / min_fill, budget = 16 * max_tiles;
    if (max_tiles <= 0) return 0;
    int64_t descents = 0;
    int lo, span, allowed;
    strip_bounds(col, lane_rp, e0, &lo, &span, &allowed);
    if (span <= 0) return 0;
    if (span > STRIP_BM_WORDS * 32) {
        if (wv == 0) {
            const int tiles = strip_tiles_of(rowptr, col, M, strip, lane_rp, e0, e1, min_fill, bm);
            if (lane == 0) flags[1] = tiles;
        }
        __syncthreads();
        return flags[1];
    }
    const int words = (span + 31) >> 5;
    for (int w = (int)threadIdx.x; w < words; w += WIDE_BLOCK) bm[w] = 0u;
    __syncthreads();
    // (a row's tile columns change at most as often as the strip's, and its first entry has none before it)
    const int s = __builtin_amdgcn_readlane(lane_rp, wv), e = __builtin_amdgcn_readlane(lane_rp, wv + 1);
    if (e > s && (strip_scan<1>(col, s, e, budget, lo, span, bm, &descents) < 0 || descents != 0) && lane == 0) atomicOr(&flags[0], 1);
    __syncthreads();
    int t = 0;
    for (int w = (int)threadIdx.x; w < words; w += WIDE_BLOCK) t += __builtin_popcount(bm[w]);
    t = wave_sum_i32(t);
    if (lane == 0 && t) atomicAdd(&flags[1], t);
    __syncthreads();
    const int tiles = flags[1];
    return flags[0] == 0 && tiles <= max_tiles && entries >= (int64_t)min_fill * tiles ? tiles : 0;
}

// The descriptors of a strip too wide for a bitmap, by the merging walk in a wavefront's first 16 lanes.
__device__ __forceinline__ void walk_descriptors(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M, int64_t strip,
                                                 int64_t at, TileDesc *__restrict__ tiles, int32_t *__restrict__ tile_cols) {
    const int lane = lane_id();
    if (lane >= 16) return;
    (void)walk_strip(rowptr, col, M, strip, lane, [&](int tj, int first, unsigned int mask) {
        TileDesc *d = tiles + at;
        d->off[lane] = first;
        d->mask[lane] = (uint16_t)mask;
        if (lane == 0) { d->strip = (int32_t)strip; d->tj = tj; d->pad[0] = 1; d->pad[1] = 0; }
        tile_cols[at * 16 + lane] = tj * 16 + lane;
        ++at;
        return true;
    });
}

// pass 2 (after the exclusive scan of strip_ntiles into strip_off): strip and tile
// column of every descriptor, in increasing tile column.  Descriptors of a strip
// that needs the merging walk are written completely here (pad[0] = 1); the others
// get their per-row fields from k_tile_rows.
static __global__ __launch_bounds__(WAVE * STRIPS_PER_BLOCK) void k_strip_tiles(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M, int64_t n_strips,
    const unsigned int *__restrict__ strip_ntiles, const unsigned int *__restrict__ strip_off,
    TileDesc *__restrict__ tiles, int32_t *__restrict__ tile_cols) {
    __shared__ unsigned int bm_all[STRIPS_PER_BLOCK][STRIP_BM_WORDS];
    const int64_t strip = (int64_t)blockIdx.x * STRIPS_PER_BLOCK + wave_in_block();
    if (strip >= n_strips) return;
    if (strip_ntiles[strip] == 0) return;
    unsigned int *bm = bm_all[wave_in_block()];
    const int lane = lane_id();
    const int64_t r = strip * 16 + lane;
    const int lane_rp = rowptr[r < M ? r : M];
    const int e0 = __builtin_amdgcn_readlane(lane_rp, 0), e1 = __builtin_amdgcn_readlane(lane_rp, 16);
    int lo, span, allowed;
    strip_bounds(col, lane_rp, e0, &lo, &span, &allowed);
    const int64_t first_desc = strip_off[strip];
    if (span > STRIP_BM_WORDS * 32) {
        walk_descriptors(rowptr, col, M, strip, first_desc, tiles, tile_cols);
        return;
    }
    const int words = (span + 31) >> 5;
    for (int w = lane; w < words; w += WAVE) bm[w] = 0u;
    wave_lds_order();
    int64_t descents;
    (void)strip_scan<1>(col, e0, e1, INT64_MAX, lo, span, bm, &descents);
    wave_lds_order();
    int64_t run = first_desc;
    for (int wb = 0; wb < words; wb += WAVE) {
        const int w = wb + lane;
        unsigned int x = w < words ? bm[w] : 0u;
        const int n = __builtin_popcount(x);
        const int incl = wave_inclusive_sum(n);
        int64_t at = run + (incl - n);
        while (x) {
            const int b = __builtin_ctz(x);
            x &= x - 1;
            *reinterpret_cast<int4 *>(tiles + at) = make_int4((int)strip, lo + w * 32 + b, 0, 0);
            write_aligned_cols(tile_cols, at, lo + w * 32 + b);
            ++at;
        }
        run += __builtin_amdgcn_readlane(incl, WAVE - 1);
    }
}

// ---- union strips --------------------------------------------------------------------
// A 16-row strip whose rows are similar but not aligned to 16-column blocks (mesh
// rows that share most of their neighbours) wastes the aligned tiles: its columns are
// spread over many of them.  Here the strip's tiles are cut from the sorted UNION of
// its column lists instead, 16 union columns per tile, so a B row is gathered once
// for the rows of the strip that have it -- the role of the active-column lists of
// src/competitors/gpu/gpu_preprocessing.hpp:57-141.  Same machinery as above with a
// bitmap of columns instead of tile columns: popcount = size of the union, the rank
// of a column gives its tile and its position in the tile.
constexpr int UNION_BM_WORDS = 4096;          // a column span of 131072 per strip

__device__ __forceinline__ int max16(int v) { return -min16(-v); }

// descriptors of the union strips: header and the 16 union columns of every tile
static __global__ __launch_bounds__(WAVE * STRIPS_PER_BLOCK) void k_union_tiles(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M, int64_t n_strips,
    const unsigned int *__restrict__ ustrip_ntiles, const unsigned int *__restrict__ ustrip_off,
    TileDesc *__restrict__ tiles, int32_t *__restrict__ tile_cols) {
    __shared__ unsigned int bm_all[STRIPS_PER_BLOCK][UNION_BM_WORDS];
    const int64_t strip = (int64_t)blockIdx.x * STRIPS_PER_BLOCK + wave_in_block();
    if (strip >= n_strips) return;
    const unsigned int ntiles = ustrip_ntiles[strip];
    if (ntiles == 0) return;
    unsigned int *bm = bm_all[wave_in_block()];
    const int lane = lane_id();
    const int64_t r = strip * 16 + lane;
    const int lane_rp = rowptr[r < M ? r : M];
    const int e0 = __builtin_amdgcn_readlane(lane_rp, 0), e1 = __builtin_amdgcn_readlane(lane_rp, 16);
    int lo, span, allowed;
    strip_bounds<0>(col, lane_rp, e0, &lo, &span, &allowed);
    const int words = (span + 31) >> 5;
    for (int w = lane; w < words; w += WAVE) bm[w] = 0u;
    wave_lds_order();
    int64_t descents = 0;
    (void)strip_scan<2>(col, e0, e1, INT64_MAX, lo, span, bm, &descents);
    wave_lds_order();
    const int64_t first = ustrip_off[strip];
    int64_t run = 0;                              // union columns before this batch of words
    for (int wb = 0; wb < words; wb += WAVE) {
        const int w = wb + lane;
        unsigned int x = w < words ? bm[w] : 0u;
        const int n = __builtin_popcount(x);
        const int incl = wave_inclusive_sum(n);
        int64_t rank = run + (incl - n);
        while (x) {
            const int b = __builtin_ctz(x);
            x &= x - 1;
            const int c = lo + w * 32 + b;
            const int64_t t = first + (rank >> 4);
            tile_cols[t * 16 + (rank & 15)] = c;
            if ((rank & 15) == 0) *reinterpret_cast<int4 *>(tiles + t) = make_int4((int)strip, c >> 4, 0, 0);
            ++rank;
        }
        run += __builtin_amdgcn_readlane(incl, WAVE - 1);
    }
    // the last tile of the strip may hold fewer than 16 columns
    const int tail = (int)(run & 15);
    if (tail != 0 && lane >= tail && lane < 16) tile_cols[(first + ntiles - 1) * 16 + lane] = INT32_MAX;
}

// ---- gathered strips ---------------------------------------------------------------
// Rows that are dense inside a column window need not be neighbours to share tiles:
// any 16 rows whose windows overlap form a strip for the matrix cores as well as 16
// consecutive ones do.  Candidate rows (not owned yet, at least min_len entries that
// fill a quarter of their column span or more) are sorted by (first column, row) --
// one 64-bit key per row, so the order does not depend on the order of the appends;
// every 16 consecutive rows of that order are one gathered strip, classified with
// the same bitmap and threshold as a natural strip.  TileDesc.strip of such a strip
// is GATHERED_BASE + its index, its rows are listed in a table (16 per strip, -1 for
// a missing row).
constexpr int GATHERED_BASE = 1 << 30;
constexpr int TILE_WINDOW = 4;                  // descriptors per window (what a wavefront of the tile kernels takes)

// ---- who owns a row -----------------------------------------------------------------------
// The classifiers of a plan in one launch: a wavefront looks at a 16-row strip (dense tiles), then at its two 8-row panels;
// the workgroup looks together at those of its four strips that could be union strips (their bitmap takes the LDS of all
// four); the first wavefront then offers the rows that are left to the gathered strips and classifies them.  As five
// launches they read the row pointer five times and waited for each other (new pattern
// with every call: 36 000 banded rows 226 -> 188 us, 30 000 near-dense and short rows 199 -> 180).
struct OwnRules {
    int strip_fill, panel_min, union_fill, cand_min;     // 0: not looked for
    int panels_below;                                     // entries per tile from which a strip of two panels stays a strip
    int pseg;                                             // entries of a panel's work items
    int ts, seg;                                          // row classes (k_classify_count)
};
struct OwnArrays {
    unsigned char *owner;                                 // 1: strip, 2: panel, 4: union strip, 0: nobody
    unsigned int *strip_ntiles, *panel_counts, *ustrip_ntiles;
    unsigned long long *cand_keys;
    unsigned int *items, *short_entries, *long_rows;      // per block of the row scan, cleared
    unsigned int *either;                                 // tiles of a strip that is two panels as well, else 0
};

// 8 rows from row0 on with one column list?  (Equal lengths make them equally spaced in the CSR arrays: row r starts at
// s0 + r * len, so the 7 comparisons of one position are independent loads.)  Every parts-th 64 columns of it.
__device__ __forceinline__ bool same_lists(const int32_t *__restrict__ col, int s0, int len, int part = 0, int parts = 1) {
    bool differ = false;
    for (int e = part * WAVE + lane_id(); e < len; e += parts * WAVE) {
        const int32_t *at = col + s0 + e;
        const int c0 = at[0];
        int d = 0;
#pragma unroll
        for (int r = 1; r < 8; ++r) d |= at[(int64_t)r * len] ^ c0;
        differ |= d != 0;
    }
    return __ballot(differ) == 0;
}

// WIDE: a workgroup of 16 wavefronts per strip, where the strips are long and too few for the chip's wavefronts.  (A
// wavefront reads 1 024 entries per round trip: 35 strips of 33 000 entries 79 us, so 17.)
template <bool WIDE>
static __global__ __launch_bounds__(WIDE ? WIDE_BLOCK : WAVE * STRIPS_PER_BLOCK) void k_own_rows(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M, int64_t n_strips, int strips_per_wave,
    OwnRules rules, OwnArrays out, DevCounters *pc) {
    static_assert(STRIPS_PER_BLOCK == 4 && STRIPS_PER_BLOCK * STRIP_BM_WORDS == UNION_BM_WORDS, "one buffer for both bitmaps");
    constexpr int STRIPS = WIDE ? 1 : STRIPS_PER_BLOCK, WAVES = WIDE ? 16 : STRIPS_PER_BLOCK;
    __shared__ unsigned int bm_all[UNION_BM_WORDS];
    __shared__ int rp_of[STRIPS][17], own_of[STRIPS][16];
    __shared__ int lo_of[STRIPS], span_of[STRIPS], allowed_of[STRIPS];   // span 0: no union strip
    __shared__ int found, descents_found;
    __shared__ int flags[4];                                              // WIDE: strip_tiles_of_wide; lists of a half that differ
    const int lane = lane_id(), wv = wave_in_block(), tid = (int)threadIdx.x;
    const bool speaks = lane == 0 && (!WIDE || wv == 0);                  // for its strip
    if (WIDE) {
        if (tid < 4) flags[tid] = 0;
        __syncthreads();
    }
    unsigned int rows_sum[3] = {0, 0, 0}, entries_sum[3] = {0, 0, 0};      // wave 0: short, medium, long
    for (int g = 0; g < strips_per_wave; ++g) {
        const int64_t first = ((int64_t)blockIdx.x * strips_per_wave + g) * STRIPS;
        if (first >= n_strips) break;                                     // workgroup-uniform
        const int64_t strip = first + (WIDE ? 0 : wv), r = strip * 16 + lane;
        const int lane_rp = rowptr[r < M ? r : M];                        // (a strip past the last one has no entries)
        const int e0 = __builtin_amdgcn_readlane(lane_rp, 0), e1 = __builtin_amdgcn_readlane(lane_rp, 16);
        const int next_rp = __shfl_down(lane_rp, 1, WAVE);
        const int len = lane < 16 ? next_rp - lane_rp : 0;
        int owned = 0;                                                    // lane < 16: owner of its row
        int tiles = 0, items[2] = {0, 0};
        if (rules.strip_fill)
            tiles = WIDE ? strip_tiles_of_wide(rowptr, col, M, strip, lane_rp, e0, e1, rules.strip_fill, bm_all, flags)
                         : strip_tiles_of(rowptr, col, M, strip, lane_rp, e0, e1, rules.strip_fill, bm_all + (WIDE ? 0 : wv) * STRIP_BM_WORDS);
        const unsigned int strip_tiles = (unsigned int)tiles;
        bool either = false;
        // A strip of two panels stays a strip where its tiles are well filled.
        if (rules.panel_min) {
            int list[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int s0 = __builtin_amdgcn_readlane(lane_rp, 8 * h), l0 = __builtin_amdgcn_readlane(len, 8 * h);
                const bool alike = (__ballot(len == l0) >> (8 * h) & 0xFFull) == 0xFFull;
                const bool panel = (WIDE || !(tiles && h && !items[0])) && strip * 16 + 8 * h + 8 <= M && l0 >= rules.panel_min && alike;
                if (WIDE) {
                    if (panel && !same_lists(col, s0, l0, wv, WAVES) && lane == 0) atomicOr(&flags[2 + h], 1);
                    items[h] = panel;
                } else {
                    items[h] = panel && same_lists(col, s0, l0);
                }
                list[h] = l0;
            }
            if (WIDE) {
                __syncthreads();
                items[0] = items[0] && !flags[2];
                items[1] = items[1] && !flags[3];
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) items[h] = items[h] ? (list[h] + rules.pseg - 1) / rules.pseg : 0;
            // (or of one, where the matrix ends after 8 rows)
            either = tiles && items[0] && (items[1] || strip * 16 + 8 == M);
            if (either) {
                const bool panels = (int64_t)e1 - e0 < (int64_t)rules.panels_below * tiles;
                if (speaks) {
                    spread_add(pc, K_EITHER_TILES, (unsigned long long)tiles);
                    spread_add(pc, panels ? K_NNZ_EITHER_PANELS : K_NNZ_EITHER_STRIP, (unsigned long long)(e1 - e0));
                }
                if (panels) tiles = 0;
                else items[0] = items[1] = 0;
            } else if (tiles) items[0] = items[1] = 0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (!items[h]) continue;
                if (lane >> 3 == h) owned = 2;
                if (speaks) {
                    spread_add(pc, K_PANELS, 1ull);
                    spread_add(pc, K_NNZ_PANELS, (unsigned long long)list[h] * 8ull);
                }
            }
        }
        if (tiles) owned = 1;
        int lo = 0, span = 0, allowed = 0;
        if (rules.union_fill) {
            // the strip must be free as a whole, and even its longest row alone must not need
            // more tiles than the threshold allows
            const int64_t entries = (int64_t)e1 - (int64_t)e0;
            const int longest = __builtin_amdgcn_readfirstlane(max16(len));
            if (!tiles && !items[0] && !items[1] && entries >= (int64_t)rules.union_fill * ((longest + 15) / 16) && entries >= rules.union_fill) {
                strip_bounds<0>(col, lane_rp, e0, &lo, &span, &allowed);
                if (span > UNION_BM_WORDS * 32) span = 0;
            }
        }
        if (strip < n_strips && speaks) {
            if (rules.strip_fill && rules.panel_min) out.either[strip] = either ? strip_tiles : 0u;
            if (rules.strip_fill) {
                out.strip_ntiles[strip] = (unsigned int)tiles;
                if (tiles) {
                    spread_add(pc, K_TILES, (unsigned long long)tiles);
                    spread_add(pc, K_NNZ_TILES, (unsigned long long)(e1 - e0));
                }
            }
            if (rules.panel_min) {
                if (2 * strip < M / 8) out.panel_counts[2 * strip] = (unsigned int)items[0];
                if (2 * strip + 1 < M / 8) out.panel_counts[2 * strip + 1] = (unsigned int)items[1];
            }
        }
        if (!WIDE || wv == 0) {
            const int at = WIDE ? 0 : wv;
            if (lane < 17) rp_of[at][lane] = lane_rp;
            if (lane < 16) own_of[at][lane] = owned;
            if (lane == 0) { lo_of[at] = lo; span_of[at] = span > 0 ? span : 0; allowed_of[at] = allowed; }
        }
        __syncthreads();
        if (rules.union_fill) {
            for (int w = 0; w < STRIPS; ++w) {
                const int u_span = span_of[w];
                int u_tiles = 0;
                const int u0 = rp_of[w][0], u1 = rp_of[w][16];
                if (u_span > 0) {                                         // workgroup-uniform
                    const int words = (u_span + 31) >> 5;
                    for (int k = tid; k < words; k += WAVE * WAVES) bm_all[k] = 0u;
                    if (tid == 0) { found = 0; descents_found = 0; }
                    __syncthreads();
                    // as many entries each
                    const int64_t n = (int64_t)u1 - u0;
                    const int a = u0 + (int)(n * wv / WAVES), b = u0 + (int)(n * (wv + 1) / WAVES);
                    if (b > a) {
                        int64_t descents = 0;
                        (void)strip_scan<2>(col, a, b, INT64_MAX, lo_of[w], u_span, bm_all, &descents);
                        const int over = a > u0 && col[a] <= col[a - 1] ? 1 : 0;   // (the scan does not see the entry before its first)
                        if (lane == 0) atomicAdd(&descents_found, (int)descents + over);
                    }
                    __syncthreads();
                    int t = 0;
                    for (int k = tid; k < words; k += WAVE * WAVES) t += __builtin_popcount(bm_all[k]);
                    t = wave_sum_i32(t);
                    if (lane == 0 && t) atomicAdd(&found, t);
                    __syncthreads();
                    u_tiles = (found + 15) / 16;
                    if (descents_found != allowed_of[w] || u_tiles == 0 || n < (int64_t)rules.union_fill * u_tiles) u_tiles = 0;
                    if (u_tiles && tid < 16) own_of[w][tid] = 4;
                    if (u_tiles && tid == 0) {
                        spread_add(pc, K_UTILES, (unsigned long long)u_tiles);
                        spread_add(pc, K_NNZ_UTILES, (unsigned long long)n);
                    }
                    __syncthreads();                                      // (the next strip's bitmap; own_of)
                }
                if (tid == 0 && first + w < n_strips) out.ustrip_ntiles[first + w] = (unsigned int)u_tiles;
            }
        }
        if (wv == 0) {
            // one row per lane
            const int64_t row = first * 16 + lane;
            const bool mine = row < M && lane < 16 * STRIPS;
            const int at = WIDE ? 0 : lane >> 4, s = rp_of[at][lane & 15], n = rp_of[at][(lane & 15) + 1] - s;
            const int who = own_of[at][lane & 15];
            if (mine) out.owner[row] = (unsigned char)who;
            const unsigned int l = mine && who == 0 ? (unsigned int)n : 0u;
            if (rules.cand_min) {
                bool cand = l >= (unsigned int)rules.cand_min;
                int at0 = 0;
                if (cand) {
                    at0 = col[s];
                    const int64_t width = (int64_t)col[s + n - 1] - at0 + 1;
                    cand = width > 0 && (int64_t)n * 4 >= width;
                }
                const unsigned long long m = __ballot(cand);
                if (m) {                                                  // one append per wave
                    unsigned long long base = 0;
                    if (lane == 0) base = atomicAdd(&pc->n_candidates, (unsigned long long)__popcll(m));
                    base = ((unsigned long long)(unsigned int)__builtin_amdgcn_readfirstlane((int)(base >> 32)) << 32) |
                           (unsigned int)__builtin_amdgcn_readfirstlane((int)base);
                    if (cand)
                        out.cand_keys[base + (unsigned long long)__popcll(m & ((1ull << lane) - 1ull))] =
                            ((unsigned long long)(unsigned int)at0 << 32) | (unsigned long long)(unsigned int)row;
                }
            }
            // (sums of entries stay below the number of entries, which is an int)
            const unsigned int cnt = row_item_count(l, rules.ts, rules.seg);
            const int kind = cnt == 0 ? 0 : cnt == 1 ? 1 : 2;
            const int n_items = wave_sum_i32((int)cnt);
            unsigned int part[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                rows_sum[k] += (unsigned int)__popcll(__ballot(l != 0 && kind == k));
                part[k] = (unsigned int)wave_sum_i32(kind == k ? (int)l : 0);
                entries_sum[k] += part[k];
            }
            const unsigned int n_long = (unsigned int)__popcll(__ballot(l != 0 && kind == 2));
            if (lane == 0) {
                const int64_t block = first * 16 / SCAN_TILE;
                if (n_items) atomicAdd(&out.items[block], (unsigned int)n_items);
                if (part[0]) atomicAdd(&out.short_entries[block], part[0]);
                if (n_long) atomicAdd(&out.long_rows[block], n_long);
            }
        }
        __syncthreads();                                                  // (the next group's bitmaps and rows)
    }
    if (tid == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            spread_add(pc, K_ROWS_SHORT + k, rows_sum[k]);
            spread_add(pc, K_NNZ_SHORT + k, entries_sum[k]);
        }
    }
}

// Strips of two panels that k_own_rows sent either way all go one way, a strip per thread.
static __global__ __launch_bounds__(256) void k_settle_owners(const int32_t *__restrict__ rowptr, int M, int64_t n_strips,
                                                              int to_panels, int pseg, OwnArrays out, DevCounters *pc) {
    const int64_t strip = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned int tiles = strip < n_strips ? out.either[strip] : 0u;
    const bool moves = tiles != 0u && (out.strip_ntiles[strip] != 0u) == (to_panels != 0);
    int entries = 0;
    int panels = 0;
    if (moves) {                                               // (two panels, or one at the end of the matrix)
        out.strip_ntiles[strip] = to_panels ? 0u : tiles;
        for (; panels < 2 && strip * 16 + 8 * panels + 8 <= M; ++panels) {
            const int n = rowptr[strip * 16 + 8 * panels + 8] - rowptr[strip * 16 + 8 * panels];
            entries += n;
            out.panel_counts[2 * strip + panels] = to_panels ? (unsigned int)((n / 8 + pseg - 1) / pseg) : 0u;
            for (int r = 0; r < 8; ++r) out.owner[strip * 16 + 8 * panels + r] = to_panels ? 2 : 1;
        }
    }
    if (!__ballot(moves)) return;
    const unsigned long long all = (unsigned long long)wave_sum_i32(panels);
    const unsigned long long t = (unsigned long long)wave_sum_i32(moves ? (int)tiles : 0), n = (unsigned long long)wave_sum_i32(entries);
    if (lane_id() == 0) {                                      // (the sums wrap around: the slots add up to the difference)
        spread_add(pc, K_TILES, to_panels ? 0ull - t : t);
        spread_add(pc, K_NNZ_TILES, to_panels ? 0ull - n : n);
        spread_add(pc, K_PANELS, to_panels ? all : 0ull - all);
        spread_add(pc, K_NNZ_PANELS, to_panels ? n : 0ull - n);
    }
}

// The candidate keys in increasing order when there are at most RANK_SORT_MAX of them: every
// workgroup holds all keys in LDS and finds the ranks of 8 of them, 32 threads per key (keys are
// distinct, one per row, so the ranks are a permutation).  One short launch instead of the
// passes of a radix sort over 64-bit keys.
#ifndef SDDMM_RANK_SORT_SPLIT
#define SDDMM_RANK_SORT_SPLIT 32
#endif
constexpr int RANK_SORT_MAX = 8192, RANK_SORT_BLOCK = 256, RANK_SORT_SPLIT = SDDMM_RANK_SORT_SPLIT;
static __global__ __launch_bounds__(RANK_SORT_BLOCK) void k_rank_sort(const unsigned long long *__restrict__ in,
                                                               unsigned long long *__restrict__ out, int n) {
    __shared__ unsigned long long v[RANK_SORT_MAX];
    for (int i = (int)threadIdx.x; i < n; i += RANK_SORT_BLOCK) v[i] = in[i];
    __syncthreads();
    const int idx = (int)blockIdx.x * (RANK_SORT_BLOCK / RANK_SORT_SPLIT) + (int)(threadIdx.x / RANK_SORT_SPLIT);
    const int part = (int)(threadIdx.x % RANK_SORT_SPLIT);
    const unsigned long long mine = v[idx < n ? idx : n - 1];
    int below = 0;
#pragma unroll 8
    for (int i = part; i < n; i += RANK_SORT_SPLIT) below += v[i] < mine ? 1 : 0;
#pragma unroll
    for (int o = 1; o < RANK_SORT_SPLIT; o <<= 1) below += __shfl_xor(below, o, WAVE);
    if (part == 0 && idx < n) out[below] = mine;
}

// Gathered strips come in PAIRS: 32 consecutive candidates of the sorted order, the first 16
// as strip 2p, the rest as strip 2p+1, with ONE list of tile columns -- every tile column that
// any of the 32 rows touches -- so that the two strips have the same descriptors in the same
// order and a wavefront can use every B tile it loads for both (tile_window_pair_wave).  The
// list is padded with absent tile columns to a multiple of TILE_WINDOW, so that no window of
// four descriptors holds two strips, and stored window by window, the four descriptors of
// strip 2p followed by the four of strip 2p+1.
//
// Rows, extent and column span of pair vp; lanes 0..31 keep one row each.
struct GatheredHead {
    int row, s, e;        // per lane (row -1: none)
    int lo, span;         // wave-uniform, in tile columns
    int halves;           // wave-uniform: 2 when the second strip has rows, else 1
    int64_t entries;      // wave-uniform
};
__device__ __forceinline__ GatheredHead gathered_head(const int32_t *__restrict__ rowptr,
                                                      const int32_t *__restrict__ col,
                                                      const unsigned long long *__restrict__ sorted_keys,
                                                      int64_t n_cand, int64_t vp) {
    GatheredHead h;
    const int lane = lane_id();
    const int64_t idx = vp * 32 + lane;
    h.row = lane < 32 && idx < n_cand ? (int)(unsigned int)sorted_keys[idx] : -1;   // low half of the key
    h.s = h.row >= 0 ? rowptr[h.row] : 0;
    h.e = h.row >= 0 ? rowptr[h.row + 1] : 0;
    const bool has = h.e > h.s;
    const int first = has ? (col[h.s] >> 4) : INT32_MAX;
    const int last = has ? (col[h.e - 1] >> 4) : -1;
    // lanes 32..63 hold the neutral values; the 16-lane reductions of rows 0 and 1 of the wave make the pair's
    const int l16 = min16(first), h16 = min16(-last), n16 = sum16(h.e - h.s);
    const int l0 = __builtin_amdgcn_readlane(l16, 0), l1 = __builtin_amdgcn_readlane(l16, 16);
    const int g0 = __builtin_amdgcn_readlane(h16, 0), g1 = __builtin_amdgcn_readlane(h16, 16);
    const int l = l0 < l1 ? l0 : l1, hneg = g0 < g1 ? g0 : g1;
    h.lo = l;
    h.span = l == INT32_MAX ? 0 : -hneg - l + 1;
    h.entries = (int64_t)__builtin_amdgcn_readlane(n16, 0) + (int64_t)__builtin_amdgcn_readlane(n16, 16);
    h.halves = vp * 32 + 16 < n_cand ? 2 : 1;
    return h;
}

// One workgroup of 16 wavefronts per pair: wave i streams rows i and 16+i of the pair into the
// pair's tile-column bitmap in LDS (the rows are not neighbours in the CSR arrays, so they are
// independent streams).  Returns false when a row is not sorted.  Every wave of the workgroup
// must call it.
constexpr int GATHERED_BLOCK = 16 * WAVE;

__device__ __forceinline__ bool gathered_mark(const int32_t *__restrict__ col, const GatheredHead &h, unsigned int *bm,
                                              int *unsorted_flag) {
    const int words = (h.span + 31) >> 5;
    for (int w = (int)threadIdx.x; w < words; w += GATHERED_BLOCK) bm[w] = 0u;
    if (threadIdx.x == 0) *unsorted_flag = 0;
    __syncthreads();
    const int wi = wave_in_block();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int si = half ? __builtin_amdgcn_readlane(h.s, (wi & 15) + 16) : __builtin_amdgcn_readlane(h.s, wi & 15);
        const int ei = half ? __builtin_amdgcn_readlane(h.e, (wi & 15) + 16) : __builtin_amdgcn_readlane(h.e, wi & 15);
        if (ei > si) {                               // wave-uniform
            int64_t descents = 0;
            (void)strip_scan<1>(col, si, ei, INT64_MAX, h.lo, h.span, bm, &descents);
            if (descents != 0 && lane_id() == 0) atomicOr(unsorted_flag, 1);
        }
    }
    __syncthreads();
    return *unsorted_flag == 0;
}

// The row classes as k_classify_count left them.
struct RowClasses {
    unsigned int *items, *short_entries, *long_rows;           // per block of the row scan
    int ts, seg;
};
// The 64 lanes' rows (len 0: none) leave the classes, for they have found an owner.
__device__ __forceinline__ void leave_classes(const RowClasses &c, DevCounters *pc, int row, unsigned int len) {
    const unsigned int cnt = row_item_count(len, c.ts, c.seg);
    const int64_t block = row / SCAN_TILE;
    if (cnt) atomicSub(&c.items[block], cnt);
    else if (len) atomicSub(&c.short_entries[block], len);
    if (cnt > 1) atomicSub(&c.long_rows[block], 1u);
    const int kind = cnt == 0 ? 0 : cnt == 1 ? 1 : 2;
#pragma unroll
    for (int k = 0; k < 3; ++k) {                              // (sums of entries stay below the number of entries, an int)
        const unsigned long long m = __ballot(len != 0 && kind == k);
        if (m == 0ull) continue;
        const int entries = wave_sum_i32(kind == k ? (int)len : 0);
        if (lane_id() == 0) {                                  // (the sums wrap around: the slots add up to the difference)
            spread_add(pc, K_ROWS_SHORT + k, 0ull - (unsigned long long)__popcll(m));
            spread_add(pc, K_NNZ_SHORT + k, 0ull - (unsigned long long)entries);
        }
    }
}

// pass 1 of the gathered strips: descriptors per strip of the pair (0: not taken; the same for
// both strips), the strips' row table, ownership of the rows of a taken pair, which leave the row classes (counting
// all rows again was a launch of 6 us and one that cleared the counters).  The bitmap of a taken pair is kept for pass 2
// where there is room (stride words per pair: first tile column, span, bitmap; 0: no room).
static __global__ __launch_bounds__(GATHERED_BLOCK) void k_gathered_count(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
    const unsigned long long *__restrict__ sorted_keys,
    int64_t n_cand, int64_t n_vpairs, int min_fill, unsigned int *__restrict__ vstrip_ntiles,
    int32_t *__restrict__ vrows, unsigned char *__restrict__ owner, DevCounters *pc, RowClasses classes,
    unsigned int *__restrict__ kept, int stride) {
    __shared__ unsigned int bm[STRIP_BM_WORDS];
    __shared__ int unsorted_flag, tile_total;
    const int64_t vp = blockIdx.x;
    const int lane = lane_id();
    const bool first = wave_in_block() == 0;
    const GatheredHead h = gathered_head(rowptr, col, sorted_keys, n_cand, vp);   // the same in every wave
    if (first && lane < 32) vrows[vp * 32 + lane] = h.row;
    int tiles = 0;
    bool take = false;
    if (h.span > 0 && h.span <= STRIP_BM_WORDS * 32 && h.entries >= min_fill) {   // workgroup-uniform
        const bool sorted = gathered_mark(col, h, bm, &unsorted_flag);
        if (threadIdx.x == 0) tile_total = 0;
        __syncthreads();
        const int words = (h.span + 31) >> 5;
        int t = 0;
        for (int w = (int)threadIdx.x; w < words; w += GATHERED_BLOCK) t += __builtin_popcount(bm[w]);
        t = wave_sum_i32(t);
        if (lane == 0 && t) atomicAdd(&tile_total, t);
        __syncthreads();
        tiles = tile_total;
        // the threshold is per 16x16 tile: each tile column of the pair is one tile per strip that has rows
        take = sorted && tiles > 0 && h.entries >= (int64_t)min_fill * tiles * h.halves;
    }
    const int padded = (tiles + TILE_WINDOW - 1) / TILE_WINDOW * TILE_WINDOW;
    if (take && stride) {                                      // (the span of a taken pair fits the bitmap and stays below N)
        unsigned int *to = kept + vp * stride;
        for (int w = (int)threadIdx.x; w < (h.span + 31) >> 5; w += GATHERED_BLOCK) to[2 + w] = bm[w];
        if (threadIdx.x == 0) { to[0] = (unsigned int)h.lo; to[1] = (unsigned int)h.span; }
    }
    if (take && wave_in_block() == 1) leave_classes(classes, pc, h.row, h.row >= 0 ? (unsigned int)(h.e - h.s) : 0u);
    if (first) {
        if (take && h.row >= 0) owner[h.row] = 3;
        if (lane == 0) {
            vstrip_ntiles[2 * vp] = take ? (unsigned int)padded : 0u;
            vstrip_ntiles[2 * vp + 1] = take ? (unsigned int)padded : 0u;
            if (take) {
                spread_add(pc, K_TILES, 2ull * (unsigned long long)padded);
                spread_add(pc, K_NNZ_TILES, (unsigned long long)h.entries);
            }
        }
    }
}

// A descriptor that stands for nothing (no row has an entry in it): complete, k_tile_rows skips it.
__device__ __forceinline__ void write_empty_desc(TileDesc *__restrict__ tiles, int32_t *__restrict__ tile_cols,
                                                 int64_t at, int strip, int tj) {
    int4 *d = reinterpret_cast<int4 *>(tiles + at);
    d[0] = make_int4(strip, tj, 1, 0);
#pragma unroll
    for (int k = 1; k < (int)(sizeof(TileDesc) / 16); ++k) d[k] = make_int4(0, 0, 0, 0);
    write_aligned_cols(tile_cols, at, tj);
}

// The descriptors of a strip, or of a pair of gathered strips window by window (descriptor 8k + 4h + j of the pair: strip h,
// the (4k+j)-th tile column), from base on, by a workgroup of 16 wavefronts; lds.bm holds the tile columns from lo on.
// Wave i writes what the descriptors say of rows i and 16+i: it walks the row, marks every entry in the mask of its tile
// (LDS), and the entries in the masks before a tile tell where the row enters it.  (As a binary search per tile and row
// afterwards, k_tile_rows: 13.8 us for 20 000 tiles.)
constexpr int GATHERED_MASKS = 384;                            // tile columns whose masks fit the LDS
struct DescriptorLds {
    unsigned int bm[STRIP_BM_WORDS];
    int before[STRIP_BM_WORDS];                                // tile columns in the words before
    int totals[16], highest, unsorted;
    unsigned int masks[16][GATHERED_MASKS];
};
template <bool PAIR>
__device__ __forceinline__ void write_descriptors(const int32_t *__restrict__ col, int row_s, int row_e, int lo, int words, int per_strip,
                                                  int strip0, int64_t base, TileDesc *__restrict__ tiles,
                                                  int32_t *__restrict__ tile_cols, DescriptorLds &lds) {
    __syncthreads();
    // one thread per word: tile columns in the words before it
    static_assert(STRIP_BM_WORDS <= GATHERED_BLOCK, "one word per thread");
    const int t = (int)threadIdx.x, lane = lane_id(), wv = wave_in_block();
    const unsigned int mine = t < words ? lds.bm[t] : 0u;
    const int n = __builtin_popcount(mine);
    const int incl = wave_inclusive_sum(n);
    if (lane == WAVE - 1) lds.totals[wv] = incl;
    if (t == 0) lds.highest = -1;
    __syncthreads();
    int run = incl - n, all = 0;
    for (int w = 0; w < GATHERED_BLOCK / WAVE; ++w) {
        run += w < wv ? lds.totals[w] : 0;
        all += lds.totals[w];
    }
    if (t < words) lds.before[t] = run;
    if (mine) atomicMax(&lds.highest, t * 32 + 31 - __builtin_clz(mine));
    __syncthreads();
    auto place = [&](int rank) { return PAIR ? base + 2 * TILE_WINDOW * (rank / TILE_WINDOW) + (rank % TILE_WINDOW) : base + rank; };
    auto put = [&](int rank, int tj) {
        const int64_t at = place(rank);
        *reinterpret_cast<int4 *>(tiles + at) = make_int4(strip0, tj, 1, 0);
        write_aligned_cols(tile_cols, at, tj);
        if (PAIR) {
            *reinterpret_cast<int4 *>(tiles + at + TILE_WINDOW) = make_int4(strip0 + 1, tj, 1, 0);
            write_aligned_cols(tile_cols, at + TILE_WINDOW, tj);
        }
    };
    // one thread per tile column of the span
    for (int b = t; b < words * 32; b += GATHERED_BLOCK) {
        const unsigned int x = lds.bm[b >> 5], bit = 1u << (b & 31);
        if (x & bit) put(lds.before[b >> 5] + __builtin_popcount(x & (bit - 1u)), lo + b);
    }
    // the padding: tile columns beyond the pair's last one, which no row of the pair has (the masks come out empty, the
    // positions say where the row ends)
    if (all + t < per_strip) put(all + t, lo + lds.highest + 1 + t);
    // the rows' part of the descriptors
    auto rank_of = [&](int c) {
        const int b = (c >> 4) - lo;
        return lds.before[b >> 5] + __builtin_popcount(lds.bm[b >> 5] & ((1u << (b & 31)) - 1u));
    };
    unsigned int *mk = lds.masks[wv];
    for (int half = 0; half < (PAIR ? 2 : 1); ++half) {
        const int s = __builtin_amdgcn_readlane(row_s, (wv & 15) + 16 * half), e = __builtin_amdgcn_readlane(row_e, (wv & 15) + 16 * half);
        int at = s;                                            // where the row enters the next tile
        // (a pair of more tile columns than there is room for: some of them at a time)
        for (int r0 = 0; r0 < per_strip; r0 += GATHERED_MASKS) {
            const int n_here = per_strip - r0 < GATHERED_MASKS ? per_strip - r0 : GATHERED_MASKS;
            for (int k = lane; k < n_here; k += WAVE) mk[k] = 0u;
            wave_lds_order();
            // (the entries of a tile that one lane holds as one: neighbours in one word of LDS wait for each other)
            constexpr int AHEAD = 4;
            for (int p = s; p < e; p += AHEAD * PER_LOAD) {
                I4u c[AHEAD];
                load_entries(col, p, e, c);
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    const int i0 = p + u * PER_LOAD + 4 * lane;
                    const int q[4] = {c[u].x, c[u].y, c[u].z, c[u].w};
                    unsigned int m = 0;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        m |= 1u << (q[j] & 15);
                        if (i0 + j < e && (j == 3 || i0 + j + 1 >= e || (q[j < 3 ? j + 1 : 3] >> 4) != (q[j] >> 4))) {
                            const int k = rank_of(q[j]) - r0;
                            if ((unsigned int)k < (unsigned int)n_here) atomicOr(&mk[k], m);
                            m = 0;
                        }
                    }
                }
            }
            wave_lds_order();
            for (int k0 = 0; k0 < n_here; k0 += WAVE) {
                const int k = k0 + lane;
                const unsigned int m = k < n_here ? mk[k] : 0u;
                const int n_in = __builtin_popcount(m);
                const int upto = wave_inclusive_sum(n_in);
                if (k < n_here) {
                    TileDesc *d = tiles + place(r0 + k) + half * TILE_WINDOW;
                    d->off[wv & 15] = at + upto - n_in;
                    d->mask[wv & 15] = (uint16_t)m;
                }
                at += __builtin_amdgcn_readlane(upto, WAVE - 1);
            }
            wave_lds_order();                                  // (the masks of the next columns or row)
        }
    }
}

// pass 2 of the strips where there are few of them: a workgroup per strip, complete descriptors.
static __global__ __launch_bounds__(WIDE_BLOCK) void k_strip_tiles_wide(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col, int M,
    const unsigned int *__restrict__ strip_ntiles, const unsigned int *__restrict__ strip_off,
    TileDesc *__restrict__ tiles, int32_t *__restrict__ tile_cols) {
    __shared__ DescriptorLds lds;
    const int64_t strip = blockIdx.x;
    const int per_strip = (int)strip_ntiles[strip];
    if (per_strip == 0) return;                                // workgroup-uniform
    const int lane = lane_id(), wv = wave_in_block();
    const int64_t r = strip * 16 + lane;
    const int row_s = rowptr[r < M ? r : M], row_e = __shfl_down(row_s, 1, WAVE);
    int lo, span, allowed;
    strip_bounds(col, row_s, __builtin_amdgcn_readlane(row_s, 0), &lo, &span, &allowed);
    if (span > STRIP_BM_WORDS * 32) {
        if (wv == 0) walk_descriptors(rowptr, col, M, strip, strip_off[strip], tiles, tile_cols);
        return;
    }
    const int words = (span + 31) >> 5;
    for (int w = (int)threadIdx.x; w < words; w += WIDE_BLOCK) lds.bm[w] = 0u;
    __syncthreads();
    const int s = __builtin_amdgcn_readlane(row_s, wv), e = __builtin_amdgcn_readlane(row_e, wv);
    int64_t descents;
    if (e > s) (void)strip_scan<1>(col, s, e, INT64_MAX, lo, span, lds.bm, &descents);
    write_descriptors<false>(col, row_s, row_e, lo, words, per_strip, (int)strip, strip_off[strip], tiles, tile_cols, lds);
}

// pass 2 of the gathered strips.  `tiles` / `tile_cols`
// point at the first gathered descriptor; the `lead` descriptors before it (fewer than
// TILE_WINDOW) fill the last window of the strips that precede the gathered ones.
static __global__ __launch_bounds__(GATHERED_BLOCK) void k_gathered_tiles(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
    const unsigned long long *__restrict__ sorted_keys,
    int64_t n_cand, int64_t n_vpairs, const unsigned int *__restrict__ vstrip_ntiles,
    const unsigned int *__restrict__ vstrip_off, TileDesc *__restrict__ tiles, int32_t *__restrict__ tile_cols,
    int lead, const unsigned int *__restrict__ kept, int stride) {
    __shared__ DescriptorLds lds;
    const int64_t vp = blockIdx.x;
    // (strip -1 is nobody's: the window that holds them is walked tile by tile, and they write nothing)
    if (vp == 0 && (int)threadIdx.x < lead) write_empty_desc(tiles, tile_cols, -(int64_t)lead + threadIdx.x, -1, 0);
    const unsigned int per_strip = vstrip_ntiles[2 * vp];
    if (per_strip == 0) return;                      // workgroup-uniform
    const int lane = lane_id();
    int lo, words, row_s, row_e;                               // lanes 0..31: a row of the pair each
    if (stride) {
        const unsigned int *from = kept + vp * stride;
        lo = (int)from[0];
        words = ((int)from[1] + 31) >> 5;
        const int64_t idx = vp * 32 + lane;
        const int row = lane < 32 && idx < n_cand ? (int)(unsigned int)sorted_keys[idx] : -1;
        for (int w = (int)threadIdx.x; w < words; w += GATHERED_BLOCK) lds.bm[w] = from[2 + w];
        row_s = row >= 0 ? rowptr[row] : 0;
        row_e = row >= 0 ? rowptr[row + 1] : 0;
    } else {
        const GatheredHead h = gathered_head(rowptr, col, sorted_keys, n_cand, vp);
        (void)gathered_mark(col, h, lds.bm, &lds.unsorted);
        lo = h.lo;
        words = (h.span + 31) >> 5;
        row_s = h.s;
        row_e = h.e;
    }
    write_descriptors<true>(col, row_s, row_e, lo, words, (int)per_strip, GATHERED_BASE + (int)(2 * vp), vstrip_off[2 * vp], tiles, tile_cols, lds);
}

// pass 3 (strips and union strips): one thread per (descriptor, row): CSR position of the row's first entry
// at or after the tile's first column, and the mask of the tile's columns present.
// Bit n of the mask stands for the n-th of the tile's 16 columns; a row's entries
// inside a tile are consecutive in CSR, in the order of the tile's columns.
static __global__ __launch_bounds__(256) void k_tile_rows(const int32_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ col, int M,
                                                   const int32_t *__restrict__ tile_cols,
                                                   TileDesc *__restrict__ tiles, int64_t n_tiles, int64_t nnz) {
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t t = slot >> 4;
    const int sub = (int)(slot & 15);
    if (t >= n_tiles) return;
    TileDesc *d = tiles + t;
    const int4 head = *reinterpret_cast<const int4 *>(d);     // strip, tj, pad[0], pad[1]
    if (head.z != 0) return;                                   // written by the merging walk
    const int64_t row = (int64_t)head.x * 16 + sub;
    int p = 0, end = 0;
    if (row < M) { p = rowptr[row]; end = rowptr[row + 1]; }
    int tc[16];
    {
        const int4 *src = reinterpret_cast<const int4 *>(tile_cols + t * 16);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int4 v = src[k];
            tc[4 * k] = v.x; tc[4 * k + 1] = v.y; tc[4 * k + 2] = v.z; tc[4 * k + 3] = v.w;
        }
    }
    int top = tc[0];                                           // last real column of the tile
#pragma unroll
    for (int k = 1; k < 16; ++k) top = tc[k] != INT32_MAX ? tc[k] : top;
    const int target = tc[0];
    int a = p, b = end;
    while (a < b) {
        const int mid = a + ((b - a) >> 1);
        if (col[mid] < target) a = mid + 1; else b = mid;
    }
    unsigned int mask = 0;
    if (a < end) {
        const int last = end - 1;
        int cs[16];
        if (a + 16 <= nnz) {
            // sixteen entries in four loads (as sixteen loads: 16.0 us for 20 000 tiles, four: 9.5; a load whose 64 lanes
            // touch as many lines takes the address unit 64 cycles whatever its width)
#pragma unroll
            for (int j = 0; j < 16; j += 4) {
                const I4u v = *reinterpret_cast<const I4u *>(col + a + j);
                cs[j] = v.x; cs[j + 1] = v.y; cs[j + 2] = v.z; cs[j + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) cs[j] = col[a + j < last ? a + j : last];
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if (a + j <= last && cs[j] <= top) {
                int n = 0;                                     // number of tile columns below this one
#pragma unroll
                for (int k = 0; k < 16; ++k) n += tc[k] < cs[j] ? 1 : 0;
                mask |= 1u << n;
            }
        }
    }
    d->off[sub] = a;
    d->mask[sub] = (uint16_t)mask;
}

// generic exclusive scan of n unsigned ints: block sums, then apply
static __global__ __launch_bounds__(SCAN_BLOCK) void k_scan_sums(const unsigned int *__restrict__ in, int64_t n,
                                                          unsigned int *__restrict__ block_sums) {
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    unsigned int mine = 0;
    for (int q = 0; q < SCAN_ITEMS; ++q) mine += base + q < n ? in[base + q] : 0u;
    unsigned int total;
    (void)block_exclusive_scan(mine, &total);
    if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}
static __global__ __launch_bounds__(SCAN_BLOCK) void k_scan_apply(const unsigned int *__restrict__ in, int64_t n,
                                                           const unsigned int *__restrict__ block_offsets,
                                                           unsigned int *__restrict__ out) {
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    unsigned int v[SCAN_ITEMS], mine = 0;
    for (int q = 0; q < SCAN_ITEMS; ++q) { v[q] = base + q < n ? in[base + q] : 0u; mine += v[q]; }
    unsigned int total;
    unsigned int at = block_offsets[blockIdx.x] + block_exclusive_scan(mine, &total);
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        if (base + q < n) out[base + q] = at;
        at += v[q];
    }
}

// ---- the MFMA kernel ------------------------------------------------------------
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

// ---- rows as the tile and panel kernels read them ---------------------------------------
// Step s of these kernels takes the units (16 bytes) 4s .. 4s+3 of a row.  WholeRows: rows of STEPS * 64 bytes.
// RaggedRows: rows of any other length up to that (more than ragged_whole_steps).  A unit past the end
// of the row is the last one loaded again, and is zeroed (trim) once it has arrived, in both operands: what a product
// adds there is 0 * 0 whatever the rows hold.  fp32 rows of no whole number of units are read as the gather kernels
// read them (UnitF32x4u).
constexpr int ragged_whole_steps(int steps) {
    return steps <= 1 ? 0 : steps == 2 ? 1 : steps == 4 ? 2 : steps == 6 ? 4 : steps == 8 ? 6 : steps == 12 ? 8 : 12;
}

template <int STEPS>
struct WholeRows {
    static constexpr bool RAGGED = false;
    using Row = const uint4 *;
    explicit __device__ __forceinline__ WholeRows(int) {}
    __device__ __forceinline__ Row row(const void *base, int64_t r) const { return (const uint4 *)base + r * (STEPS * 4); }
    __device__ __forceinline__ const uint4 &unit(const void *, Row row, int u, int) const { return row[u]; }
    __device__ __forceinline__ uint4 trim(const uint4 &v, int, int) const { return v; }
    __device__ __forceinline__ int last_unit() const { return STEPS * 4 - 1; }
};

template <class U_, int STEPS>
struct RaggedRows {
    using U = U_;
    static constexpr bool RAGGED = true;
    static constexpr int WHOLE_STEPS = ragged_whole_steps(STEPS);
    using Row = uint32_t;                                     // byte offset: operands below 4 GiB
    int len, last;                                            // length as U takes it, last unit
    __device__ __forceinline__ int last_unit() const { return last; }
    explicit __device__ __forceinline__ RaggedRows(int len_) : len(len_), last(U::units(len_) - 1) {}
    __device__ __forceinline__ Row row(const void *, int64_t r) const { return (uint32_t)r * U::row_bytes(len); }
    // unit u of a row; step: the step it belongs to as far as the compiler knows it (STEPS: any)
    __device__ __forceinline__ uint4 unit(const void *base, Row row, int u, int step) const {
        const uint32_t at = step < WHOLE_STEPS ? (uint32_t)u * 16u : U::unit_off(u < last ? u : last, len);
        return __builtin_bit_cast(uint4, load_unit<U, uint32_t>(base, row + at));
    }
    __device__ __forceinline__ uint4 trim(const uint4 &v, int u, int step) const {
        if (step < WHOLE_STEPS) return v;
        const uint4 t = __builtin_bit_cast(uint4, U::trim(__builtin_bit_cast(typename U::T, v), u, len));
        const bool in = u <= last;
        return make_uint4(in ? t.x : 0u, in ? t.y : 0u, in ? t.z : 0u, in ? t.w : 0u);
    }
};

// acc += the products of one unit of 16 rows with one of 16 columns.  Where CHAINS is 4 the four components of an fp32
// unit have an accumulator each.
template <int DT, int CHAINS>
__device__ __forceinline__ void mfma_unit(const uint4 &a, const uint4 &b, f32x4_t (&acc)[CHAINS]) {
    if constexpr (DT == DT_BF16) {
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                         acc[0], 0, 0, 0);
    } else if constexpr (DT == DT_F16) {
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b),
                                                        acc[0], 0, 0, 0);
    } else {
        auto part = [&](uint32_t x, uint32_t y, f32x4_t &c) {
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y), c, 0, 0, 0);
        };
        part(a.x, b.x, acc[0]);
        part(a.y, b.y, acc[1 % CHAINS]);
        part(a.z, b.z, acc[2 % CHAINS]);
        part(a.w, b.w, acc[3 % CHAINS]);
    }
}

// f(S0) + ... + f(S0 + N - 1), added in pairs
template <int S0, int N, class F>
__device__ __forceinline__ auto pairwise(F &&f) {
    if constexpr (N == 1) return f(std::integral_constant<int, S0>{});
    else return pairwise<S0, (N + 1) / 2>(f) + pairwise<S0 + (N + 1) / 2, N / 2>(f);
}

// The 16x16 products of N steps; b(s): the column operand of step s.  Whole rows: one accumulator.
// The gather kernels, which took ragged rows before, add up chains of an eighth of a row; one accumulator over all of it is
// further from the exact sum (fp32 K = 250 1.5e-7 of the result's norm against 1.2e-7, bf16 K = 456 1.0e-7 against 0.7e-7),
// so every step starts from zero and the steps are added in pairs (0.9e-7 and 0.7e-7).
template <int DT, class R, int N, class F>
__device__ __forceinline__ f32x4_t mfma_steps(const uint4 (&a)[N], F &&b) {
    if constexpr (R::RAGGED) {
        return pairwise<0, N>([&](auto s) {
            constexpr int CHAINS = DT == DT_F32 ? 4 : 1;
            f32x4_t acc[CHAINS] = {};
            mfma_unit<DT, CHAINS>(a[(int)s], b((int)s), acc);
            if constexpr (CHAINS == 4) {
                const f32x4_t sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
                // (steps that overlap take sixteen registers each: near-dense rows K = 33 23 -> 52 us without this, in spills)
                __builtin_amdgcn_sched_barrier(0);
                return sum;
            } else return acc[0];
        });
    } else {
        f32x4_t acc[1] = {};
#pragma unroll
        for (int s = 0; s < N; ++s) mfma_unit<DT, 1>(a[s], b(s), acc);
        return acc[0];
    }
}

// One wavefront computes `tiles_per_wave` consecutive tiles.  Operand layout of
// both MFMA shapes used: lane l supplies row (l & 15) of its operand and the k
// positions selected by (l >> 4); the result register i of lane l is row
// 4*(l >> 4) + i, column (l & 15).  In step s operand lane l holds the 16-byte unit
// 4*s + (l >> 4) of its row; which k positions end up in which MFMA does not matter
// as long as A and B agree.  STEPS = row bytes / 64.
// The units are READ in another layout -- four neighbouring lanes on the 64
// contiguous bytes of one row, 16 line segments per instruction instead of the 64 a
// load in operand layout touches -- and moved into the operand layout through the
// LDS crossbar (ds_bpermute): the vector memory pipeline pays per line segment that
// neighbouring lanes touch, not per byte.
//
// Software pipeline, three tiles deep, every load unconditional so that the wait
// counts stay exact (loads return in issue order):
//   iteration t issues   B rows + S values of tile t+1   (needs descriptor t+1)
//                        descriptor of tile t+2
//   and then computes    MFMAs of tile t, scale, scatter (operands landed during t-1)
// The A panel of the current strip stays in registers and is reloaded only when
// the strip changes (a wave-uniform branch placed before the iteration's loads).
// tiles [w*tiles_per_wave, (w+1)*tiles_per_wave) on the calling wavefront
template <int DT, int STEPS, class R>
__device__ __forceinline__ void tile_wave(const R &rows, const void *__restrict__ A, const void *__restrict__ B, int M, int N,
                                          const int32_t *__restrict__ vrows, const int32_t *__restrict__ tile_cols,
                                          const TileDesc *__restrict__ tiles, int64_t n_tiles, int tiles_per_wave,
                                          const float *__restrict__ sval, float *__restrict__ P, int64_t w) {
    int64_t t = w * tiles_per_wave;
    if (t >= n_tiles) return;
    int64_t t_end = t + tiles_per_wave;
    t_end = t_end < n_tiles ? t_end : n_tiles;
    const int64_t t_last = t_end - 1;
    const int lane = lane_id();
    const int r16 = lane & 15, q = lane >> 4;        // operand / result layout
    const int lrow = lane >> 2, lunit = lane & 3;    // memory layout: four neighbouring lanes on 64 bytes of a row
    const int to_operand_from = (4 * r16 + q) << 2;  // ds_bpermute address: operand lane (r16,q) <- memory lane 4*r16+q
    const unsigned int below = (1u << r16) - 1u;
    auto to_operand = [&](const uint4 &v, int s) {     // unit 4s + q of the lane's row
        uint4 r;
        r.x = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.x);
        r.y = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.y);
        r.z = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.z);
        r.w = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.w);
        return rows.trim(r, 4 * s + q, s);
    };

    struct Desc {
        int strip, bcol;    // bcol: the B row this lane loads (memory layout)
        int4 off;
        uint2 mask;
    };
    struct Oper {
        uint4 b[STEPS];
        float s[4];
        int pos[4];
        unsigned int act;   // bit i: result register i is a stored entry
    };
    auto load_desc = [&](int64_t ti) {
        ti = ti < t_last ? ti : t_last;
        const TileDesc *d = tiles + ti;
        Desc r;
        r.strip = d->strip;
        r.bcol = tile_cols[ti * 16 + lrow];
        r.off = *(const int4 *)&d->off[q * 4];
        r.mask = *(const uint2 *)&d->mask[q * 4];
        return r;
    };
    auto load_oper = [&](const Desc &d) {
        Oper o;
        int64_t brow = d.bcol;
        brow = brow < N ? brow : N - 1;   // columns past N (and the filler of a short union tile) are never in a mask
        const typename R::Row src = rows.row(B, brow);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) o.b[s] = rows.unit(B, src, 4 * s + lunit, s);
        const int offs[4] = {d.off.x, d.off.y, d.off.z, d.off.w};
        const unsigned int masks[4] = {d.mask.x & 0xFFFFu, d.mask.x >> 16, d.mask.y & 0xFFFFu, d.mask.y >> 16};
        o.act = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool on = (masks[i] >> r16) & 1u;
            o.act |= on ? (1u << i) : 0u;
            // position of (row 4q+i, column r16) in the CSR arrays; entry 0 when absent
            o.pos[i] = on ? offs[i] + __builtin_popcount(masks[i] & below) : 0;
            o.s[i] = sval[o.pos[i]];
        }
        return o;
    };

    Desc d_cur = load_desc(t);
    Oper o_cur = load_oper(d_cur);
    Desc d_nxt = load_desc(t + 1);
    int cur_strip = -1;
    uint4 a[STEPS];
    for (; t < t_end; ++t) {
        const int strip = __builtin_amdgcn_readfirstlane(d_cur.strip);
        if (strip != cur_strip) {
            cur_strip = strip;
            int64_t arow = strip >= GATHERED_BASE ? (int64_t)vrows[(int64_t)(strip - GATHERED_BASE) * 16 + lrow]
                                                  : (int64_t)strip * 16 + lrow;
            arow = arow < 0 ? 0 : (arow < M ? arow : M - 1);   // missing rows are never in a mask
            const typename R::Row src = rows.row(A, arow);
#pragma unroll
            for (int s = 0; s < STEPS; ++s) a[s] = to_operand(rows.unit(A, src, 4 * s + lunit, s), s);
        }
        const Oper o_nxt = load_oper(d_nxt);
        const Desc d_nn = load_desc(t + 2);
        const f32x4_t sum = mfma_steps<DT, R>(a, [&](int s) { return to_operand(o_cur.b[s], s); });
        // scale by S and scatter: result register i is row 4*q+i, column r16
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if ((o_cur.act >> i) & 1u) P[o_cur.pos[i]] = sum[i] * o_cur.s[i];
        o_cur = o_nxt;
        d_cur = d_nxt;
        d_nxt = d_nn;
    }
}

// ---- windows of four tiles ---------------------------------------------------------
// A wavefront that walks its tiles one after the other spends its life waiting: a launch
// of this path lasts a dozen microseconds, a dependent memory round trip about one, and
// the walk chains descriptor -> operands -> result for every tile.  So the unit of work is
// a WINDOW of TILE_WINDOW consecutive descriptors of one strip, handled as a batch with
// two round trips: (1) the window record, one dword per lane; (2) everything else at once
// -- the A panel, the B rows of all its tiles, and the S values and column indices.
//
// S and P are not accessed per (row, tile): the entries of row r inside the window's
// tiles are consecutive in the CSR arrays (the tiles are consecutive present tiles of the
// strip, so nothing of the row lies between them), cnt[r] entries from p0[r].  Four
// lanes per row read and write them 16 bytes at a time whatever the fill of the tiles
// (the last lane of a row moves its four entries back so that they end with the row's
// run: some entries are written twice with the same value, none is written in parts).
// The products come from the matrix cores in result layout, pass through LDS (written
// by columns of 16 rows, 16 bytes per lane) and are picked up per entry: its column says
// which tile and which column of the tile.  Per window of four tiles with 92 entries
// each: 20 memory instructions instead of 56.
//
// A window whose descriptors are not plain aligned tiles of one strip (a strip ends
// inside it, union tiles) is flagged by the plan and walked tile by tile (tile_wave).
constexpr int WIN_PITCH = 20;                 // floats per result column in LDS: 16 rows, padded, 16-byte aligned
constexpr int WIN_LDS_FLOATS = TILE_WINDOW * 16 * WIN_PITCH;

struct alignas(16) TileWindow {               // lane l < 48 loads dword l
    int32_t arow[16];    // row of A for strip row r (row 0 where the strip has no such row: then cnt is 0)
    int32_t p0[16];      // CSR position of row r's first entry inside the window
    uint16_t cnt[16];    // entries of row r inside the window (consecutive from p0)
    int32_t tj[TILE_WINDOW];   // tile columns, -1 where the window has fewer tiles
    int32_t flags;       // != 0: walk the window tile by tile
    int32_t maxcnt;      // largest cnt
    int32_t paired;      // != 0: a window of a pair of gathered strips (same tile columns as its neighbour)
    int32_t pad;
};
static_assert(sizeof(TileWindow) == 192, "TileWindow layout");

// plan: one thread per (window, strip row)
static __global__ __launch_bounds__(256) void k_tile_windows(const int32_t *__restrict__ vrows, int M, int64_t nnz,
                                                      const TileDesc *__restrict__ tiles, int64_t n_tiles,
                                                      int64_t union_lo, int64_t union_hi, int64_t gathered_lo,
                                                      TileWindow *__restrict__ win, int64_t n_win) {
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t w = slot >> 4;
    const int r = (int)(slot & 15);
    if (w >= n_win) return;                   // groups of 16 lanes leave together
    const int64_t t0 = w * TILE_WINDOW;
    const int n = (int)(n_tiles - t0 < TILE_WINDOW ? n_tiles - t0 : TILE_WINDOW);
    const int4 h0 = *reinterpret_cast<const int4 *>(tiles + t0);          // strip, tj, pad[0], pad[1]
    // the 16-byte accesses of the batch need four entries to exist
    bool mixed = (t0 < union_hi && t0 + n > union_lo) || nnz < 4;
    int tj[TILE_WINDOW];
#pragma unroll
    for (int k = 0; k < TILE_WINDOW; ++k) {
        tj[k] = -1;
        if (k < n) {
            const int4 h = *reinterpret_cast<const int4 *>(tiles + t0 + k);
            tj[k] = h.y;
            mixed |= h.x != h0.x;
        }
    }
    const int strip = h0.x;
    const int64_t row = strip >= GATHERED_BASE ? (int64_t)vrows[(int64_t)(strip - GATHERED_BASE) * 16 + r]
                                               : (int64_t)strip * 16 + r;
    const bool valid = row >= 0 && row < M;
    const TileDesc *last = tiles + t0 + n - 1;
    const int p0 = tiles[t0].off[r];
    int cnt = valid && !mixed ? last->off[r] + __builtin_popcount((unsigned int)last->mask[r]) - p0 : 0;
    cnt = cnt < 0 ? 0 : (cnt > 16 * TILE_WINDOW ? 16 * TILE_WINDOW : cnt);
    const int mx = max16(cnt);
    TileWindow *o = win + w;
    o->arow[r] = valid ? (int32_t)row : 0;
    o->p0[r] = p0;
    o->cnt[r] = (uint16_t)cnt;
    if (r == 0) {
#pragma unroll
        for (int k = 0; k < TILE_WINDOW; ++k) o->tj[k] = tj[k];
        o->flags = mixed ? 1 : 0;
        o->maxcnt = mx;
        o->paired = t0 >= gathered_lo ? 1 : 0;
        o->pad = 0;
    }
}

// window w on the calling wavefront; lds: WIN_LDS_FLOATS floats of its own
template <int DT, int STEPS, class R>
__device__ __forceinline__ void tile_window_wave(const R &rows, const void *__restrict__ A, const void *__restrict__ B, int M, int N,
                                                 const int32_t *__restrict__ vrows,
                                                 const int32_t *__restrict__ tile_cols,
                                                 const TileDesc *__restrict__ tiles, int64_t n_tiles,
                                                 const TileWindow *__restrict__ win, int64_t n_win,
                                                 const int32_t *__restrict__ col, const float *__restrict__ sval,
                                                 float *__restrict__ P, int64_t nnz, int64_t w, float *lds,
                                                 const int32_t *__restrict__ order = nullptr) {
    if (w >= n_win) return;
    if (order) w = order[w];                              // the plan's order of the windows (k_window_order)
    const int lane = lane_id();
    if (win == nullptr) {                                 // the plan chose the tile-by-tile walk for this matrix
        tile_wave<DT, STEPS>(rows, A, B, M, N, vrows, tile_cols, tiles, n_tiles, TILE_WINDOW, sval, P, w);
        return;
    }
    const int32_t *rec = reinterpret_cast<const int32_t *>(win + w);
    const int dw = rec[lane < 48 ? lane : 47];
    if (__builtin_amdgcn_readlane(dw, 44) != 0) {
        tile_wave<DT, STEPS>(rows, A, B, M, N, vrows, tile_cols, tiles, n_tiles, TILE_WINDOW, sval, P, w);
        return;
    }
    const int maxcnt = __builtin_amdgcn_readlane(dw, 45);
    if (maxcnt <= 0) return;
    const int r16 = lane & 15, q = lane >> 4;        // operand / result layout
    const int lrow = lane >> 2, lunit = lane & 3;    // memory layout: four neighbouring lanes on 64 bytes of a row
    const int to_operand_from = (4 * r16 + q) << 2;
    auto to_operand = [&](const uint4 &v, int s) {     // unit 4s + q of the lane's row
        uint4 r;
        r.x = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.x);
        r.y = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.y);
        r.z = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.z);
        r.w = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.w);
        return rows.trim(r, 4 * s + q, s);
    };
    int tj[TILE_WINDOW];
#pragma unroll
    for (int k = 0; k < TILE_WINDOW; ++k) tj[k] = __builtin_amdgcn_readlane(dw, 40 + k);
    // the row of the S/P accesses of this lane: strip row lane>>2, its entries 4(lane&3)+16m.. of the window
    const int p0 = __shfl(dw, 16 + lrow, WAVE);
    const int cw = __shfl(dw, 32 + (lrow >> 1), WAVE);
    const int cnt = (lrow & 1) ? (int)((unsigned int)cw >> 16) : (cw & 0xFFFF);
    const int64_t arow = __shfl(dw, lrow, WAVE);
    auto entry_pos = [&](int m) {
        int ws = 4 * lunit + 16 * m;
        ws = ws < cnt - 4 ? ws : cnt - 4;
        ws = ws < 0 ? 0 : ws;
        const int64_t pos = (int64_t)p0 + ws;
        return pos < nnz - 4 ? pos : nnz - 4;            // only rows of fewer than four entries can get here
    };
    // ---- second round trip: everything at once ----------------------------------------
    uint4 a_mem[STEPS];
    {
        const typename R::Row src = rows.row(A, arow);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) a_mem[s] = rows.unit(A, src, 4 * s + lunit, s);
    }
    auto load_b = [&](int k, uint4 (&dst)[STEPS]) {
        int64_t brow = (int64_t)(tj[k] < 0 ? 0 : tj[k]) * 16 + lrow;
        brow = brow < N ? brow : N - 1;                   // columns past N are in no row's entries
        const typename R::Row src = rows.row(B, brow);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) dst[s] = rows.unit(B, src, 4 * s + lunit, s);
    };
    // rows of up to 128 bytes: the B rows of all four tiles in flight; longer rows two tiles at a time (at 256
    // bytes four in flight cost 13 registers and a wave per SIMD of the launch that also runs rows: 22.0 -> 21.2 us)
    constexpr bool ALL_B = STEPS <= 2;
    uint4 b[ALL_B ? TILE_WINDOW : 2][STEPS];
    if constexpr (ALL_B) {
#pragma unroll
        for (int k = 0; k < TILE_WINDOW; ++k) load_b(k, b[k]);
    } else {
        load_b(0, b[0]);
    }
    const int iters = (maxcnt + 15) >> 4;                 // wave-uniform, 1..4
    I4u c_pre[2];
    F4u s_pre[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int64_t pos = entry_pos(m < iters ? m : 0);
        c_pre[m] = *reinterpret_cast<const I4u *>(col + pos);
        s_pre[m] = *reinterpret_cast<const F4u *>(sval + pos);
    }
    // ---- products of every tile into LDS ------------------------------------------------
    uint4 a[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) a[s] = to_operand(a_mem[s], s);
    auto product = [&](const uint4 (&bt)[STEPS], int k) {
        const f32x4_t sum = mfma_steps<DT, R>(a, [&](int s) { return to_operand(bt[s], s); });
        // result register i of lane (r16, q) is row 4q+i, column r16 of tile k
        *reinterpret_cast<f32x4_t *>(lds + (k * 16 + r16) * WIN_PITCH + 4 * q) = sum;
    };
    if constexpr (ALL_B) {
#pragma unroll
        for (int k = 0; k < TILE_WINDOW; ++k)
            if (tj[k] >= 0) product(b[k], k);             // wave-uniform
    } else {
#pragma unroll
        for (int k = 0; k < TILE_WINDOW; ++k) {
            if (tj[k] < 0) break;                         // wave-uniform
            if (k + 1 < TILE_WINDOW && tj[k + 1 < TILE_WINDOW ? k + 1 : k] >= 0) load_b(k + 1, b[(k + 1) & 1]);
            product(b[k & 1], k);
        }
    }
    wave_lds_order();
    // ---- entries: four per lane, 16 per row and iteration -----------------------------------
    const int t1 = tj[1], t2 = tj[2], t3 = tj[3];
    auto pick = [&](int c) {
        const int tc = c >> 4;
        const int k = (tc == t1 ? 1 : 0) + (tc == t2 ? 2 : 0) + (tc == t3 ? 3 : 0);
        return lds[(k * 16 + (c & 15)) * WIN_PITCH + lrow];
    };
    for (int m = 0; m < iters; ++m) {
        I4u c4;
        F4u s4;
        if (m < 2) { c4 = c_pre[m]; s4 = s_pre[m]; }
        else {
            const int64_t pos = entry_pos(m);
            c4 = *reinterpret_cast<const I4u *>(col + pos);
            s4 = *reinterpret_cast<const F4u *>(sval + pos);
        }
        const bool active = cnt >= 4 && 4 * lunit + 16 * m < cnt;
        const F4u out{pick(c4.x) * s4.x, pick(c4.y) * s4.y, pick(c4.z) * s4.z, pick(c4.w) * s4.w};
        if (active) *reinterpret_cast<F4u *>(P + entry_pos(m)) = out;
    }
    // rows with one to three entries in the window: entry by entry
    if (cnt > 0 && cnt < 4 && lunit == 0) {
        for (int e = 0; e < cnt; ++e) P[(int64_t)p0 + e] = pick(col[(int64_t)p0 + e]) * sval[(int64_t)p0 + e];
    }
    wave_lds_order();                                     // the next window of this wave reuses the buffer
}

constexpr int PAIR_MAX_STEPS = 4;             // row bytes / 64 up to which pairs of windows share a wavefront
// (not with ragged fp32 rows, whose sums take more registers: near-dense rows K = 48 39 us in pairs, 23 without)
constexpr bool tile_pairs(bool ragged, bool f32, int steps) { return steps <= PAIR_MAX_STEPS && !(ragged && f32); }
// Windows wa and wa+1 of a pair of gathered strips on the calling wavefront: the same four tile
// columns for 2 x 16 rows.  Every B tile is loaded and moved into operand layout once and
// multiplied with both A panels; the products of the second strip wait in registers while the
// entries of the first are picked out of the LDS buffer (one buffer, as for a single window).
template <int DT, int STEPS, class R>
__device__ __forceinline__ void tile_window_pair_wave(const R &rows, const void *__restrict__ A, const void *__restrict__ B, int M, int N,
                                                      const int32_t *__restrict__ vrows,
                                                      const int32_t *__restrict__ tile_cols,
                                                      const TileDesc *__restrict__ tiles, int64_t n_tiles,
                                                      const TileWindow *__restrict__ win, int64_t n_win,
                                                      const int32_t *__restrict__ col, const float *__restrict__ sval,
                                                      float *__restrict__ P, int64_t nnz, int64_t wa, float *lds) {
    if (wa >= n_win) return;
    const int lane = lane_id();
    const int li = lane < 48 ? lane : 47;
    const int dw0 = reinterpret_cast<const int32_t *>(win + wa)[li];
    const int dw1 = reinterpret_cast<const int32_t *>(win + (wa + 1 < n_win ? wa + 1 : wa))[li];
    bool plain = wa + 1 < n_win && __builtin_amdgcn_readlane(dw0, 44) == 0 && __builtin_amdgcn_readlane(dw1, 44) == 0 &&
                 __builtin_amdgcn_readlane(dw0, 46) != 0 && __builtin_amdgcn_readlane(dw1, 46) != 0;
    int tj[TILE_WINDOW];
#pragma unroll
    for (int k = 0; k < TILE_WINDOW; ++k) {
        tj[k] = __builtin_amdgcn_readlane(dw0, 40 + k);
        plain = plain && tj[k] == __builtin_amdgcn_readlane(dw1, 40 + k);
    }
    if (!plain) {                                         // wave-uniform: one window after the other
        for (int64_t w = wa; w < wa + 2; ++w)
            tile_window_wave<DT, STEPS>(rows, A, B, M, N, vrows, tile_cols, tiles, n_tiles, win, n_win, col, sval, P, nnz, w, lds);
        return;
    }
    const int maxcnt0 = __builtin_amdgcn_readlane(dw0, 45), maxcnt1 = __builtin_amdgcn_readlane(dw1, 45);
    if (maxcnt0 <= 0 && maxcnt1 <= 0) return;
    const int r16 = lane & 15, q = lane >> 4;        // operand / result layout
    const int lrow = lane >> 2, lunit = lane & 3;    // memory layout: four neighbouring lanes on 64 bytes of a row
    const int to_operand_from = (4 * r16 + q) << 2;
    auto to_operand = [&](const uint4 &v, int s) {     // unit 4s + q of the lane's row
        uint4 r;
        r.x = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.x);
        r.y = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.y);
        r.z = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.z);
        r.w = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.w);
        return rows.trim(r, 4 * s + q, s);
    };
    // S/P accesses of this lane in either strip: strip row lane>>2, its entries 4(lane&3)+16m.. of the window
    struct Rows { int p0, cnt; };
    auto rows_of = [&](int dw) {
        Rows r;
        r.p0 = __shfl(dw, 16 + lrow, WAVE);
        const int cw = __shfl(dw, 32 + (lrow >> 1), WAVE);
        r.cnt = (lrow & 1) ? (int)((unsigned int)cw >> 16) : (cw & 0xFFFF);
        return r;
    };
    const Rows rows0 = rows_of(dw0), rows1 = rows_of(dw1);
    auto entry_pos = [&](const Rows &r, int m) {
        int ws = 4 * lunit + 16 * m;
        ws = ws < r.cnt - 4 ? ws : r.cnt - 4;
        ws = ws < 0 ? 0 : ws;
        const int64_t pos = (int64_t)r.p0 + ws;
        return pos < nnz - 4 ? pos : nnz - 4;
    };
    // ---- second round trip: both A panels, the B tiles, the first column indices and S values ----
    uint4 a0[STEPS], a1[STEPS];
    {
        const int64_t ar0 = __shfl(dw0, lrow, WAVE), ar1 = __shfl(dw1, lrow, WAVE);
        const typename R::Row s0 = rows.row(A, ar0), s1 = rows.row(A, ar1);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            a0[s] = rows.unit(A, s0, 4 * s + lunit, s);
            a1[s] = rows.unit(A, s1, 4 * s + lunit, s);
        }
    }
    auto load_b = [&](int k, uint4 (&dst)[STEPS]) {
        int64_t brow = (int64_t)(tj[k] < 0 ? 0 : tj[k]) * 16 + lrow;
        brow = brow < N ? brow : N - 1;                   // columns past N are in no row's entries
        const typename R::Row src = rows.row(B, brow);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) dst[s] = rows.unit(B, src, 4 * s + lunit, s);
    };
    uint4 b[2][STEPS];                                    // two B tiles in flight
    load_b(0, b[0]);
    if (tj[1] >= 0) load_b(1, b[1]);                      // wave-uniform
    struct Pre { I4u c[2]; F4u s[2]; };
    auto prefetch = [&](const Rows &r, int iters) {
        Pre p;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int64_t pos = entry_pos(r, m < iters ? m : 0);
            p.c[m] = *reinterpret_cast<const I4u *>(col + pos);
            p.s[m] = *reinterpret_cast<const F4u *>(sval + pos);
        }
        return p;
    };
    const int iters0 = (maxcnt0 + 15) >> 4, iters1 = (maxcnt1 + 15) >> 4;      // wave-uniform, 0..4
    const Pre pre0 = prefetch(rows0, iters0);
    // ---- products: strip 0's into LDS, strip 1's kept ----------------------------------------------
#pragma unroll
    for (int s = 0; s < STEPS; ++s) { a0[s] = to_operand(a0[s], s); a1[s] = to_operand(a1[s], s); }
    f32x4_t keep[TILE_WINDOW];
#pragma unroll
    for (int k = 0; k < TILE_WINDOW; ++k) {
        keep[k] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (tj[k] < 0) continue;                          // wave-uniform
        f32x4_t sum0, sum1;
        if constexpr (R::RAGGED) {
            uint4 bo[STEPS];
#pragma unroll
            for (int s = 0; s < STEPS; ++s) bo[s] = to_operand(b[k & 1][s], s);
            sum0 = mfma_steps<DT, R>(a0, [&](int s) { return bo[s]; });
            sum1 = mfma_steps<DT, R>(a1, [&](int s) { return bo[s]; });
        } else {
            f32x4_t acc0[1] = {}, acc1[1] = {};
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const uint4 bo = to_operand(b[k & 1][s], s);
                mfma_unit<DT, 1>(a0[s], bo, acc0);
                mfma_unit<DT, 1>(a1[s], bo, acc1);
            }
            sum0 = acc0[0];
            sum1 = acc1[0];
        }
        // the registers of this B tile are free: the tile after the next one
        if (k + 2 < TILE_WINDOW && tj[k + 2 < TILE_WINDOW ? k + 2 : k] >= 0) load_b(k + 2, b[k & 1]);
        // result register i of lane (r16, q) is row 4q+i, column r16 of tile k
        *reinterpret_cast<f32x4_t *>(lds + (k * 16 + r16) * WIN_PITCH + 4 * q) = sum0;
        keep[k] = sum1;
    }
    wave_lds_order();
    const Pre pre1 = prefetch(rows1, iters1);             // lands while strip 0's entries are written
    // ---- entries: four per lane, 16 per row and iteration ---------------------------------------------
    const int t1 = tj[1], t2 = tj[2], t3 = tj[3];
    auto pick = [&](int c) {
        const int tc = c >> 4;
        const int k = (tc == t1 ? 1 : 0) + (tc == t2 ? 2 : 0) + (tc == t3 ? 3 : 0);
        return lds[(k * 16 + (c & 15)) * WIN_PITCH + lrow];
    };
    auto entries = [&](const Rows &r, const Pre &pre, int iters) {
        for (int m = 0; m < iters; ++m) {
            I4u c4;
            F4u s4;
            if (m < 2) { c4 = pre.c[m]; s4 = pre.s[m]; }
            else {
                const int64_t pos = entry_pos(r, m);
                c4 = *reinterpret_cast<const I4u *>(col + pos);
                s4 = *reinterpret_cast<const F4u *>(sval + pos);
            }
            const bool active = r.cnt >= 4 && 4 * lunit + 16 * m < r.cnt;
            const F4u out{pick(c4.x) * s4.x, pick(c4.y) * s4.y, pick(c4.z) * s4.z, pick(c4.w) * s4.w};
            if (active) *reinterpret_cast<F4u *>(P + entry_pos(r, m)) = out;
        }
        // rows with one to three entries in the window: entry by entry
        if (r.cnt > 0 && r.cnt < 4 && lunit == 0) {
            for (int e = 0; e < r.cnt; ++e) P[(int64_t)r.p0 + e] = pick(col[(int64_t)r.p0 + e]) * sval[(int64_t)r.p0 + e];
        }
    };
    entries(rows0, pre0, iters0);
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < TILE_WINDOW; ++k)
        if (tj[k] >= 0) *reinterpret_cast<f32x4_t *>(lds + (k * 16 + r16) * WIN_PITCH + 4 * q) = keep[k];
    wave_lds_order();
    entries(rows1, pre1, iters1);
    wave_lds_order();                                     // the next window of this wave reuses the buffer
}

// Wavefront `unit` of a tile launch: windows [0, n_single) one per wavefront, the windows after them (pairs of
// gathered strips) two per wavefront.
template <int DT, int STEPS, class R>
__device__ __forceinline__ void tile_unit_wave(const R &rows, const void *__restrict__ A, const void *__restrict__ B, int M, int N,
                                               const int32_t *__restrict__ vrows, const int32_t *__restrict__ tile_cols,
                                               const TileDesc *__restrict__ tiles, int64_t n_tiles,
                                               const TileWindow *__restrict__ win, int64_t n_win, int64_t n_single,
                                               const int32_t *__restrict__ col, const float *__restrict__ sval,
                                               float *__restrict__ P, int64_t nnz, int64_t unit, float *lds,
                                               const int32_t *__restrict__ order) {
    // (rows beyond 256 bytes: the second A panel and the kept products do not fit the registers, the
    // plan gives such launches one wavefront per window throughout)
    constexpr bool PAIRS = tile_pairs(R::RAGGED, DT == DT_F32, STEPS);
    if (!PAIRS || win == nullptr || unit < n_single) {     // wave-uniform
        tile_window_wave<DT, STEPS>(rows, A, B, M, N, vrows, tile_cols, tiles, n_tiles, win, n_win, col, sval, P, nnz, unit, lds,
                                    order);
        return;
    }
    if constexpr (PAIRS)
        tile_window_pair_wave<DT, STEPS>(rows, A, B, M, N, vrows, tile_cols, tiles, n_tiles, win, n_win, col, sval, P, nnz,
                                         n_single + 2 * (unit - n_single), lds);
}

template <int DT, int STEPS, class R>
__global__ __launch_bounds__(BLOCK) void k_tile(int64_t nblocks, const TileWindow *__restrict__ win, int64_t n_win,
    int64_t n_single, const int32_t *__restrict__ order, const void *__restrict__ A, const void *__restrict__ B, int len,
    int M, int N, const int32_t *__restrict__ vrows, const int32_t *__restrict__ tile_cols,
    const TileDesc *__restrict__ tiles, int64_t n_tiles, const int32_t *__restrict__ col, const float *__restrict__ sval,
    float *__restrict__ P, int64_t nnz) {
    __shared__ __attribute__((aligned(16))) float win_lds[WAVES_PER_BLOCK][WIN_LDS_FLOATS];
    const int64_t blk = xcd_remap(blockIdx.x, nblocks);
    if (blk < 0) return;
    tile_unit_wave<DT, STEPS>(R(len), A, B, M, N, vrows, tile_cols, tiles, n_tiles, win, n_win, n_single, col, sval, P, nnz,
                              blk * WAVES_PER_BLOCK + wave_in_block(), win_lds[wave_in_block()], order);
}

// ---- long rows, well-filled tiles: the four waves of a workgroup split K -----------------------
// A tile of long rows is 16 KB of B (1 KiB rows) for 16 MFMAs: a wavefront that walks tiles alone has
// two of them in flight, fills half the register file with them and still waits for memory most of
// the time, and a launch of a few thousand tiles is two such wavefronts per SIMD.  Here a workgroup
// takes one window of TILE_WINDOW tiles and wave j the j-th quarter of K of all of them: a quarter of
// the registers per tile, all four tiles of the window in flight, four times the wavefronts.  The
// partial 16x16 products meet in LDS (1 KiB per tile and wave); wave j then adds up tile j, scales it
// by S and scatters it from the descriptor's masks, which it loaded at the start.
constexpr int KSPLIT = WAVES_PER_BLOCK;
static_assert(KSPLIT == 4 && TILE_WINDOW == 4, "one finishing wave per tile of a window");
constexpr int KSPLIT_LDS_FLOATS = TILE_WINDOW * KSPLIT * 256;

// LONG: rows of any length (RaggedRows), STEPS of them at a time.  Error against 64 bits, of the result's norm, K = 260 .. 1 024:
// gather kernels fp32 0.96 .. 1.26e-7, fp16 0.99 .. 1.20e-7, bf16 0.65 .. 0.88e-7; here and in the panel kernel's turns, whose sums
// pass through P, 0.84 .. 0.97e-7, 0.76 .. 0.81e-7, 0.66 .. 0.72e-7 (bf16 K = 520, most of it the rounding of the result: 0.654 and
// 0.657, panels 0.656 and 0.666).
template <int DT, int STEPS, class R, bool LONG = false>
__global__ __launch_bounds__(BLOCK) void k_tile_ksplit(int64_t nblocks, const int32_t *__restrict__ order,
    const TileDesc *__restrict__ tiles, int64_t n_tiles, const int32_t *__restrict__ tile_cols, const void *__restrict__ A,
    const void *__restrict__ B, int len, int M, int N, const int32_t *__restrict__ vrows, const float *__restrict__ sval,
    float *__restrict__ P) {
    static_assert(STEPS % KSPLIT == 0, "K in four equal parts of whole 64-byte steps");
    static_assert(!LONG || R::RAGGED, "rows of any length are ragged ones");
    constexpr int SW = STEPS / KSPLIT;                    // steps of this wave
    __shared__ __attribute__((aligned(16))) float part[KSPLIT_LDS_FLOATS];
    int64_t w = xcd_remap(blockIdx.x, nblocks);
    if (w < 0) return;                                    // whole workgroups leave
    if (order) w = order[w];
    const int64_t t0 = w * TILE_WINDOW;
    if (t0 >= n_tiles) return;
    const int n = (int)(n_tiles - t0 < TILE_WINDOW ? n_tiles - t0 : TILE_WINDOW);
    const int j = wave_in_block();
    const int lane = lane_id();
    const int r16 = lane & 15, q = lane >> 4;        // operand / result layout
    const int lrow = lane >> 2, lunit = lane & 3;    // memory layout: four neighbouring lanes on 64 bytes of a row
    const int to_operand_from = (4 * r16 + q) << 2;
    const R rows(len);
    const int quarter = j * SW * 4;                       // this wave's quarter of every row: whole rows have it in the base
    const void *Aq = R::RAGGED ? A : (const void *)((const uint4 *)A + (uint32_t)quarter);
    const void *Bq = R::RAGGED ? B : (const void *)((const uint4 *)B + (uint32_t)quarter);
    int u0 = R::RAGGED ? quarter : 0;
    auto to_operand = [&](const uint4 &v, int s) {
        uint4 r;
        r.x = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.x);
        r.y = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.y);
        r.z = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.z);
        r.w = (uint32_t)__builtin_amdgcn_ds_bpermute(to_operand_from, (int)v.w);
        return rows.trim(r, u0 + 4 * s + q, STEPS);
    };
    // first round trip: strip and B rows of every tile, the per-row fields of this wave's own tile
    // (one load each: lane u of every quad asks for tile u, the values are dealt out inside the quad)
    int strip[TILE_WINDOW], bcol[TILE_WINDOW];
    {
        const int64_t t = t0 + (lunit < n ? lunit : n - 1);
        const int st = tiles[t].strip;
        const int bc = tile_cols[t * 16 + lrow];
        strip[0] = __builtin_amdgcn_readlane(st, 0); strip[1] = __builtin_amdgcn_readlane(st, 1);
        strip[2] = __builtin_amdgcn_readlane(st, 2); strip[3] = __builtin_amdgcn_readlane(st, 3);
        bcol[0] = dpp_i32<0x00>(bc); bcol[1] = dpp_i32<0x55>(bc);       // quad_perm: every lane takes lane k of its quad
        bcol[2] = dpp_i32<0xAA>(bc); bcol[3] = dpp_i32<0xFF>(bc);
    }
    const TileDesc *mine = tiles + t0 + (j < n ? j : n - 1);
    const int4 off4 = *(const int4 *)&mine->off[q * 4];
    const uint2 mask2 = *(const uint2 *)&mine->mask[q * 4];
    auto a_rows = [&](int st) {
        int64_t arow = st >= GATHERED_BASE ? (int64_t)vrows[(int64_t)(st - GATHERED_BASE) * 16 + lrow]
                                           : (int64_t)st * 16 + lrow;
        arow = arow < 0 ? 0 : (arow < M ? arow : M - 1);      // missing rows are never in a mask
        return rows.row(Aq, arow);
    };
    // second round trip: this wave's quarter of the A panel and of all B tiles, the S values of its own tile
    uint4 a[SW], b[TILE_WINDOW][SW];
    auto load = [&]() {
        const typename R::Row src = a_rows(strip[0]);
#pragma unroll
        for (int s = 0; s < SW; ++s) a[s] = rows.unit(Aq, src, u0 + 4 * s + lunit, STEPS);
#pragma unroll
        for (int k = 0; k < TILE_WINDOW; ++k) {
            int64_t brow = bcol[k];
            brow = brow < N ? brow : N - 1;               // columns past N (and the filler of a short union tile) are in no mask
            const typename R::Row src_b = rows.row(Bq, brow);
#pragma unroll
            for (int s = 0; s < SW; ++s) b[k][s] = rows.unit(Bq, src_b, u0 + 4 * s + lunit, STEPS);
        }
    };
    load();
    const unsigned int below = (1u << r16) - 1u;
    const int offs[4] = {off4.x, off4.y, off4.z, off4.w};
    const unsigned int masks[4] = {mask2.x & 0xFFFFu, mask2.x >> 16, mask2.y & 0xFFFFu, mask2.y >> 16};
    unsigned int act = 0;
    int pos[4];
    float sv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool on = j < n && ((masks[i] >> r16) & 1u);
        act |= on ? (1u << i) : 0u;
        pos[i] = on ? offs[i] + __builtin_popcount(masks[i] & below) : 0;   // (row 4q+i, column r16); entry 0 when absent
        sv[i] = sval[pos[i]];
    }
    auto products = [&](auto &&take) {                    // take(k, the sums of tile k)
#pragma unroll
        for (int s = 0; s < SW; ++s) a[s] = to_operand(a[s], s);
#pragma unroll
        for (int k = 0; k < TILE_WINDOW; ++k) {
            if (k >= n) break;                            // workgroup-uniform
            if (k > 0 && strip[k] != strip[k - 1]) {      // workgroup-uniform: the window reaches into the next strip
                const typename R::Row src = a_rows(strip[k]);
#pragma unroll
                for (int s = 0; s < SW; ++s) a[s] = to_operand(rows.unit(Aq, src, u0 + 4 * s + lunit, STEPS), s);
            }
            take(k, mfma_steps<DT, R>(a, [&](int s) { return to_operand(b[k][s], s); }));
        }
    };
    auto keep = [&](int k, const f32x4_t &sum) { *reinterpret_cast<f32x4_t *>(part + (k * KSPLIT + j) * 256 + lane * 4) = sum; };
    if constexpr (LONG) {
        f32x4_t total[TILE_WINDOW] = {};
        for (;;) {                                        // (the same number of turns in every wave)
            products([&](int k, const f32x4_t &sum) { total[k] += sum; });
            u0 += 4 * STEPS;
            if (u0 - quarter > rows.last) break;
            load();
        }
#pragma unroll
        for (int k = 0; k < TILE_WINDOW; ++k) keep(k, total[k]);
    } else {
        products(keep);
    }
    __syncthreads();
    if (j < n) {
        f32x4_t sum = *reinterpret_cast<const f32x4_t *>(part + (j * KSPLIT) * 256 + lane * 4);
#pragma unroll
        for (int jj = 1; jj < KSPLIT; ++jj) {
            const f32x4_t v = *reinterpret_cast<const f32x4_t *>(part + (j * KSPLIT + jj) * 256 + lane * 4);
            sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
        }
        // result register i is row 4*q+i, column r16
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if ((act >> i) & 1u) P[pos[i]] = sum[i] * sv[i];
    }
}

// Order of the windows for operands that exceed an XCD's L2.  The launch gives every XCD a
// contiguous eighth of the logical windows (xcd_remap); sorted by the key below, that eighth is
// one block of a RB x CB grid over (strip rows, tile columns), RB * CB = 8, walked by finer
// column slices: the XCD keeps its part of A resident and streams through its part of B once,
// instead of touching all of B from every strip (the storage order of the descriptors).
// Counting sort in three launches: histogram, scan of the WINDOW_BINS counters, scatter (the
// order inside a bin is whatever the atomics give; every entry is computed on its own, so the
// result does not depend on it).
constexpr int WINDOW_SLICES = 8;                      // column slices inside a block
constexpr int WINDOW_BINS = NUM_XCD * WINDOW_SLICES;
__device__ __forceinline__ int window_bin(const TileDesc *__restrict__ tiles, int64_t w, int64_t strip_span,
                                          int64_t tile_col_span, int RB, int CB) {
    const int4 h = *reinterpret_cast<const int4 *>(tiles + w * TILE_WINDOW);        // strip, tj, ..
    int64_t strip = h.x >= GATHERED_BASE ? h.x - GATHERED_BASE : h.x;
    strip = strip < strip_span ? strip : strip_span - 1;
    int64_t tj = h.y < 0 ? 0 : h.y;
    tj = tj < tile_col_span ? tj : tile_col_span - 1;
    const int rb = (int)(strip * RB / strip_span);
    const int fine = (int)(tj * (CB * WINDOW_SLICES) / tile_col_span);               // cb * WINDOW_SLICES + slice
    return rb * (CB * WINDOW_SLICES) + fine;
}
static __global__ __launch_bounds__(256) void k_window_histogram(const TileDesc *__restrict__ tiles, int64_t n_win,
                                                          int64_t strip_span, int64_t tile_col_span, int RB, int CB,
                                                          unsigned int *__restrict__ bins) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w < n_win) atomicAdd(&bins[window_bin(tiles, w, strip_span, tile_col_span, RB, CB)], 1u);
}
// one workgroup of WINDOW_BINS threads: counts -> start positions (also the scatter's cursors)
static __global__ __launch_bounds__(WINDOW_BINS) void k_window_offsets(unsigned int *__restrict__ bins) {
    __shared__ unsigned int v[WINDOW_BINS];
    v[threadIdx.x] = bins[threadIdx.x];
    __syncthreads();
    unsigned int before = 0;
    for (int i = 0; i < (int)threadIdx.x; ++i) before += v[i];
    bins[threadIdx.x] = before;
}
static __global__ __launch_bounds__(256) void k_window_scatter(const TileDesc *__restrict__ tiles, int64_t n_win,
                                                        int64_t strip_span, int64_t tile_col_span, int RB, int CB,
                                                        unsigned int *__restrict__ cursors, int32_t *__restrict__ order) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= n_win) return;
    const unsigned int at = atomicAdd(&cursors[window_bin(tiles, w, strip_span, tile_col_span, RB, CB)], 1u);
    order[at] = (int32_t)w;
}

// The same by one workgroup where there are few windows (the four launches and their gaps
// 35 us of a plan more, 340 to 3 000 windows).
constexpr int WINDOW_ORDER_BLOCK = 1024, WINDOW_ORDER_EACH = 8;
static __global__ __launch_bounds__(WINDOW_ORDER_BLOCK) void k_window_order(const TileDesc *__restrict__ tiles, int n_win,
                                                                            int64_t strip_span, int64_t tile_col_span, int RB, int CB,
                                                                            int32_t *__restrict__ order) {
    static_assert(WINDOW_BINS <= WINDOW_ORDER_BLOCK, "a bin per thread");
    __shared__ unsigned int count[WINDOW_BINS], cursor[WINDOW_BINS];
    const int tid = (int)threadIdx.x;
    if (tid < WINDOW_BINS) count[tid] = 0u;
    __syncthreads();
    int bin[WINDOW_ORDER_EACH];
#pragma unroll
    for (int k = 0; k < WINDOW_ORDER_EACH; ++k) {
        const int w = k * WINDOW_ORDER_BLOCK + tid;
        bin[k] = w < n_win ? window_bin(tiles, w, strip_span, tile_col_span, RB, CB) : -1;
    }
#pragma unroll
    for (int k = 0; k < WINDOW_ORDER_EACH; ++k)
        if (bin[k] >= 0) atomicAdd(&count[bin[k]], 1u);
    __syncthreads();
    if (tid < WINDOW_BINS) {
        unsigned int before = 0;
        for (int i = 0; i < tid; ++i) before += count[i];
        cursor[tid] = before;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < WINDOW_ORDER_EACH; ++k)
        if (bin[k] >= 0) order[atomicAdd(&cursor[bin[k]], 1u)] = k * WINDOW_ORDER_BLOCK + tid;
}

// AUTO in one launch when a matrix has tiles and rows: logical blocks are dealt out
// evenly between tile blocks (tile_wave), segment-item blocks and short-row blocks,
// so that every XCD gets its share of each.  Kernels of one stream run one after
// the other; two short launches leave the chip half idle twice, one launch does not.
// L: a 32-bit-offset layout of 4 * STEPS units, full-K for rows of STEPS * 64 bytes.
#ifndef SDDMM_FUSED_WAVES
#define SDDMM_FUSED_WAVES 5
#endif
template <class L, int STEPS>
__global__ __launch_bounds__(BLOCK, STEPS <= 2 ? SDDMM_FUSED_WAVES : STEPS == 4 ? 4 : 1)
void k_auto_tiles(int tile_blocks, int nblocks, int short_blocks, int longest_first, int n_win, int n_single,
                  const TileWindow *__restrict__ win, const int2 *__restrict__ short_list, const void *__restrict__ A,
                  const void *__restrict__ B, const int32_t *__restrict__ col, const float *__restrict__ sval,
                  float *__restrict__ P, int64_t nnz, int M, int N, int KU, int ts, int rpw,
                  const int32_t *__restrict__ rowptr, const unsigned char *__restrict__ owner,
                  const RowItem *__restrict__ items, int64_t n_items, const int32_t *__restrict__ vrows,
                  const int32_t *__restrict__ tile_cols, const TileDesc *__restrict__ tiles, int64_t n_tiles,
                  int64_t n_short_list, const int32_t *__restrict__ order) {
    __shared__ __attribute__((aligned(16))) float win_lds[WAVES_PER_BLOCK][WIN_LDS_FLOATS];
    int64_t tile_block = -1, item_block = -1, short_block = -1;
    if (longest_first) {
        // Workgroups start in the order of their ids, round-robin over the XCDs: on every XCD the
        // tile windows first (the longest wavefronts), then the segment items, then the chunks of
        // the entry list, each XCD with its contiguous eighth of each kind.
        // (a launch has fewer than 2^24 workgroups: eight times that is an int)
        const int x = (int)(blockIdx.x % NUM_XCD);
        int j = (int)(blockIdx.x / NUM_XCD);
        const int item_blocks = nblocks - tile_blocks - short_blocks;
        const int t_lo = x * tile_blocks / NUM_XCD, t_n = (x + 1) * tile_blocks / NUM_XCD - t_lo;
        const int i_lo = x * item_blocks / NUM_XCD, i_n = (x + 1) * item_blocks / NUM_XCD - i_lo;
        const int s_lo = x * short_blocks / NUM_XCD, s_n = (x + 1) * short_blocks / NUM_XCD - s_lo;
        if (j < t_n) tile_block = t_lo + j;
        else if ((j -= t_n) < i_n) item_block = i_lo + j;
        else if ((j -= i_n) < s_n) short_block = s_lo + j;
        else return;
    } else {
        const int64_t blk = xcd_remap(blockIdx.x, nblocks);
        if (blk < 0) return;
        const int64_t tiles_before = blk * tile_blocks / nblocks;
        if (((blk + 1) * tile_blocks / nblocks) != tiles_before) {
            tile_block = tiles_before;
        } else {
            const int64_t rb = blk - tiles_before, rest = nblocks - tile_blocks;
            const int64_t item_blocks = rest - short_blocks;
            const int64_t items_before = rb * item_blocks / rest;
            if (((rb + 1) * item_blocks / rest) != items_before) item_block = items_before;
            else short_block = rb - items_before;
        }
    }
    if (tile_block >= 0) {
        // (a ragged fp32 row is read element-wise at its end, whatever the unit of the row kernels)
        constexpr bool F32 = L::U::DT == DT_F32;
        using R = std::conditional_t<L::FULLK, WholeRows<STEPS>,
                                     RaggedRows<std::conditional_t<F32, UnitF32x4u, typename L::U>, STEPS>>;
        tile_unit_wave<L::U::DT, STEPS>(R(F32 && L::U::WHOLE ? 4 * KU : KU), A, B, M, N, vrows, tile_cols, tiles, n_tiles, win, n_win, n_single, col, sval, P,
                                        nnz, tile_block * WAVES_PER_BLOCK + wave_in_block(),
                                        win_lds[wave_in_block()], order);
        return;
    }
    if (item_block >= 0) {
        const int64_t w = item_block * WAVES_PER_BLOCK + wave_in_block();
        if (w >= n_items) return;
        const RowItem it = items[w];
        const int row = __builtin_amdgcn_readfirstlane(it.row);
        const int start = __builtin_amdgcn_readfirstlane(it.start);
        const int end = __builtin_amdgcn_readfirstlane(it.end);
        row_segment_body<L>(A, B, KU, col, sval, P, row, start, end, lane_id());
    } else {
        const int64_t sb = short_block;
        if (short_list) {
            entry_list_body<L>(A, B, KU, short_list, n_short_list, col, sval, P, sb * WAVES_PER_BLOCK + wave_in_block(),
                               lane_id());
            return;
        }
        const int64_t r0 = (sb * WAVES_PER_BLOCK + wave_in_block()) * rpw;
        if (r0 >= M) return;
        short_rows_body<L>(A, B, KU, rowptr, owner, col, sval, P, M, ts, r0, rpw, lane_id());
    }
}

// ---------------------------------------------------------------------------
// ROW PANEL on the matrix cores: 8 consecutive rows with one column list (see
// k_own_rows).  One wavefront per work item = entries [start,end) of the shared
// list, 16 columns per MFMA accumulator:
//
//     D[c][r] = sum_k B[col_c][k] * A[row0+r][k]      c = 0..15, r = 0..7 (8..15 unused)
//
// The 16 gathered B rows are the "row" operand (lane l: B row of column l&15,
// 16-byte unit 4s + (l>>4) in step s), the 8 A rows of the panel the "column"
// operand, held in registers for the whole item.  Result register i of lane l is
// D[4*(l>>4)+i][l&15]: four consecutive entries of row (l&15).  The column indices
// are read once for the 8 rows, each gathered B unit serves 8 rows.
//
// The vector memory pipeline spends its time per instruction (address cycles for 64
// lanes) and per line segment that neighbouring lanes touch (one cache lookup each),
// not per byte, so memory is accessed in a layout of its own, four neighbouring
// lanes on 64 contiguous bytes, and values change layout inside the wave through
// the LDS crossbar (ds_bpermute: no memory traffic):
//   * B:   load lane l reads gathered row l>>2, unit 4s + (l&3): 16 segments per
//          instruction instead of the 64 a load in operand layout would touch;
//          operand lane (n,q) then takes its unit from load lane 4n+q;
//   * S,P: two groups of 16 columns share one access: lane l reads / writes the four
//          consecutive entries 4(l&7).. (of the 32) of row l>>3 as one 16-byte access
//          (rows start at arbitrary 4-byte offsets; global 16-byte accesses need no
//          more alignment than that): 8 rows x 128 bytes per instruction.  Lanes 8..15
//          of every 16 hold the panel's rows a second time, so the second group's
//          results are already in place there: a select merges the two accumulators,
//          the merged one is moved into the memory layout (lane l takes from result
//          lane 16(l&3) + (l>>3) + 8((l>>2)&1)) and multiplied by S there.
//
// Pipeline: the entries are walked in chunks of 64 = 4 groups of 16 columns.  While
// chunk c computes, the B units and S values of chunk c+1 are in flight (a group is
// re-requested as soon as its registers have been consumed) and the column indices
// of chunk c+2 are being read; every load is issued whatever the position (clamped),
// so the wait counts stay exact and a group only waits for loads issued four groups
// earlier.
//
// fp32 rows of 128 bytes and more use v_mfma_f32_4x4x1_16b_f32 instead of the 16x16x4
// shape, whose accumulator the 8 panel rows fill only by half (fp32 MFMA runs at the rate
// of two plain FMAs per lane, so a half-used 16x16 accumulator is no faster than vector
// FMAs).  The instruction computes 16 independent 4x4 outer products, block b = lanes
// 4b..4b+3:  D_b[i][j] += srcA[lane 4b+i] * srcB[lane 4b+j]  (result register i of lane
// 4b+j).  Blocks are numbered (q, cg): q = k quarter (the 16-byte unit 4s+q of a row, as
// above), cg = four of the 16 gathered columns.  srcB is the gathered B row of column
// 4cg+j -- the operand layout of the 16x16 shape, unchanged.  srcA is the panel: with
// cbsz = 2 the four blocks of one q take srcA from the block that abid names, so the four
// blocks of a q hold four different things -- block cg: panel rows 4(cg&1).. of unit
// 4(2s'+(cg>>1))+q -- and one register covers two steps and both row halves: the panel
// costs STEPS/2 registers of 16 bytes (the 16x16 layout needs STEPS and repeats every
// row).  Every MFMA does 256 useful multiply-adds.  Results: register i of lane (q,cg,j)
// is (row i or 4+i, column 4cg+j), partial over q; v_permlane32_swap and
// v_permlane16_swap add the four k quarters while they deal the row halves and the two
// groups of a pair out to the lanes, a 4x4 transpose inside every quad (two DPP stages)
// turns (register = row, lane = column) into (lane = row, register = column): four
// consecutive entries of a row per lane, which then move to the memory layout as above.
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

template <int ABID>
__device__ __forceinline__ f32x4_t mfma_blocks(float a, float b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 2, ABID, 0);
}
// both row halves of the panel against one component of a gathered unit; AB = 2 * (step parity)
template <int AB>
__device__ __forceinline__ void mfma_blocks_unit(const uint4 &r, const uint4 &b, f32x4_t &lo, f32x4_t &hi) {
    lo = mfma_blocks<AB>(__builtin_bit_cast(float, r.x), __builtin_bit_cast(float, b.x), lo);
    hi = mfma_blocks<AB + 1>(__builtin_bit_cast(float, r.x), __builtin_bit_cast(float, b.x), hi);
    lo = mfma_blocks<AB>(__builtin_bit_cast(float, r.y), __builtin_bit_cast(float, b.y), lo);
    hi = mfma_blocks<AB + 1>(__builtin_bit_cast(float, r.y), __builtin_bit_cast(float, b.y), hi);
    lo = mfma_blocks<AB>(__builtin_bit_cast(float, r.z), __builtin_bit_cast(float, b.z), lo);
    hi = mfma_blocks<AB + 1>(__builtin_bit_cast(float, r.z), __builtin_bit_cast(float, b.z), hi);
    lo = mfma_blocks<AB>(__builtin_bit_cast(float, r.w), __builtin_bit_cast(float, b.w), lo);
    hi = mfma_blocks<AB + 1>(__builtin_bit_cast(float, r.w), __builtin_bit_cast(float, b.w), hi);
}
// a + b where lane l of the result pairs (first, second) as the swap instruction deals them:
// permlane32_swap: lanes 0..31 get first[l] + first[l+32], lanes 32..63 second[l-32] + second[l]
__device__ __forceinline__ float swap32_add(float first, float second) {
    const u32x2_t r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned int, first),
                                                       __builtin_bit_cast(unsigned int, second), false, false);
    // (element values first: a bit cast applied to a vector element expression reads element 0)
    const unsigned int x = r.x, y = r.y;
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
// permlane16_swap: even 16-lane rows get first[row] + first[row+1], odd rows second[row-1] + second[row]
__device__ __forceinline__ float swap16_add(float first, float second) {
    const u32x2_t r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned int, first),
                                                       __builtin_bit_cast(unsigned int, second), false, false);
    const unsigned int x = r.x, y = r.y;
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
// 4x4 transpose inside every quad of lanes: f[i] of lane j  <->  f[j] of lane i
__device__ __forceinline__ void quad_transpose(float (&f)[4], int lane) {
    const bool b0 = (lane & 1) != 0, b1 = (lane & 2) != 0;
    {
        const float t01 = dpp_f32<DPP_QUAD_XOR1>(b0 ? f[0] : f[1]);
        const float t23 = dpp_f32<DPP_QUAD_XOR1>(b0 ? f[2] : f[3]);
        f[0] = b0 ? t01 : f[0]; f[1] = b0 ? f[1] : t01;
        f[2] = b0 ? t23 : f[2]; f[3] = b0 ? f[3] : t23;
    }
    {
        const float t02 = dpp_f32<DPP_QUAD_XOR2>(b1 ? f[0] : f[2]);
        const float t13 = dpp_f32<DPP_QUAD_XOR2>(b1 ? f[1] : f[3]);
        f[0] = b1 ? t02 : f[0]; f[2] = b1 ? f[2] : t02;
        f[1] = b1 ? t13 : f[1]; f[3] = b1 ? f[3] : t13;
    }
}

// Wavefronts per workgroup: the launch is a few workgroups per CU (one work item per
// 8-row panel), so small workgroups spread more evenly over the CUs; measured 2 % faster
// with 2 than with 4 at rows of 128-256 bytes, 2-5 % slower at 512 bytes.
constexpr int panel_mfma_waves(int steps) { return steps <= 4 ? 2 : 4; }

// FUSED (rows of 128 to 512 bytes in fp32, 64 to 256 bytes in bf16 / fp16): the kernel also adds the panel's part of
//
//     O[row0+r][:] += sum over the item's columns c of P[row0+r][c] * B[col_c][:]
//
// with the same instruction in another role: block b = gathered column b of the group,
// srcA = the P values of rows 4h.. in that column (lane 4b+i: row 4h+i), srcB = the B
// unit as it was loaded (lane 4b+j: components 4j.. of unit 4s+j, no layout change), so
// register i of lane 4b+j of accumulator (h,s,comp) collects O[4h+i][16s+4j+comp] over
// the columns that block b has seen.  The P values of a pair move from the memory layout
// to srcA through a tile of LDS (one 16-byte write, four 4-byte reads per lane).  After
// the last column the 16 blocks are added with lane swaps and row rotations and every
// lane adds 2*STEPS values to O atomically (O is cleared before the launch; a row may
// be cut into several items).  Columns past the end of the item enter with srcB = 0,
// whatever their B rows hold.  16-bit operands: a B unit holds 8 components, widened to fp32 for
// the second product (P and O are fp32 whatever the operands are), so there are 8 accumulators
// per (h, s) and register i of lane 4b+j of accumulator (h,s,comp) collects O[4h+i][32s+8j+comp].
constexpr int DPP_ROW_ROR4 = 0x124, DPP_ROW_ROR8 = 0x128;   // rotation by 4 / 8 lanes inside every row of 16
constexpr int PANEL_TILE_PITCH = 48;                        // floats per row of the P tile: conflict-free 4-byte reads

// waves per SIMD the register allocation aims at: the fused kernel keeps 2 * K accumulators of the
// output rows, K = 16 * STEPS in fp32 and 32 * STEPS in 16 bits (3 waves at K = 32 -- 4 were no
// faster --, 2 at K = 64, measured 89 us against 114 us with 1; at K = 128 the accumulators leave
// room for one)
constexpr int panel_mfma_min_waves(int steps, bool fused, bool half_width = false) {
    const int k = steps * (half_width ? 32 : 16);
    return fused ? (k <= 32 ? 3 : k == 64 ? 2 : 1) : steps == 8 ? 4 : 1;
}

// SLICED: rows of any length, STEPS of them per launch from unit0 on; the launches add their sums to P in turn, the last one
// multiplies by S.
template <int DT, int STEPS, bool FUSED = false, class R = WholeRows<STEPS>, bool SLICED = false>
__global__ __launch_bounds__(panel_mfma_waves(STEPS) * WAVE, panel_mfma_min_waves(STEPS, FUSED, DT != DT_F32))
void k_panel_mfma(const RowItem *__restrict__ items, int64_t n_items, int64_t nblocks, const int32_t *__restrict__ rowptr,
                  const int32_t *__restrict__ col, const void *__restrict__ A, const void *__restrict__ B, int len,
                  const float *__restrict__ sval, float *__restrict__ P, float *__restrict__ O, int unit0) {
    static_assert(!SLICED || R::RAGGED, "rows of any length are ragged ones");
    static_assert(!FUSED || !R::RAGGED, "fused panels: whole rows");
    static_assert(!FUSED || (DT == DT_F32 ? (STEPS == 2 || STEPS == 4 || STEPS == 8) : (STEPS == 1 || STEPS == 2 || STEPS == 4)),
                  "fused panels: 32, 64 or 128 components per row");
    __shared__ __attribute__((aligned(16))) float p_tiles[FUSED ? panel_mfma_waves(STEPS) : 1][FUSED ? PANEL_ROWS * PANEL_TILE_PITCH : 4];
    const int64_t blk = xcd_remap(blockIdx.x, nblocks);
    if (blk < 0) return;
    const int64_t w = blk * panel_mfma_waves(STEPS) + wave_in_block();
    if (w >= n_items) return;
    const RowItem it = items[w];
    const int row0 = __builtin_amdgcn_readfirstlane(it.row);
    const int start = __builtin_amdgcn_readfirstlane(it.start);
    const int end = __builtin_amdgcn_readfirstlane(it.end);
    if (start >= end) return;
    const int lane = lane_id();
    const int n = lane & 15, q = lane >> 4;          // operand / result layout
    const int lrow = lane >> 2, lunit = lane & 3;    // memory layout: row, 16-byte unit inside 64 bytes
    const int to_operand_from = (4 * n + q) << 2;    // ds_bpermute address: operand lane (n,q) <- memory lane 4n+q
    // S/P layout of a pair of groups: row l>>3, 16-byte unit l&7 of the 128 bytes; units 4..7 are the
    // second group's, whose results sit in lanes 8..15 of every 16
    const int prow = lane >> 3, punit = lane & 7;
    // fp32 rows of 128 bytes and more: 4x4 blocks, every multiply-add useful (see above)
    constexpr bool BLOCKS = DT == DT_F32 && STEPS % 2 == 0;
    // the 8 rows of a panel have one length and follow each other in the CSR arrays
    const int rs0 = __builtin_amdgcn_readfirstlane(it.extra);
    const int row_len = __builtin_amdgcn_readfirstlane(rowptr[row0 + 1]) - rs0;
    const int64_t out_row = (int64_t)rs0 + (int64_t)prow * row_len;   // this lane's S/P row starts here
    // ROTATE: the S/P window of a row lags the compute window by `rot` 16-byte units, chosen so
    // that the 128 bytes which the 8 lanes of a row read and write per pair are one whole line of
    // the output array (rows start wherever the CSR arrays put them).  A lane takes unit
    // (punit - rot) mod 8 of every pair; lanes with punit < rot store it one pair later, next to
    // the first units of that pair (`held` keeps it until then), and one more store-only step
    // follows the last pair.  Unrotated accesses straddle two lines each: every line of S is then
    // requested twice and every line of P written in two halves, and both wait in L2 in between.
    constexpr bool ROTATE = !FUSED;
    int rot = 0, src_unit = punit;
    if constexpr (ROTATE) {
        rot = (int)(((((uintptr_t)P) >> 2) + (uint64_t)(out_row + start)) & 31u) >> 2;
        src_unit = (punit - rot) & 7;
    }
    const bool use_now = punit >= rot;
    const bool any_rot = ROTATE && __ballot(rot != 0) != 0;
    const int to_memory_from =
        (BLOCKS ? 32 * (prow >> 2) + 16 * (src_unit >> 2) + 4 * (src_unit & 3) + (prow & 3)
                : 16 * (src_unit & 3) + prow + 8 * (src_unit >> 2)) << 2;
    // groups of 16 columns in flight; rows of 512 bytes and more leave registers for two
    constexpr int GROUPS = STEPS >= 8 ? 2 : 4;
    const R rows(len);
    const int first_unit = SLICED ? unit0 : 0;
    const bool add = SLICED && unit0 > 0, scale = !SLICED || unit0 + 4 * STEPS > rows.last_unit();
    auto step_of = [](int s) { return SLICED ? STEPS : s; };   // (any step can hold the end of a row)
    constexpr int A_REGS = BLOCKS ? STEPS / 2 : STEPS;
    uint4 a[A_REGS];
    if constexpr (BLOCKS) {
        // block cg of every k quarter: rows 4(cg&1).. of the units 4(2s'+(cg>>1))+q
        const int cg = (lane >> 2) & 3, t = lane & 3;
        const typename R::Row src = rows.row(A, row0 + 4 * (cg & 1) + t);
        const int u0 = first_unit + 4 * (cg >> 1) + q;
#pragma unroll
        for (int s2 = 0; s2 < A_REGS; ++s2)
            a[s2] = rows.trim(rows.unit(A, src, 8 * s2 + u0, step_of(2 * s2 + 1)), 8 * s2 + u0, step_of(2 * s2 + 1));
    } else {
        // panel rows: lanes 8..15 of every 16 repeat rows 0..7, their results are not stored
        const typename R::Row src = rows.row(A, row0 + (n & 7));
#pragma unroll
        for (int s = 0; s < STEPS; ++s) a[s] = rows.trim(rows.unit(A, src, first_unit + 4 * s + q, step_of(s)), first_unit + 4 * s + q, step_of(s));
    }
    const int last = end - 1;
    auto cols_of_chunk = [&](int base) {                        // column of entry base + lane (clamped)
        const int e = base + lane < last ? base + lane : last;
        return col[rs0 + e];
    };
    struct Oper {
        uint4 b[STEPS];
    };
    auto load_oper = [&](int cc, int u) {                       // group u of the chunk whose columns are in cc
        Oper o;
        const int c = __shfl(cc, u * 16 + lrow, WAVE);
        const typename R::Row src = rows.row(B, c);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) o.b[s] = rows.unit(B, src, first_unit + 4 * s + lunit, step_of(s));
        return o;
    };
    // The S values of entries g0+4*(punit-rot) .. +3 of this lane's row: one access for the pair of
    // groups that starts at g0.  The window is clamped into the row (rows of a panel hold at
    // least 4 entries); a clamped window is never used: lanes whose four entries are not all
    // inside the item fetch their S values again.  (Requested one chunk ahead of its products;
    // two chunks ahead was measured slower, in a loop 34 against 30 us and cold 53 against 48 us
    // at 128-byte rows: a request that waits for HBM holds its place in the vector memory queue.)
    struct Window {
        F4u s, p;                                                // SLICED: and the sums so far
    };
    auto load_s = [&](int g0) {
        int e = g0 + 4 * (punit - rot);
        e = e < row_len - 4 ? e : row_len - 4;
        e = e > 0 ? e : 0;
        Window w{F4u{1.f, 1.f, 1.f, 1.f}, F4u{0.f, 0.f, 0.f, 0.f}};
        if (scale) w.s = *reinterpret_cast<const F4u *>(sval + out_row + e);          // (wave-uniform)
        if (add) w.p = *reinterpret_cast<const F4u *>(P + out_row + e);
        return w;
    };
    auto permute4 = [&](int from, uint32_t x, uint32_t y, uint32_t z, uint32_t w_) {
        uint4 r;
        r.x = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)x);
        r.y = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)y);
        r.z = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)z);
        r.w = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)w_);
        return r;
    };
    auto b_operand = [&](const Oper &o, int s) {
        return rows.trim(permute4(to_operand_from, o.b[s].x, o.b[s].y, o.b[s].z, o.b[s].w), first_unit + 4 * s + q, step_of(s));
    };
    // 4x4 blocks: both row halves of 16 columns, partial over the k quarters
    auto compute_blocks = [&](const Oper &o, f32x4_t &lo, f32x4_t &hi) {
        lo = f32x4_t{0.f, 0.f, 0.f, 0.f};
        hi = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if constexpr (BLOCKS && R::RAGGED) {                     // (added as in mfma_steps)
            struct Halves {
                f32x4_t lo, hi;
                __device__ __forceinline__ Halves operator+(const Halves &x) const { return {lo + x.lo, hi + x.hi}; }
            };
            const Halves sum = pairwise<0, STEPS>([&](auto step) {
                constexpr int s = decltype(step)::value;
                const uint4 b = b_operand(o, s);
                Halves r{};
                mfma_blocks_unit<2 * (s % 2)>(a[s / 2], b, r.lo, r.hi);
                __builtin_amdgcn_sched_group_barrier(0x080, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
                return r;
            });
            lo = sum.lo;
            hi = sum.hi;
        } else if constexpr (BLOCKS) {
#pragma unroll
            for (int s2 = 0; s2 < A_REGS; ++s2) {
                {
                    const uint4 b = b_operand(o, 2 * s2);
                    mfma_blocks_unit<0>(a[s2], b, lo, hi);
                    __builtin_amdgcn_sched_group_barrier(0x080, 4, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
                }
                {
                    const uint4 b = b_operand(o, 2 * s2 + 1);
                    mfma_blocks_unit<2>(a[s2], b, lo, hi);
                    __builtin_amdgcn_sched_group_barrier(0x080, 4, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
                }
            }
        }
    };
    auto compute = [&](const Oper &o) {
        if constexpr (BLOCKS) return f32x4_t{0.f, 0.f, 0.f, 0.f};
        else if constexpr (R::RAGGED) {
            // (the gathered rows are the "row" operand)
            uint4 b[STEPS];
#pragma unroll
            for (int s = 0; s < STEPS; ++s) b[s] = b_operand(o, s);
            return mfma_steps<DT, R>(b, [&](int s) { return a[s]; });
        } else {
            f32x4_t acc[1] = {};
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                mfma_unit<DT, 1>(b_operand(o, s), a[s], acc);
                // Order of issue: the four permutes of a step, then its four MFMAs.  Left alone the
                // compiler pairs every MFMA with one permute and a wait for it (16 LDS round trips
                // per 16 columns in the wave's dependency chain instead of 4); whole groups of 8 or
                // 16 permutes ahead of their MFMAs were measured slower than either.
                if constexpr (DT == DT_F32) {
                    __builtin_amdgcn_sched_group_barrier(0x080, 4, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                }
            }
            return acc[0];
        }
    };
    // FUSED: accumulator (h, s, comp) of the output rows, see above
    constexpr int COMPS = DT == DT_F32 ? 4 : 8;                 // components of a 16-byte unit
    f32x4_t oacc[2][STEPS][COMPS];
    if constexpr (FUSED) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int k = 0; k < COMPS; ++k) oacc[h][s][k] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    auto fused_accumulate = [&](const Oper &o, float p_lo, float p_hi, int gbase) {
        const bool live = gbase + lrow < end;                    // this block's column belongs to the item
#pragma unroll
        for (int s = 0; s < (FUSED ? STEPS : 0); ++s) {
            const uint4 b = o.b[s];
            const unsigned int ux = live ? b.x : 0u, uy = live ? b.y : 0u, uz = live ? b.z : 0u, uw = live ? b.w : 0u;
            float bv[COMPS];
            if constexpr (DT == DT_F32) {
                bv[0] = __builtin_bit_cast(float, ux); bv[1] = __builtin_bit_cast(float, uy);
                bv[2] = __builtin_bit_cast(float, uz); bv[3] = __builtin_bit_cast(float, uw);
            } else {
                using U16 = std::conditional_t<DT == DT_BF16, UnitBF16x8, UnitF16x8>;
                bv[0] = U16::lo(ux); bv[1] = U16::hi(ux); bv[2] = U16::lo(uy); bv[3] = U16::hi(uy);
                bv[4] = U16::lo(uz); bv[5] = U16::hi(uz); bv[6] = U16::lo(uw); bv[7] = U16::hi(uw);
            }
#pragma unroll
            for (int k = 0; k < COMPS; ++k) {
                oacc[0][s][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(p_lo, bv[k], oacc[0][s][k], 0, 0, 0);
                oacc[1][s][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(p_hi, bv[k], oacc[1][s][k], 0, 0, 0);
            }
        }
    };
    // groups o0 (entries g0..g0+15) and o1 (g0+16..g0+31) of the shared column list
    float held[4] = {0.f, 0.f, 0.f, 0.f};                        // ROTATE: the unit taken from the previous pair
    auto compute_store_pair = [&](const Oper &o0, const Oper &o1, const Window &win, int g0) {
        if (g0 >= end + (any_rot ? 32 : 0)) return;              // wave-uniform
        const bool past = g0 >= end;                             // the store-only step after the last pair
        float r0 = 0.f, r1 = 0.f, r2 = 0.f, r3 = 0.f;
        if (past) {
        } else if constexpr (BLOCKS) {
            f32x4_t lo0, hi0, lo1, hi1;
            compute_blocks(o0, lo0, hi0);
            compute_blocks(o1, lo1, hi1);                        // columns clamped past the end: computed, not stored
            // register i of lane (q,cg,j): row i (lo) / 4+i (hi), column 4cg+j of its group, partial
            // over q = (bit 5, bit 4) of the lane.  First swap: the two lane halves add up, the lower
            // keeps rows 0..3, the upper rows 4..7; second swap: the 16-lane rows add up, even rows
            // keep the first group, odd rows the second.  Lane (b5,b4,cg,j), register i is then
            // (row 4 b5 + i, column 16 b4 + 4 cg + j of the pair); the transpose makes it
            // (row 4 b5 + j, columns 16 b4 + 4 cg + i).
            float f[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float g_first = swap32_add(lo0[i], hi0[i]);
                const float g_second = swap32_add(lo1[i], hi1[i]);
                f[i] = swap16_add(g_first, g_second);
            }
            quad_transpose(f, lane);
            r0 = f[0]; r1 = f[1]; r2 = f[2]; r3 = f[3];
        } else {
            const f32x4_t acc0 = compute(o0);
            const f32x4_t acc1 = compute(o1);                    // columns clamped past the end: computed, not stored
            // result lane (n,q) holds entries 4q.. of its group for row n&7: lanes with n < 8 keep
            // the first group's, lanes with n >= 8 the second group's; memory lane l wants row l>>3,
            // entries g0+4(l&7)..
            // (element values first: a bit cast applied to a vector element expression reads element 0)
            const bool second = (n & 8) != 0;
            r0 = second ? acc1[0] : acc0[0]; r1 = second ? acc1[1] : acc0[1];
            r2 = second ? acc1[2] : acc0[2]; r3 = second ? acc1[3] : acc0[3];
        }
        const uint4 m = permute4(to_memory_from, __builtin_bit_cast(uint32_t, r0), __builtin_bit_cast(uint32_t, r1),
                                 __builtin_bit_cast(uint32_t, r2), __builtin_bit_cast(uint32_t, r3));
        float d0 = __builtin_bit_cast(float, m.x), d1 = __builtin_bit_cast(float, m.y);
        float d2 = __builtin_bit_cast(float, m.z), d3 = __builtin_bit_cast(float, m.w);
        if constexpr (ROTATE) {
            const float n0 = d0, n1 = d1, n2 = d2, n3 = d3;
            d0 = use_now ? n0 : held[0]; d1 = use_now ? n1 : held[1];
            d2 = use_now ? n2 : held[2]; d3 = use_now ? n3 : held[3];
            held[0] = n0; held[1] = n1; held[2] = n2; held[3] = n3;
        }
        const int e = g0 + 4 * (punit - rot);
        float p[4] = {0.f, 0.f, 0.f, 0.f};                       // FUSED: the P values, 0 past the end of the item
        if (e < start) {
            // ROTATE, first pair: these lanes' first unit comes with the next pair
        } else if (e + 4 <= end) {
            // four consecutive entries inside the item (so the S window was not clamped)
            const F4u sw = win.s;
            if constexpr (SLICED) { d0 += win.p.x; d1 += win.p.y; d2 += win.p.z; d3 += win.p.w; }
            F4u out{d0 * sw.x, d1 * sw.y, d2 * sw.z, d3 * sw.w};
            *reinterpret_cast<F4u *>(P + out_row + e) = out;
            p[0] = out.x; p[1] = out.y; p[2] = out.z; p[3] = out.w;
        } else {
            // the item ends inside these four: entry by entry, S values fetched again
            const float d[4] = {d0, d1, d2, d3};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (e + i < end) {
                    float sum = d[i];
                    if constexpr (SLICED) sum += add ? P[out_row + e + i] : 0.f;
                    p[i] = scale ? sum * sval[out_row + e + i] : sum;
                    P[out_row + e + i] = p[i];
                }
        }
        if constexpr (FUSED) {
            float *tile = p_tiles[wave_in_block()];
            const f32x4_t pv = {p[0], p[1], p[2], p[3]};
            *reinterpret_cast<f32x4_t *>(tile + prow * PANEL_TILE_PITCH + 4 * punit) = pv;
            wave_lds_order();
            // lane 4b+i: row 4h+i, column b of the first / second group
            const float *src = tile + (lane & 3) * PANEL_TILE_PITCH + lrow;
            const float p0_lo = src[0], p0_hi = src[4 * PANEL_TILE_PITCH];
            const float p1_lo = src[16], p1_hi = src[4 * PANEL_TILE_PITCH + 16];
            wave_lds_order();
            fused_accumulate(o0, p0_lo, p0_hi, g0);
            fused_accumulate(o1, p1_lo, p1_hi, g0 + 16);
        }
    };

    constexpr int CHUNK = GROUPS * 16;                          // columns per loop iteration (<= 64)
    Oper o[GROUPS];
    // Loads complete in issue order and a wait names how many of the most recent ones
    // may still be in flight.  The waits inside the loop must hold on the way in from
    // this prologue too, so the prologue issues its loads in the order the loop does
    // (both column loads first, then the groups in the order they are consumed);
    // otherwise the loop would wait for almost everything it has just requested.
    Window s_cur[GROUPS / 2];
    const int cc0 = cols_of_chunk(start);
    int cc_nxt = cols_of_chunk(start + CHUNK);                  // columns of the next chunk
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < GROUPS; ++u) {
        o[u] = load_oper(cc0, u);
        if ((u & 1) == 0) s_cur[u / 2] = load_s(start + 16 * u);
        __builtin_amdgcn_sched_barrier(0);
    }
    const int walk_end = end + (any_rot ? 32 : 0);
    for (int base = start; base < walk_end; base += CHUNK) {
        const int cc_nn = cols_of_chunk(base + 2 * CHUNK);
#pragma unroll
        for (int u = 0; u < GROUPS; u += 2) {
            compute_store_pair(o[u], o[u + 1], s_cur[u / 2], base + 16 * u);
            o[u] = load_oper(cc_nxt, u);
            o[u + 1] = load_oper(cc_nxt, u + 1);
            s_cur[u / 2] = load_s(base + CHUNK + 16 * u);
        }
        cc_nxt = cc_nn;
    }
    if constexpr (FUSED) {
        // Register i of lane 4b+j of accumulator (h,s,comp) is O[4h+i][(4s+j) COMPS + comp] over block
        // b's columns.  The swaps add the four rows of 16 lanes while dealing the registers out: row r
        // of the wave keeps register {0,2,1,3}[r]; the rotations add the four blocks of a row.  All
        // four blocks then hold the same 16 sums; block cg adds the ones of components cg (and 4+cg) to O.
        const int r16 = lane >> 4, cg = (lane >> 2) & 3;
        const int orow = row0 + ((r16 & 1) << 1 | (r16 >> 1));
        constexpr int K = STEPS * 4 * COMPS;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
#pragma unroll
                for (int c4 = 0; c4 < COMPS; c4 += 4) {
                    float w4[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const f32x4_t v = oacc[h][s][c4 + k];
                        const float t0 = swap32_add(v[0], v[1]);
                        const float t1 = swap32_add(v[2], v[3]);
                        float x = swap16_add(t0, t1);
                        x += dpp_f32<DPP_ROW_ROR4>(x);
                        x += dpp_f32<DPP_ROW_ROR8>(x);
                        w4[k] = x;
                    }
                    const float mine = cg == 0 ? w4[0] : cg == 1 ? w4[1] : cg == 2 ? w4[2] : w4[3];
                    atomicAdd(O + (int64_t)(orow + 4 * h) * K + (4 * s + (lane & 3)) * COMPS + c4 + cg, mine);
                }
            }
        }
    }
}

}  // namespace sddmm
