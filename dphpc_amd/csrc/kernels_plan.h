// Structure kernels of the plan phase: validation, CSR<->COO index expansion,
// row statistics.  Everything that looks at S's pattern runs here, on the
// device; the host reads back only the small PlanCounters block.
#pragma once
#include "device_utils.h"
#include "plan_rules.h"

namespace sddmm {

// Host-side summary of what the structure kernels counted.
struct PlanCounters {
    unsigned int bad_pattern;      // != 0: malformed CSR/COO
    unsigned int coo_unsorted;     // != 0: COO rows not non-decreasing
    unsigned int max_len;          // longest row
    unsigned long long coo_jumps;  // entries that share neither row nor column with the one before them
    unsigned long long col_pairs, col_near;     // a sample of neighbouring entries, those in the same 16 columns
    unsigned long long rows_nonempty;
    unsigned long long rows_short, rows_medium, rows_long;
    unsigned long long nnz_short, nnz_medium, nnz_long;
    unsigned long long n_items;    // work items of the wave-per-segment kernel
    unsigned long long n_tiles, nnz_tiles, tiles_scanned;     // dense-tile path: 16-row and gathered strips
    unsigned long long n_utiles, nnz_utiles, utiles_scanned;  // dense-tile path: union strips
    unsigned long long n_panels, nnz_panels, panel_items;     // row-panel path
    unsigned long long either_tiles, nnz_either_strip, nnz_either_panels;      // strips of two panels: tiles, entries of either choice
    unsigned int fused_longest;    // fused call: longest row that its gather kernels take
    unsigned int fused_window;     // fused call: most pieces of cut rows among the rows of a wavefront
    unsigned long long rows_alike; // fused call, every fourth row: work-item rows like the next row (its length, its first column)
};

// The same counters on the device.  Sums that thousands of workgroups contribute to
// are spread over SPREAD slots chosen by workgroup id (same-address atomics were
// measured at ~10 ns each, which made the counting kernels atomic-bound);
// report_totals adds the slots up.
constexpr int SPREAD = 64;
enum CounterKind {
    K_ROWS_NONEMPTY = 0,
    K_ROWS_SHORT, K_ROWS_MEDIUM, K_ROWS_LONG, K_NNZ_SHORT, K_NNZ_MEDIUM, K_NNZ_LONG,   // row classifier
    K_ROWS_ALIKE, K_LONGEST, K_WINDOW,                                                 // and for the fused call (two maxima)
    K_TILES, K_NNZ_TILES, K_UTILES, K_NNZ_UTILES,                                      // ownership classifiers
    K_EITHER_TILES, K_NNZ_EITHER_STRIP, K_NNZ_EITHER_PANELS, K_PANELS, K_NNZ_PANELS,
    K_COO_JUMPS,                                                                       // validation of COO entries
    K_COL_PAIRS, K_COL_NEAR,                                                           // and of column indices (a sample)
    K_KINDS
};
struct DevCounters {
    unsigned int bad_pattern, coo_unsorted, pad0, pad1;
    // (from here on in the order of DevTotals)
    unsigned long long n_items, tiles_scanned, panel_items;          // scan totals, one writer each
    unsigned long long n_candidates;                                 // rows offered to the gathered strips
    unsigned long long utiles_scanned, short_scanned;                // scan totals: union strips, entries of the short rows
    unsigned long long long_scanned;                                 // scan total: rows of more than one item
    unsigned long long fused_pieces, fused_cut;                      // places given to the pieces of cut rows, to those rows
    unsigned long long block_items[2];                               // work items of k_flat_blocks: segments, gaps
    unsigned int max_len[SPREAD];
    unsigned long long k[K_KINDS][SPREAD];
};

__device__ __forceinline__ void spread_add(DevCounters *dc, int kind, unsigned long long v) {
    if (v) atomicAdd(&dc->k[kind][blockIdx.x & (SPREAD - 1)], v);
}

// What the host reads: the scan totals (in the order of DevCounters) and the sums, or maxima, over the slots.  The last launch
// before the host waits writes it to pinned memory (k_scan_jobs).  (A copy of the slots was a launch and a gap more, and their
// sum work of the host: new pattern with every call, 30 000 near-dense and short rows 170 us, so 167; graph of 200 000 rows 242
// and 234.)
struct DevTotals {
    unsigned int bad_pattern, coo_unsorted, max_len, pad;
    unsigned long long n_items, tiles_scanned, panel_items, n_candidates, utiles_scanned, short_scanned, long_scanned;
    unsigned long long k[K_KINDS];
};
constexpr int SCAN_TOTALS = 7;

inline PlanCounters summarize(const DevTotals &d) {
    PlanCounters p{};
    p.bad_pattern = d.bad_pattern;
    p.coo_unsorted = d.coo_unsorted;
    p.max_len = d.max_len;
    p.rows_nonempty = d.k[K_ROWS_NONEMPTY];
    p.coo_jumps = d.k[K_COO_JUMPS];
    p.col_pairs = d.k[K_COL_PAIRS]; p.col_near = d.k[K_COL_NEAR];
    p.rows_alike = d.k[K_ROWS_ALIKE];
    p.rows_short = d.k[K_ROWS_SHORT]; p.rows_medium = d.k[K_ROWS_MEDIUM]; p.rows_long = d.k[K_ROWS_LONG];
    p.nnz_short = d.k[K_NNZ_SHORT]; p.nnz_medium = d.k[K_NNZ_MEDIUM]; p.nnz_long = d.k[K_NNZ_LONG];
    p.n_tiles = d.k[K_TILES]; p.nnz_tiles = d.k[K_NNZ_TILES];
    p.n_utiles = d.k[K_UTILES]; p.nnz_utiles = d.k[K_NNZ_UTILES]; p.utiles_scanned = d.utiles_scanned;
    p.n_panels = d.k[K_PANELS]; p.nnz_panels = d.k[K_NNZ_PANELS];
    p.either_tiles = d.k[K_EITHER_TILES];
    p.nnz_either_strip = d.k[K_NNZ_EITHER_STRIP]; p.nnz_either_panels = d.k[K_NNZ_EITHER_PANELS];
    p.fused_longest = (unsigned int)d.k[K_LONGEST];
    p.fused_window = (unsigned int)d.k[K_WINDOW];
    p.n_items = d.n_items; p.tiles_scanned = d.tiles_scanned; p.panel_items = d.panel_items;
    return p;
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    return v;
}
// (values below 2^31)
__device__ __forceinline__ unsigned int wave_max_u32(unsigned int v) {
    const int m = min16(-(int)v);
    const int a = __builtin_amdgcn_readlane(m, 0), b = __builtin_amdgcn_readlane(m, 16);
    const int c = __builtin_amdgcn_readlane(m, 32), e = __builtin_amdgcn_readlane(m, 48);
    const int x = a < b ? a : b, y = c < e ? c : e;
    return (unsigned int)-(x < y ? x : y);
}

// What a plan clears before its classifiers run, in one launch (a fill through the
// runtime is a launch of its own for every region): the row-ownership bytes (owner_bytes 0: k_own_rows writes them all),
// the sums of the row classes (n_sums words) and every counter except what validation measured (non-empty rows, longest row).
static __global__ __launch_bounds__(256) void k_plan_reset(unsigned char *__restrict__ owner, int64_t owner_bytes,
                                                    unsigned int *__restrict__ sums, int64_t n_sums, DevCounters *pc) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_sums) sums[i] = 0u;
    // 16 bytes per thread (the array is 256-byte aligned and padded to 64 bytes past the rows)
    const int64_t at = i * 16;
    if (at + 16 <= owner_bytes) *reinterpret_cast<uint4 *>(owner + at) = make_uint4(0u, 0u, 0u, 0u);
    else for (int64_t q = at; q < owner_bytes; ++q) owner[q] = 0;
    if (blockIdx.x == 0) {
        for (int k = K_ROWS_SHORT; k <= K_NNZ_PANELS; ++k)
            for (int sl = threadIdx.x; sl < SPREAD; sl += blockDim.x) pc->k[k][sl] = 0ull;
        if (threadIdx.x == 0) {
            pc->n_items = 0ull;
            pc->short_scanned = 0ull;
            pc->long_scanned = 0ull;
            pc->tiles_scanned = 0ull; pc->panel_items = 0ull; pc->n_candidates = 0ull; pc->utiles_scanned = 0ull;
        }
    }
}

// What a new pattern starts from, in one launch (as fills of the runtime 14 us): no entry of P computed, no counter counted.
// P is 16-byte aligned.
static __global__ __launch_bounds__(256) void k_clear_pattern(float *__restrict__ P, int64_t nnz, unsigned int *__restrict__ pc) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = t * 4; i < nnz; i += stride * 4) {
        if (i + 4 <= nnz) *reinterpret_cast<float4 *>(P + i) = make_float4(0.f, 0.f, 0.f, 0.f);
        else for (int64_t q = i; q < nnz; ++q) P[q] = 0.f;
    }
    if (blockIdx.x == 0)
        for (int q = (int)threadIdx.x; q < (int)(sizeof(DevCounters) / sizeof(unsigned int)); q += 256) pc[q] = 0u;
}

// bits of DevCounters::bad_pattern
constexpr unsigned int BAD_POINTER = 1, BAD_INDEX = 2;

// rowptr[0]==0, rowptr[M]==nnz, non-decreasing; also counts non-empty rows and the
// longest row.  One lane per row, one set of atomics per workgroup.
static __global__ __launch_bounds__(256) void k_check_rowptr(const int32_t *__restrict__ rowptr, int M,
                                                      int64_t nnz, DevCounters *pc) {
    __shared__ unsigned int sh_ne, sh_mx, sh_bad;
    if (threadIdx.x == 0) { sh_ne = 0; sh_mx = 0; sh_bad = 0; }
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned int bad = 0, len = 0;
    if (i < M) {
        const int32_t s = rowptr[i], e = rowptr[i + 1];
        if (e < s || s < 0) bad = 1; else len = (unsigned int)(e - s);
        if (i == 0 && s != 0) bad = 1;
        if (i == M - 1 && (int64_t)e != nnz) bad = 1;
    }
    const unsigned int ne = (unsigned int)__builtin_popcountll(__ballot(len > 0));
    const unsigned int mx = wave_max_u32(len);
    const unsigned long long anybad = __ballot(bad != 0);
    if (lane_id() == 0) {
        if (ne) atomicAdd(&sh_ne, ne);
        if (mx) atomicMax(&sh_mx, mx);
        if (anybad) atomicOr(&sh_bad, 1u);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        spread_add(pc, K_ROWS_NONEMPTY, sh_ne);
        if (sh_mx) atomicMax(&pc->max_len[blockIdx.x & (SPREAD - 1)], sh_mx);
        if (sh_bad) atomicOr(&pc->bad_pattern, BAD_POINTER);
    }
}

// every column index in [0,N).  Does nothing after a launch of k_check_rowptr that found the row pointer malformed: the
// array need not hold n values then (the host reads both verdicts at once: one wait for the device, 20 us, instead of two).
// sample: also counts, on some of the entries, how often neighbours lie in the same 16 columns.
static __global__ __launch_bounds__(256) void k_check_index(const int32_t *__restrict__ idx, int64_t n,
                                                     int bound, int sample, DevCounters *pc) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x * 4;
    if (pc->bad_pattern & BAD_POINTER) return;              // (this kernel sets the other bit only)
    unsigned int bad = 0, pairs = 0, near = 0;
    for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; i < n; i += stride) {
        if (i + 4 <= n) {
            const I4u c = *reinterpret_cast<const I4u *>(idx + i);
            bad |= (unsigned int)c.x >= (unsigned int)bound || (unsigned int)c.y >= (unsigned int)bound ||
                   (unsigned int)c.z >= (unsigned int)bound || (unsigned int)c.w >= (unsigned int)bound ? 1u : 0u;
            pairs += 3;
            near += ((c.x >> 4) == (c.y >> 4)) + ((c.y >> 4) == (c.z >> 4)) + ((c.z >> 4) == (c.w >> 4));
        } else {
            for (int64_t q = i; q < n; ++q) bad |= (unsigned int)idx[q] >= (unsigned int)bound ? 1u : 0u;
        }
    }
    if (__ballot(bad != 0) && lane_id() == 0) atomicOr(&pc->bad_pattern, BAD_INDEX);
    if (!sample) return;
    // 64 to 128 workgroups count (thousands would wait for each other's atomics: 14 M entries 13 us, 24 with 1 700 of them)
    const unsigned int each = gridDim.x > SPREAD ? gridDim.x / SPREAD : 1u;
    if (blockIdx.x % each == 0) {
        pairs = wave_sum_i32(pairs);
        near = wave_sum_i32(near);
        if (lane_id() == 0) {
            atomicAdd(&pc->k[K_COL_PAIRS][(blockIdx.x / each) & (SPREAD - 1)], (unsigned long long)pairs);
            atomicAdd(&pc->k[K_COL_NEAR][(blockIdx.x / each) & (SPREAD - 1)], (unsigned long long)near);
        }
    }
}

// rowptr -> row index per stored entry (what the flat kernels read).  A wavefront
// takes 64 rows: short rows are written by their own lane, long ones by the
// whole wavefront.  Positions outside [0, limit) are never written, whatever the
// row pointer holds (it may come unvalidated from the caller).
static __global__ __launch_bounds__(256) void k_expand_rows(const int32_t *__restrict__ rowptr, int M,
                                                     int32_t *__restrict__ rowidx, int64_t limit) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = lane_id();
    int32_t s = 0, e = 0;
    if (i < M) {
        s = rowptr[i];
        e = rowptr[i + 1];
        s = s < 0 ? 0 : s;
        e = (int64_t)e > limit ? (int32_t)limit : e;
    }
    const int len = e - s;
    constexpr int SHORT = 8;
    if (len <= SHORT) {
        for (int q = 0; q < len; ++q) rowidx[s + q] = (int32_t)i;
    }
    unsigned long long longmask = __ballot(len > SHORT);
    while (longmask) {
        const int src = __builtin_ctzll(longmask);
        longmask &= longmask - 1;
        const int32_t ss = __shfl(s, src, WAVE), ee = __shfl(e, src, WAVE);
        const int32_t rr = (int32_t)(i - lane + src);
        for (int32_t q = ss + lane; q < ee; q += WAVE) rowidx[q] = rr;
    }
}

// COO rows non-decreasing?  (one lane per entry)  Also counts the entries that share neither row nor column
// with the entry before them.  One set of atomics per workgroup: from every wavefront, the flag alone took
// 214 us for 1.2 M entries in no order (6 us now).
static __global__ __launch_bounds__(256) void k_check_coo_sorted(const int32_t *__restrict__ row,
                                                          const int32_t *__restrict__ col, int64_t nnz,
                                                          DevCounters *pc) {
    __shared__ unsigned int sh_uns, sh_jumps;
    if (threadIdx.x == 0) { sh_uns = 0; sh_jumps = 0; }
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    unsigned int uns = 0, jumps = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i + 1 < nnz; i += stride) {
        const int r0 = row[i], r1 = row[i + 1];
        uns |= r0 > r1 ? 1u : 0u;
        jumps += r0 != r1 && col[i] != col[i + 1] ? 1u : 0u;
    }
    const unsigned int any = __ballot(uns != 0) != 0 ? 1u : 0u;
    for (int o = 32; o > 0; o >>= 1) jumps += __shfl_xor(jumps, o, WAVE);
    if (lane_id() == 0) {
        if (any) atomicOr(&sh_uns, 1u);
        atomicAdd(&sh_jumps, jumps);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (sh_uns) atomicOr(&pc->coo_unsorted, 1u);
        spread_add(pc, K_COO_JUMPS, sh_jumps);
    }
}

// sorted COO row array -> rowptr.  Entry n closes every row in (row[n-1], row[n]].
static __global__ __launch_bounds__(256) void k_rowptr_from_sorted_coo(const int32_t *__restrict__ row,
                                                                int64_t nnz, int M,
                                                                int32_t *__restrict__ rowptr) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n > nnz) return;
    const int lo = n == 0 ? -1 : row[n - 1];
    const int hi = n == nnz ? M : row[n];
    for (int r = lo + 1; r <= hi; ++r) rowptr[r] = (int32_t)n;
}

}  // namespace sddmm

// ===========================================================================
// Row classifier of the AUTO strategy.
//
// A row is "short" when it has fewer than `ts` stored entries; short rows are
// computed by k_short_rows straight from rowptr, 64 consecutive rows per
// wavefront, and need no list.  Every other row becomes ceil(len/seg) work items
// of the wave-per-segment kernel; the item list is built with an exclusive scan
// of the per-row item counts (three kernels: block sums, scan of the block sums,
// write).  Nothing here touches col/values: the cost is O(M).
namespace sddmm {

constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 4;                       // rows per thread
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;  // rows per block

// owner (may be null): one byte per row, non-zero when the dense-tile path (1: a
// 16-row strip, 3: a strip of rows gathered by column window) or the row-panel path
// (2) computes the row; such rows count as empty here
// (only != 0: just the rows of that owner count as empty)
__device__ __forceinline__ unsigned int row_item_count(unsigned int len, int ts, int seg) {
    return len >= (unsigned int)ts ? (len + seg - 1) / seg : 0u;
}

// lengths of the SCAN_ITEMS rows from `base` on, 0 for those that do not exist or have an owner (as row_item_count)
__device__ __forceinline__ void row_lengths(const int32_t *__restrict__ rowptr, const unsigned char *__restrict__ owner,
                                            int64_t base, int M, unsigned int (&len)[SCAN_ITEMS], int only = 0) {
    static_assert(SCAN_ITEMS == 4, "one 16-byte load of the row pointer");
    if (base + SCAN_ITEMS <= M) {                              // one round trip instead of one per row
        const I4u p = *reinterpret_cast<const I4u *>(rowptr + base);
        const int last = rowptr[base + SCAN_ITEMS];
        uint32_t own = 0;
        if (owner) own = *reinterpret_cast<const uint32_t *>(owner + base);
        const int at[SCAN_ITEMS + 1] = {p.x, p.y, p.z, p.w, last};
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS; ++q) {
            const uint32_t o = (own >> (8 * q)) & 0xFFu;
            len[q] = (only ? o == (uint32_t)only : o != 0u) ? 0u : (unsigned int)(at[q + 1] - at[q]);
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        const int64_t i = base + q;
        const bool on = i < M && !(owner && (only ? owner[i] == only : owner[i] != 0));
        len[q] = on ? (unsigned int)(rowptr[i + 1] - rowptr[i]) : 0u;
    }
}

// block-wide exclusive scan of one value per thread (SCAN_BLOCK threads); returns
// the exclusive prefix, *total receives the block sum
__device__ __forceinline__ unsigned int block_exclusive_scan(unsigned int v, unsigned int *total) {
    __shared__ unsigned int wave_sums[SCAN_BLOCK / WAVE];
    const int lane = lane_id(), wid = threadIdx.x >> 6;
    const unsigned int incl = (unsigned int)wave_inclusive_sum((int)v);
    if (lane == WAVE - 1) wave_sums[wid] = incl;
    __syncthreads();
    unsigned int before = 0, all = 0;
    for (int w = 0; w < SCAN_BLOCK / WAVE; ++w) {
        const unsigned int s = wave_sums[w];
        if (w < wid) before += s;
        all += s;
    }
    __syncthreads();
    *total = all;
    return before + incl - v;
}

// pass 1: items per block of SCAN_TILE rows, plus the row statistics
static __global__ __launch_bounds__(SCAN_BLOCK) void k_classify_count(const int32_t *__restrict__ rowptr,
                                                               const unsigned char *__restrict__ owner, int M,
                                                               int ts, int seg, unsigned int *__restrict__ block_sums,
                                                               DevCounters *pc, int only,
                                                               unsigned int *__restrict__ short_sums,
                                                               unsigned int *__restrict__ long_sums,
                                                               const int32_t *__restrict__ col, int window) {
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    unsigned int items = 0, longest = 0, pieces = 0;
    unsigned int r_alike = 0;
    unsigned long long r_short = 0, r_med = 0, r_long = 0, n_short = 0, n_med = 0, n_long = 0;
    unsigned int lens[SCAN_ITEMS];
    row_lengths(rowptr, owner, base, M, lens, only);
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        const unsigned int len = lens[q], cnt = row_item_count(len, ts, seg);
        items += cnt;
        longest = len > longest ? len : longest;
        pieces += cnt > 1 ? cnt : 0;
        if (len == 0) continue;
        if (q == 0 && col && cnt > 0 && base + 1 < M) {         // (a sample: the chain of loads of every row takes 5 us)
            const int32_t a = rowptr[base], b = rowptr[base + 1];
            if ((unsigned int)(rowptr[base + 2] - b) == len && col[a] == col[b]) r_alike = 1;
        }
        if (cnt == 0) { ++r_short; n_short += len; }
        else if (cnt == 1) { ++r_med; n_med += len; }
        else { ++r_long; n_long += len; }
    }
    unsigned int total;
    (void)block_exclusive_scan(items, &total);
    if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
    // statistics: wave sums, then one set of atomics per workgroup
    __shared__ unsigned long long sh[6];
    if (threadIdx.x < 6) sh[threadIdx.x] = 0;
    __syncthreads();
    r_short = wave_sum_u64(r_short); r_med = wave_sum_u64(r_med); r_long = wave_sum_u64(r_long);
    n_short = wave_sum_u64(n_short); n_med = wave_sum_u64(n_med); n_long = wave_sum_u64(n_long);
    if (lane_id() == 0) {
        if (r_short) atomicAdd(&sh[0], r_short);
        if (r_med) atomicAdd(&sh[1], r_med);
        if (r_long) atomicAdd(&sh[2], r_long);
        if (n_short) atomicAdd(&sh[3], n_short);
        if (n_med) atomicAdd(&sh[4], n_med);
        if (n_long) atomicAdd(&sh[5], n_long);
    }
    __syncthreads();
    if (threadIdx.x < 6) spread_add(pc, K_ROWS_SHORT + (int)threadIdx.x, sh[threadIdx.x]);
    if (only) {                                       // the fused call
        __shared__ unsigned int most[3];
        if (threadIdx.x < 3) most[threadIdx.x] = 0;
        __syncthreads();
        for (int o = 1; o < window / SCAN_ITEMS; o <<= 1) pieces += __shfl_xor(pieces, o, WAVE);
        pieces = wave_max_u32(pieces);
        longest = wave_max_u32(longest);
        const unsigned int alike = (unsigned int)__popcll(__ballot(r_alike != 0));
        if (lane_id() == 0) {
            atomicMax(&most[0], longest);
            atomicMax(&most[1], pieces);
            atomicAdd(&most[2], alike);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const int slot = blockIdx.x & (SPREAD - 1);
            atomicMax(&pc->k[K_LONGEST][slot], (unsigned long long)most[0]);
            if (most[1]) atomicMax(&pc->k[K_WINDOW][slot], (unsigned long long)most[1]);
            spread_add(pc, K_ROWS_ALIKE, most[2]);
        }
    }
    // entries of this block's short rows, for the entry list (k_short_list_write)
    if (short_sums && threadIdx.x == 0) short_sums[blockIdx.x] = (unsigned int)sh[3];
    // and its rows of more than one item, for the list of the long rows (k_long_rows)
    if (long_sums && threadIdx.x == 0) long_sums[blockIdx.x] = (unsigned int)sh[2];
}

// pass 2: exclusive scan of the block sums (one workgroup; in == out is allowed), total -> *total_out
static __global__ __launch_bounds__(SCAN_BLOCK) void k_scan_block_sums(const unsigned int *in, unsigned int *out, int n,
                                                                unsigned long long *__restrict__ total_out) {
    unsigned int carry = 0;
    for (int base = 0; base < n; base += SCAN_BLOCK) {
        const int i = base + (int)threadIdx.x;
        const unsigned int v = i < n ? in[i] : 0u;
        unsigned int total;
        const unsigned int ex = block_exclusive_scan(v, &total);
        if (i < n) out[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) *total_out = carry;
}

constexpr int SCAN_SMALL_ITEMS = 8;                // words per thread and step of a short scan
constexpr int SCAN_SMALL_MAX = 16384;

// Several short scans in one launch: workgroup j takes job j (in == out is allowed: a thread
// writes only the positions it has read).  With a place for the totals in host memory one more workgroup reports the
// counters, and every job its total if that is one of the first SCAN_TOTALS of DevCounters.
constexpr int SCAN_JOBS_MAX = 8;
struct ScanJob {
    const unsigned int *in;
    unsigned int *out;
    unsigned long long *total;
    int n;
    int pad;
};
struct ScanJobs { ScanJob job[SCAN_JOBS_MAX]; };
// The workgroup after the last job: the counters, but for the totals of this launch's own jobs, which those write.
__device__ __forceinline__ void report_totals(const ScanJobs &jobs, int n_jobs, const DevCounters *pc,
                                              DevTotals *__restrict__ totals) {
    constexpr int WAVES = SCAN_BLOCK / WAVE, EACH = (K_KINDS + WAVES - 1) / WAVES;
    const int lane = lane_id(), wv = wave_in_block(), tid = (int)threadIdx.x;
    unsigned long long v[EACH];
#pragma unroll
    for (int q = 0; q < EACH; ++q) v[q] = wv + q * WAVES < K_KINDS ? pc->k[wv + q * WAVES][lane] : 0ull;
    const unsigned int longest = wave_max_u32(pc->max_len[lane]);
#pragma unroll
    for (int q = 0; q < EACH; ++q) {
        const int kind = wv + q * WAVES;
        if (kind >= K_KINDS) break;
        // (64 numbers of 24 bits stay below 2^31; what wraps around, as the slots of a difference do, comes out right)
        unsigned long long sum = (unsigned long long)wave_sum_i32((int)(v[q] & 0xFFFFFF)) +
                                 ((unsigned long long)wave_sum_i32((int)(v[q] >> 24 & 0xFFFFFF)) << 24) +
                                 ((unsigned long long)wave_sum_i32((int)(v[q] >> 48)) << 48);
        if (kind == K_LONGEST || kind == K_WINDOW) sum = wave_max_u32((unsigned int)v[q]);
        if (lane == 0) totals->k[kind] = sum;
    }
    if (tid == 0) {
        totals->bad_pattern = pc->bad_pattern;
        totals->coo_unsorted = pc->coo_unsorted;
        totals->max_len = longest;
    }
    if (tid < SCAN_TOTALS) {
        bool of_a_job = false;
        for (int j = 0; j < n_jobs; ++j) of_a_job |= jobs.job[j].total == &pc->n_items + tid;
        if (!of_a_job) (&totals->n_items)[tid] = (&pc->n_items)[tid];
    }
}

static __global__ __launch_bounds__(SCAN_BLOCK) void k_scan_jobs(ScanJobs jobs, int n_jobs, const DevCounters *pc,
                                                                 DevTotals *__restrict__ totals) {
    if ((int)blockIdx.x == n_jobs) {
        report_totals(jobs, n_jobs, pc, totals);
        return;
    }
    const ScanJob jb = jobs.job[blockIdx.x];
    // eight words per thread and step, the next step's on the way (12 500 words one by one, step after step: 15.0 us, so 6.1)
    const bool whole = ((reinterpret_cast<uintptr_t>(jb.in) | reinterpret_cast<uintptr_t>(jb.out)) & 15) == 0;
    auto load = [&](int i0, unsigned int (&v)[SCAN_SMALL_ITEMS]) {
        if (whole && i0 + SCAN_SMALL_ITEMS <= jb.n) {
#pragma unroll
            for (int q = 0; q < SCAN_SMALL_ITEMS; q += 4) {
                const uint4 w = *reinterpret_cast<const uint4 *>(jb.in + i0 + q);
                v[q] = w.x; v[q + 1] = w.y; v[q + 2] = w.z; v[q + 3] = w.w;
            }
        } else {
#pragma unroll
            for (int q = 0; q < SCAN_SMALL_ITEMS; ++q) v[q] = i0 + q < jb.n ? jb.in[i0 + q] : 0u;
        }
    };
    unsigned int carry = 0, v[SCAN_SMALL_ITEMS], next[SCAN_SMALL_ITEMS];
    load((int)threadIdx.x * SCAN_SMALL_ITEMS, v);
    for (int base = 0; base < jb.n; base += SCAN_BLOCK * SCAN_SMALL_ITEMS) {
        const int i0 = base + (int)threadIdx.x * SCAN_SMALL_ITEMS;
        load(i0 + SCAN_BLOCK * SCAN_SMALL_ITEMS, next);
        unsigned int mine = 0;
#pragma unroll
        for (int q = 0; q < SCAN_SMALL_ITEMS; ++q) mine += v[q];
        unsigned int total;
        unsigned int at = carry + block_exclusive_scan(mine, &total);
        unsigned int o[SCAN_SMALL_ITEMS];
#pragma unroll
        for (int q = 0; q < SCAN_SMALL_ITEMS; ++q) {
            o[q] = at;
            at += v[q];
        }
        if (whole && i0 + SCAN_SMALL_ITEMS <= jb.n) {
#pragma unroll
            for (int q = 0; q < SCAN_SMALL_ITEMS; q += 4)
                *reinterpret_cast<uint4 *>(jb.out + i0 + q) = make_uint4(o[q], o[q + 1], o[q + 2], o[q + 3]);
        } else {
#pragma unroll
            for (int q = 0; q < SCAN_SMALL_ITEMS; ++q)
                if (i0 + q < jb.n) jb.out[i0 + q] = o[q];
        }
        carry += total;
#pragma unroll
        for (int q = 0; q < SCAN_SMALL_ITEMS; ++q) v[q] = next[q];
    }
    if (threadIdx.x == 0) {
        *jb.total = carry;
        const int slot = scan_total_slot(jb.total, &pc->n_items, SCAN_TOTALS);
        if (totals && slot >= 0) (&totals->n_items)[slot] = carry;
    }
}

// The entry list of the short rows: {position, row} of every stored entry of the rows that
// have fewer than ts entries and no owner, in storage order.  The kernels take it 64 entries
// per wavefront, whatever the lengths of the rows (block_offsets: exclusive scan of the
// short_sums of k_classify_count).  SHORT_LIST_SPLIT workgroups share a block of the row scan, each writes the entries
// of its part of the rows, two threads per row (one workgroup, a thread per four rows: 9.2 us for 27 000 rows of 12
// entries, 30 workgroups on 256 CUs; split 4.9).
constexpr int SHORT_LIST_SPLIT = 8, SHORT_LIST_ROWS = SCAN_TILE / SHORT_LIST_SPLIT;
static __global__ __launch_bounds__(SCAN_BLOCK) void k_short_list_write(const int32_t *__restrict__ rowptr,
                                                                 const unsigned char *__restrict__ owner, int M,
                                                                 int ts, const unsigned int *__restrict__ block_offsets,
                                                                 int2 *__restrict__ list) {
    static_assert(2 * SHORT_LIST_ROWS == SCAN_BLOCK && SHORT_LIST_ROWS % SCAN_ITEMS == 0, "two threads per row of the part");
    __shared__ unsigned int at_of[SHORT_LIST_ROWS], len_of[SHORT_LIST_ROWS];
    const int64_t block = blockIdx.x / SHORT_LIST_SPLIT;
    const int part = (int)(blockIdx.x % SHORT_LIST_SPLIT), tid = (int)threadIdx.x;
    unsigned int len[SCAN_ITEMS], mine = 0;
    row_lengths(rowptr, owner, block * SCAN_TILE + (int64_t)tid * SCAN_ITEMS, M, len);
#pragma unroll
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        if (len[q] >= (unsigned int)ts) len[q] = 0;
        mine += len[q];
    }
    unsigned int total;
    unsigned int at = block_offsets[block] + block_exclusive_scan(mine, &total);
    const int first = tid * SCAN_ITEMS - part * SHORT_LIST_ROWS;            // row of the part
    if (first >= 0 && first < SHORT_LIST_ROWS) {
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS; ++q) {
            at_of[first + q] = at;
            len_of[first + q] = len[q];
            at += len[q];
        }
    }
    __syncthreads();
    const int r = tid >> 1;
    const unsigned int n = len_of[r], to = at_of[r];
    if (n == 0) return;                                                     // (rows past the last one have none)
    const int32_t row = (int32_t)(block * SCAN_TILE + part * SHORT_LIST_ROWS + r);
    const int32_t rs = rowptr[row];
    for (unsigned int e = tid & 1; e < n; e += 2) list[to + e] = make_int2(rs + (int32_t)e, row);
}

// pass 3: write the items
static __global__ __launch_bounds__(SCAN_BLOCK) void k_classify_write(const int32_t *__restrict__ rowptr,
                                                               const unsigned char *__restrict__ owner, int M,
                                                               int ts, int seg,
                                                               const unsigned int *__restrict__ block_offsets,
                                                               RowItem *__restrict__ items, int only) {
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    unsigned int cnt[SCAN_ITEMS], lens[SCAN_ITEMS], mine = 0;
    row_lengths(rowptr, owner, base, M, lens, only);
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        cnt[q] = row_item_count(lens[q], ts, seg);
        mine += cnt[q];
    }
    unsigned int total;
    unsigned int at = block_offsets[blockIdx.x] + block_exclusive_scan(mine, &total);
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        if (cnt[q] == 0) continue;
        const int32_t row = (int32_t)(base + q);
        const int32_t s = rowptr[row], e = rowptr[row + 1];
        for (unsigned int k = 0; k < cnt[q]; ++k) {
            const int32_t a = s + (int32_t)k * seg;
            const int32_t b = e - a > seg ? a + seg : e;
            items[at++] = RowItem{row, a, b, 0};
        }
    }
}

// Places for the partial output rows of the fused call's pieces (kernels_fused.h): the pieces of a row that was cut
// into several items lie next to each other, in order; which row comes first does not matter.  One thread per item,
// the first item of a cut row writes the places of them all (they follow it in the list); one atomic per wavefront
// that holds such an item.  cut_rows (if given): the cut rows, in any order.
static __global__ __launch_bounds__(256) void k_piece_places(const int32_t *__restrict__ rowptr, RowItem *__restrict__ items,
                                                             int64_t n_items, int32_t *__restrict__ cut_rows, DevCounters *pc) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned int n = 0;
    int row = 0;
    if (w < n_items) {
        row = items[w].row;
        const int start = items[w].start, end = items[w].end;
        const int rs = rowptr[row], re = rowptr[row + 1];
        if (start == rs && end != re) n = ((unsigned int)(re - rs) + (unsigned int)(end - start) - 1u) / (unsigned int)(end - start);
    }
    if (!__ballot(n != 0)) return;
    const int lane = lane_id();
    const unsigned int incl = (unsigned int)wave_inclusive_sum((int)n);
    unsigned int first = 0;
    if (lane == WAVE - 1) first = (unsigned int)atomicAdd(&pc->fused_pieces, (unsigned long long)incl);
    first = __shfl(first, WAVE - 1, WAVE) + incl - n;
    for (unsigned int k = 0; k < n; ++k) items[w + k].extra = (int32_t)(first + k);
    if (!cut_rows) return;
    const unsigned long long cut = __ballot(n != 0);
    unsigned int at = 0;
    if (lane == 0) at = (unsigned int)atomicAdd(&pc->fused_cut, (unsigned long long)__popcll(cut));
    at = __shfl(at, 0, WAVE) + (unsigned int)__popcll(cut & ((1ull << lane) - 1ull));
    if (n != 0) cut_rows[at] = row;
}

// Items per taken panel for the fused call, in place of those of the SDDMM (fused_panel_columns).
static __global__ __launch_bounds__(256) void k_fused_panel_counts(const int32_t *__restrict__ rowptr, int64_t n_panels, int halves_from,
                                                                   unsigned int *__restrict__ counts) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_panels || counts[p] == 0) return;
    const int len = rowptr[p * 8 + 1] - rowptr[p * 8], columns = fused_panel_columns(len, halves_from);
    counts[p] = (unsigned int)((len + columns - 1) / columns);
}

// items of the taken panels: {first row, [start,end) inside the shared list}; pseg 0: of the fused call
static __global__ __launch_bounds__(256) void k_panel_items(const int32_t *__restrict__ rowptr, int64_t n_panels, int pseg, int halves_from,
                                                     const unsigned int *__restrict__ counts,
                                                     const unsigned int *__restrict__ offsets,
                                                     RowItem *__restrict__ items) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_panels) return;
    const unsigned int n = counts[p];
    if (n == 0) return;
    const int32_t row0 = (int32_t)(p * 8);
    const int32_t rs0 = rowptr[row0];
    const int32_t len = rowptr[row0 + 1] - rs0;
    const int columns = pseg ? pseg : fused_panel_columns(len, halves_from);
    unsigned int at = offsets[p];
    for (unsigned int k = 0; k < n; ++k) {
        const int32_t a = (int32_t)k * columns;
        const int32_t b = a + columns < len ? a + columns : len;
        // pad carries the CSR position of the panel's first row: the 8 rows have the same
        // length and follow each other, so row r starts at pad + r*len and a kernel can
        // start reading the column list without first waiting for a row pointer
        items[at++] = RowItem{row0, a, b, rs0};
    }
}

// ---------------------------------------------------------------------------
// Column blocks for the long rows of a flat matrix (kernels_flat.h, k_flat_blocks).
//
// Rows of several work items, in row order (block_offsets: exclusive scan of the long_sums of
// k_classify_count, so a row is long here exactly when it is there: rows below `ts` never are).
static __global__ __launch_bounds__(SCAN_BLOCK) void k_long_rows(const int32_t *__restrict__ rowptr, int M, int ts, int seg,
                                                                 const unsigned int *__restrict__ block_offsets,
                                                                 int32_t *__restrict__ long_rows) {
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    unsigned int mine = 0, is_long = 0, lens[SCAN_ITEMS];
    row_lengths(rowptr, nullptr, base, M, lens);
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        const bool l = row_item_count(lens[q], ts, seg) > 1;
        is_long |= (l ? 1u : 0u) << q;
        mine += l ? 1u : 0u;
    }
    unsigned int total;
    unsigned int at = block_offsets[blockIdx.x] + block_exclusive_scan(mine, &total);
    for (int q = 0; q < SCAN_ITEMS; ++q)
        if ((is_long >> q) & 1u) long_rows[at++] = (int32_t)(base + q);
}

// `most` lanes per long row: lane b finds where the row's columns of block b start (columns ascend inside a
// row: its entries of a block are consecutive; in a row that is not sorted the cuts fall anywhere, every
// entry still lands in exactly one segment).  Segment (b, i): block b of long row i, block-major; a row of fewer blocks
// has its segments at the first of the blocks that each of them covers.
static __global__ __launch_bounds__(256) void k_long_segments(const int32_t *__restrict__ rowptr,
                                                              const int32_t *__restrict__ col, int N,
                                                              const int32_t *__restrict__ long_rows, int n_long, int piece,
                                                              int least, int most,
                                                              int32_t *__restrict__ seg_start,
                                                              unsigned int *__restrict__ seg_items) {
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int i = (int)(slot / most), b = (int)(slot % most);
    const bool on = i < n_long;
    int lo = 0, end = 0, every = most;
    if (on) {
        const int row = long_rows[i];
        lo = rowptr[row];
        end = rowptr[row + 1];
        every = most / row_blocks(end - lo, least, most);
        const int first = (int)(((int64_t)N * b + most - 1) / most);     // (of block b, as in k_order_keys)
        int hi = end;
        if (b % every != 0 || b == 0) hi = lo;
        while (lo < hi) {
            const int mid = lo + ((hi - lo) >> 1);
            if (col[mid] < first) lo = mid + 1; else hi = mid;
        }
    }
    // the cuts of a row must ascend whatever its columns do: running maximum over its lanes
    for (int o = 1; o < most; o <<= 1) {
        const int up = __shfl_up(lo, o, WAVE);
        if (b >= o) lo = up > lo ? up : lo;
    }
    const int lane = lane_id(), ahead = (every - b % every) % every;         // to the next block that starts a segment
    const int after = __shfl(lo, (lane + ahead) & (WAVE - 1), WAVE), next_after = __shfl(lo, (lane + every) & (WAVE - 1), WAVE);
    if (!on) return;
    const int start = b + ahead < most ? after : end;
    const int next = b % every != 0 ? start : b + every < most ? next_after : end;
    seg_start[(int64_t)b * n_long + i] = start;
    seg_items[(int64_t)b * n_long + i] = (unsigned int)((next - start + piece - 1) / piece);
}

// the entries between long rows: gap i lies before long row i, the last one after all of them
static __global__ __launch_bounds__(256) void k_long_gaps(const int32_t *__restrict__ rowptr,
                                                          const int32_t *__restrict__ long_rows, int n_long, int nnz,
                                                          int piece, int32_t *__restrict__ gap_start,
                                                          unsigned int *__restrict__ gap_items) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i > n_long) return;
    const int start = i == 0 ? 0 : rowptr[long_rows[i - 1] + 1];
    const int end = i == n_long ? nnz : rowptr[long_rows[i]];
    gap_start[i] = start;
    gap_items[i] = (unsigned int)((end - start + piece - 1) / piece);
}

// One thread per work item: its range by bisection over the exclusive scan of the ranges' item counts.
// Ranges are the segments of the long rows or the gaps between those rows (items of no row).
static __global__ __launch_bounds__(256) void k_range_items(const int32_t *__restrict__ rowptr,
                                                            const int32_t *__restrict__ long_rows, int n_long, int nnz,
                                                            int gaps, int piece, const int32_t *__restrict__ start,
                                                            const unsigned int *__restrict__ offsets, int n_ranges,
                                                            const unsigned long long *__restrict__ total,
                                                            RowItem *__restrict__ items) {
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= (int64_t)*total) return;
    int lo = 0, hi = n_ranges;                              // last range whose offset does not exceed w
    while (hi - lo > 1) {
        const int mid = lo + ((hi - lo) >> 1);
        if ((int64_t)offsets[mid] <= w) lo = mid; else hi = mid;
    }
    int row = -1, end;
    if (gaps) {
        end = lo == n_long ? nnz : rowptr[long_rows[lo]];
    } else {
        row = long_rows[lo % n_long];
        end = lo + n_long < n_ranges ? start[lo + n_long] : rowptr[row + 1];
    }
    const int a = start[lo] + (int)(w - (int64_t)offsets[lo]) * piece;
    items[w] = RowItem{row, a, a + piece < end ? a + piece : end, 0};
}

// ---------------------------------------------------------------------------
// Entries in no order (a COO edge list): sorted by row, and by column block inside a row.
template <class Key>
static __global__ __launch_bounds__(256) void k_order_keys(const int32_t *__restrict__ row, const int32_t *__restrict__ col,
                                                           int64_t nnz, int N, Key *__restrict__ keys,
                                                           int32_t *__restrict__ at) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nnz) return;
    keys[n] = (Key)row[n] * COL_BLOCKS_ORDER + (Key)((int64_t)col[n] * COL_BLOCKS_ORDER / N);
    at[n] = (int32_t)n;
}
// (32-bit keys lie in row_out, `at` lies in col_out: a thread reads its element of either before it writes there)
template <class Key>
static __global__ __launch_bounds__(256) void k_order_entries(const Key *keys, const int32_t *at,
                                                              const int32_t *__restrict__ col, int64_t nnz,
                                                              int32_t *row_out, int32_t *col_out,
                                                              int32_t *__restrict__ place) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nnz) return;
    const int32_t q = at[n], row = (int32_t)(keys[n] / COL_BLOCKS_ORDER);
    row_out[n] = row;
    col_out[n] = col[q];
    place[q] = (int32_t)n;
}

}  // namespace sddmm
