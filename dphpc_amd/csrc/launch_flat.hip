// Launches of the flat gather kernel and of its variant in slices of K.
#include "context.h"
#include "kernels_flat.h"

void launch_flat(sddmm_ctx *c) {
    const Shape s = shape_of(c);
    const int64_t chunks = (c->nnz + WAVE - 1) / WAVE;
    const int cpw = (int)std::min<int64_t>(8, std::max<int64_t>(1, chunks / (WAVES_PER_BLOCK * 4096)));
    const int64_t waves = (chunks + cpw - 1) / cpw;
    const int64_t nblocks = (waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        SDDMM_LAUNCH(c, (k_flat<LT>), xcd_grid(nblocks), BLOCK, nblocks, c->nnz, cpw, s.len, c->d_rowidx, c->d_col,
                     (const void *)c->dA, (const void *)c->dB, c->d_sval, c->dP);
    });
}

namespace {

// workgroups of a launch over at most `segments` and `gaps` work items: an eighth of either kind per XCD
int64_t blocks_grid(int64_t segments, int64_t gaps, int waves) {
    auto eighth = [waves](int64_t items) {                 // workgroups per XCD, rounded up twice
        const int64_t blocks = (items + waves - 1) / waves;
        return (blocks + NUM_XCD - 1) / NUM_XCD;
    };
    return NUM_XCD * (eighth(segments) + eighth(gaps));
}

}  // namespace

// the most work items there can be, from the counts of the row classes
void block_items_max(const sddmm_ctx *c, bool cut_long_rows, int64_t *segments, int64_t *gaps) {
    const int64_t n_long = cut_long_rows ? (int64_t)c->pc.rows_long : 0, nnz_long = cut_long_rows ? (int64_t)c->pc.nnz_long : 0;
    *segments = row_block_segments(n_long, nnz_long, c->seg, c->use_order, (int)c->pc.max_len);
    *gaps = (c->nnz - nnz_long) / WAVE + n_long + 1;
}

// 0: no kernel for this row layout
int launch_flat_blocks(sddmm_ctx *c) {
    const Shape s = shape_of(c);
    const int waves = block_item_waves(s.UPL);
    const int64_t grid = blocks_grid(c->block_segments_max, c->block_gaps_max, waves);
    int launches = 0;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        if constexpr (!LT::LONG) {
            auto launch = [&](auto kernel, float *out) {
                SDDMM_LAUNCH(c, kernel, grid, waves * WAVE, (const unsigned long long *)c->d_pc->block_items,
                             (const RowItem *)c->d_block_segments, (const RowItem *)c->d_block_gaps, entry_cols(c),
                             (const float *)c->d_sval, (const void *)c->dA, (const void *)c->dB, s.len, entry_rows(c), out);
                ++launches;
            };
            if (c->use_order) launch(k_flat_blocks<LT, false>, c->d_order_dots);
            else launch(k_flat_blocks<LT, true>, c->dP);
        }
    });
    return launches;
}

void launch_unsort(sddmm_ctx *c) {
    SDDMM_LAUNCH(c, k_unsort, (c->nnz + 4 * BLOCK - 1) / (4 * BLOCK), BLOCK, (const float *)c->d_order_dots,
                 (const int32_t *)c->d_order_place, (const float *)c->d_sval, c->dP, c->nnz);
}

// Measured on power-law graphs (rows of Zipf lengths, half to two thirds of the entries in rows of more than 256) of
// 20 000 to 2.6 M vertices, K = 16 .. 250: 1.1 .. 1.4 times k_flat from 12 MB of B on; where B nearly fits the L2s
// (60 000 vertices, 128-byte rows, 7.7 MB: 0.81 times) or the launch is short (500 k entries over 25 MB: 0.97) the
// extra wavefronts cost more than the lines they save.
bool blocks_pay(const sddmm_ctx *c) {
    const int mode = env_int("SDDMM_COLUMN_BLOCKS", -1);            // -1: decide here, 0: never, 1: wherever there are long rows
    if (shape_of(c).LPN == 0 || c->pc.rows_long == 0) return false;
    int64_t segments, gaps;                                         // (a launch takes fewer than 2^32 threads)
    block_items_max(c, true, &segments, &gaps);
    // (sixteen blocks a row, whatever its length: what a launch refuses does not hang on the lengths)
    segments = std::max(segments, (int64_t)(c->pc.nnz_long / c->seg + c->pc.rows_long * 16));
    const int waves = block_item_waves(shape_of(c).UPL);
    if (blocks_grid(segments, gaps, waves) * waves * WAVE >= (int64_t)1 << 32) return false;
    if (mode >= 0) return mode != 0;
    const double b_bytes = (double)c->N * (double)c->K * (double)elem_size(c->dtype);
    return b_bytes >= 12.0 * (1 << 20) && c->nnz >= (1 << 20) && (double)c->pc.nnz_long >= 0.25 * (double)c->nnz;
}

// Entries in no order, sorted by the plan (k_unsort).  Measured on shuffled uniform, power-law, banded and tiled
// matrices of 0.1 .. 6.5 M entries, K = 32 .. 400: 1.03 .. 2.1 times the plain kernel from 192-byte rows, 1.5 MB of A
// and 150 MB of gathered B rows on, up to 3.5 times where the sorted entries can go in slices of K.  Below:
// 128-byte rows 0.5 .. 1.2 times (k_unsort costs what the A rows save), 0.9 MB of A 0.87 .. 0.94 (A is found in the
// L2s in any order), 100 MB gathered 0.7 .. 1.05.  Rows of one entry have nothing to share (0.9 .. 1.15).  Entries
// that arrive grouped, by column (0.65 .. 0.95 times) or in runs of sorted rows (0.8 .. 1.2), keep their order: most
// of them share a row or a column with the entry before.  The plan takes 0.2 ms for 1.2 M entries.
bool order_pays(const sddmm_ctx *c) {
    const int mode = env_int("SDDMM_ORDER", -1);                    // -1: decide here, 0: never, 1: wherever a kernel can
    if (shape_of(c).LPN == 0 && !slices_pay(c, 1.0)) return false;  // (no kernel takes the order)
    if (mode >= 0) return mode != 0;
    const int64_t row_bytes = (int64_t)c->K * (int64_t)elem_size(c->dtype);
    return 2 * c->coo_jumps >= c->nnz && c->nnz >= 2 * (int64_t)c->sM && row_bytes >= 192 &&
           (int64_t)c->sM * row_bytes >= 1500 * 1000 && c->nnz * row_bytes >= (int64_t)150 * 1000 * 1000;
}

namespace {

constexpr int64_t SLICE_WORKSPACE = (int64_t)1 << 26;      // floats: the partial products stay in the last-level cache

// slices (lines) that the longest row touches: rows start anywhere in a line that B's address and the
// row length lead to
int slices_of(uint64_t b_address, int64_t row_bytes) {
    int64_t most = 0;
    for (int i = 0; i < 32; ++i) most = std::max(most, (int64_t)((b_address + (uint64_t)i * (uint64_t)row_bytes) % SLICE_BYTES));
    return (int)((row_bytes + most + SLICE_BYTES - 1) / SLICE_BYTES);
}

template <class U, bool MISALIGNED, bool UNALIGNED, bool WIDE>
int launch_slices_t(sddmm_ctx *c, int slices) {
    const int row_bytes = c->K * (int)elem_size(c->dtype);
    const int64_t most = c->part_floats / slices / SLICE_ENTRIES * SLICE_ENTRIES;      // entries the workspace holds
    int launches = 0;
    for (int64_t e0 = 0; e0 < c->nnz; e0 += most) {
        const int64_t n = std::min(most, c->nnz - e0);
        const int64_t stride = (n + WAVE - 1) / WAVE * WAVE;
        const int64_t waves = (n + SLICE_ENTRIES - 1) / SLICE_ENTRIES;
        const int64_t per_slice = (waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK, nblocks = per_slice * slices;
        SDDMM_LAUNCH(c, (k_slice_dots<U, MISALIGNED, UNALIGNED, WIDE>), xcd_grid(nblocks), BLOCK, nblocks, per_slice, n,
                     entry_rows(c) + e0, entry_cols(c) + e0, (const void *)c->dA, (const void *)c->dB, row_bytes, c->d_part,
                     stride);
        SDDMM_LAUNCH(c, k_slice_sum, (n + 4 * BLOCK - 1) / (4 * BLOCK), BLOCK, (const float *)c->d_part, slices, stride,
                     (const float *)(c->use_order ? nullptr : c->d_sval + e0),
                     c->use_order ? c->d_order_dots + e0 : c->dP + e0, n);
        launches += 2;
    }
    return launches;
}

template <class U>
int launch_slices_u(sddmm_ctx *c) {
    const int64_t row_bytes = (int64_t)c->K * (int64_t)elem_size(c->dtype);
    const int slices = slices_of((uint64_t)(uintptr_t)c->dB, row_bytes);
    const bool wide = (size_t)std::max(c->M, c->N) * (size_t)row_bytes >= ((size_t)1 << 32);
    if constexpr (U::DT == DT_F32) {
        if (row_bytes % 16)
            return wide ? launch_slices_t<U, true, true, true>(c, slices) : launch_slices_t<U, true, true, false>(c, slices);
    }
    if (wide) return launch_slices_t<U, true, false, true>(c, slices);
    if (row_bytes % SLICE_BYTES || (uintptr_t)c->dB % SLICE_BYTES) return launch_slices_t<U, true, false, false>(c, slices);
    return launch_slices_t<U, false, false, false>(c, slices);
}

}  // namespace

// Measured on uniform random matrices, against the better of the other kernels; in a loop / after a flush of the caches.
// What slices gain is that a line of B is found in the L2 again, so it follows the size of B, the entries per column,
// and the length of a row, which decides how well the other kernels do:
//   up to 1 KB   entries per column:    4            8            12           24           48
//     B of  9 MB (400 B rows)                   0.88 / 0.91   0.96 / 0.99   1.09 / 1.08   1.19 / 1.14
//     B of 11 MB (600 B)           0.73 / 0.79  0.85 / 0.95   0.89 / 0.96   1.11 / 1.15   1.17 / 1.22   (first column: 6)
//     B of 15 MB (400 B)           0.91 / 0.92  0.98 / 1.00   1.04 / 1.07   1.08 / 1.10   1.10 / 1.11
//     B of 20 MB (1 KB)            1.11 / 0.87  1.27 / 0.94   1.39 / 1.05   1.65 / 1.25   1.70 / 1.32
//     B of 39 MB (1 KB)            1.17 / 0.88  1.33 / 1.03   1.41 / 1.15   1.47 / 1.24   1.43 / 1.30
//   (0.5 .. 2 per column: 0.5 .. 1.1 / 0.75 .. 1.2); hence 12 entries per column, 20 below 12 MB of B.
//   1.25 .. 2 KB: 1.0 .. 2.3 / 1.0 .. 2.4 at 0.5 .. 48 entries per column; lowest 0.93 / 0.98 (1 per column, 122 MB of B).
//   beyond 2 KB (no register layout): 1.4 times at the least.
// From 32 entries per row on, the other kernel is the row split, which reads an A row once:
//     entries per column:               2            6            12           24           48
//     B of  9 MB (1 KB rows)        0.53 / 0.68  0.80 / 0.70  0.88 / 0.73  1.05 / 0.83  1.12 / 0.95
//     B of 11 MB (600 B)            0.46 / 0.69  0.70 / 0.68  0.79 / 0.78  0.95 / 0.92  1.03 / 1.02
//     B of 15 MB (400 B)            0.65 / 0.75  1.00 / 0.92  1.14 / 1.06  1.26 / 1.20  1.32 / 1.26
//     B of 20 MB (1 KB)             0.74 / 0.63  1.05 / 0.73  1.22 / 0.93  1.46 / 1.15  1.67 / 1.32
//     B of 24 MB (1.25 KB)          1.11 / 0.93  1.18 / 0.88  1.55 / 1.15  1.84 / 1.40  2.07 / 1.60
//     B of 73 MB (1.9 KB)           1.03 / 0.83  1.46 / 1.19  1.68 / 1.43  1.85 / 1.65  1.85 / 1.77
// hence 48 below 12 MB of B, 12 from there on, 8 with rows beyond 1 KB.
// B has to exceed the L2s (0.6 .. 1.1 times below 5 MB) and one slice of it to come near to fitting (N = 65 536 is 8 MB:
// 1.05 .. 1.25; 100 000: 1.0); rows of 256 bytes 0.8 .. 1.1.  Rows of fewer than 12 entries have their A rows gathered per
// entry, which pays while the slice fits (6 entries per row: 40 000 columns 0.8 .. 1.1) and, up to 1 KB, with rows that are
// long and columns of many entries only (6 .. 11 per row, 24 per column: 1 KB rows 1.24 / 0.94, 600 bytes 0.98 / 1.03).
bool slices_pay(const sddmm_ctx *c, double entries_per_row) {
    const int64_t row_bytes = (int64_t)c->K * (int64_t)elem_size(c->dtype);
    const int mode = env_int("SDDMM_SLICES", -1);                   // -1: decide here, 0: never, 1: wherever the kernel can
    if (mode >= 0) return mode != 0 && row_bytes > SLICE_BYTES && row_bytes < (1 << 30);
    if (row_bytes > 2048) return row_bytes < (1 << 30);
    const int64_t MB = 1 << 20, b_bytes = (int64_t)c->N * row_bytes;
    const bool small_b = b_bytes < 12 * MB;
    if (row_bytes < 400 || b_bytes < 8 * MB || (int64_t)c->N * SLICE_BYTES > (entries_per_row >= 12.0 ? 8 * MB : 3 * MB)) return false;
    int per_column;
    if (entries_per_row >= 32.0) per_column = small_b ? 48 : row_bytes > 1024 ? 8 : 12;
    else if (row_bytes > 1024) return true;
    else if (entries_per_row >= 12.0) per_column = small_b ? 20 : 12;
    else if (row_bytes >= 1000) per_column = 24;
    else return false;
    return c->nnz >= per_column * (int64_t)c->sN;
}

// The partial products of all entries where they fit SLICE_WORKSPACE, of a range of entries at a time otherwise.
int64_t slice_workspace_floats(const sddmm_ctx *c) {
    const int64_t slices = ((int64_t)c->K * (int64_t)elem_size(c->dtype) + SLICE_BYTES - 1) / SLICE_BYTES + 1;   // whatever B's address
    const int64_t all = (c->nnz + SLICE_ENTRIES - 1) / SLICE_ENTRIES * SLICE_ENTRIES * slices;
    const int64_t cap = std::max((int64_t)env_int("SDDMM_SLICE_WORKSPACE", (int)SLICE_WORKSPACE), SLICE_ENTRIES * slices);
    return std::min(all, cap);
}

int launch_flat_sliced(sddmm_ctx *c) {
    if (c->dtype == SDDMM_BF16) return launch_slices_u<UnitBF16x8>(c);
    if (c->dtype == SDDMM_F16) return launch_slices_u<UnitF16x8>(c);
    return launch_slices_u<UnitF32x4>(c);
}

hipError_t load_flat() { return load_code(reinterpret_cast<const void *>(k_unsort)); }
