// Rules of the plan that are arithmetic alone: no HIP, so that a host program can check them (tests/host/test_plan_rules.cpp).
// constexpr functions run on the device as well.
#pragma once
#include <cstdint>

namespace sddmm {

// ---- reports of the counters (k_scan_jobs) -----------------------------------------------------
// Place of a scan's total among the n that are reported, counted from the first one; -1: not one of them.
constexpr int scan_total_slot(const unsigned long long *total, const unsigned long long *first, int n) {
    return total >= first && total < first + n ? (int)(total - first) : -1;
}

// ---- column blocks of a long row (kernels_flat.h) ---------------------------------------------
// A power of two, `least` to `most`, such that the segments hold COL_BLOCK_ENTRIES entries or more on average (beyond `least`
// blocks).  More blocks find more lines of B in an XCD's L2, short segments leave lanes idle and are work items more.  16 blocks
// for every row / 8 .. 64 with 32, 64, 96 entries, all with the exact grid (launch_flat_blocks): graph of 2.6 M rows K = 32
// 521 us / 524, 515, 513; 1.5 M rows K = 64 bf16 229 / 230, 225, 223; 800 000 rows K = 64 253 / 251, 249, 249; 200 000 rows
// K = 32 27.7 / 28.2, 27.3, 26.9, K = 100 116.4 / 114.6, 114.8, 115.5, K = 256 244 / 238, 241, 243.  From 4 blocks on: 532,
// 226, 259, 27.1, 118, 265.
// Entries that came in no order were sorted by row and by 16 blocks, and keep them, whatever the row: 8 and 16 / 16, with the
// unsorting, 400 000 rows K = 128 310.7 / 304.4 us, K = 200 550 / 540; 1 M rows K = 100 816 / 799, K = 75 703 / 688; 100 000 rows
// K = 200 108.6 / 106.6, K = 75 50.0 / 50.6, with new inputs in turn 53.5 / 53.2 (the same run twice differs by 2 %); up to 64
// floats a row 1 % the other way.
constexpr int COL_BLOCKS_MIN = 8, COL_BLOCKS_MAX = 64, COL_BLOCK_ENTRIES = 64;
constexpr int COL_BLOCKS_ORDER = 16;           // that the sort of COO entries knows
constexpr int row_blocks(int len, int least, int most) {
    int n = least;
    while (n < most && len >= 2 * n * COL_BLOCK_ENTRIES) n *= 2;
    return n;
}
constexpr int row_blocks_least(bool sorted_order) { return sorted_order ? COL_BLOCKS_ORDER : COL_BLOCKS_MIN; }
constexpr int row_blocks_most(bool sorted_order, int longest_row) {
    return row_blocks(longest_row, row_blocks_least(sorted_order), sorted_order ? COL_BLOCKS_ORDER : COL_BLOCKS_MAX);
}
// the most segments of pieces of `piece` entries that n_long rows of nnz_long entries can have
constexpr int64_t row_block_segments(int64_t n_long, int64_t nnz_long, int piece, bool sorted_order, int longest_row) {
    const int64_t most = n_long * row_blocks_most(sorted_order, longest_row);
    const int64_t by_length = n_long * row_blocks_least(sorted_order) + nnz_long / COL_BLOCK_ENTRIES;
    return nnz_long / piece + (most < by_length ? most : by_length);
}

// ---- rows of any length on the tile and panel kernels --------------------------------------------
// Rows of 64 * {1, 2, 4, 8, 16} bytes are always looked at.  For the others the look costs a plan 8 us (1 000 rows) to 40 (4 M
// entries), where it finds gathered strips 60, and the launch gains what `steps` 64-byte steps times the entries are worth to it.  A
// caller who plans a pattern once has the cost back soon in any case; a caller with a new pattern for every launch never has
// unless one launch gains it.  The lines lie where three to five launches of dense tiles do; of banded blocks, which gain less, it
// takes eight and more there.

// Share of the entries that lie in the same 16 columns as the one before them (a sample, from the check of the columns): 1.0
// in banded blocks and dense tiles, 0.7 where near-dense rows hold most of the entries, 0.02 .. 0.06 in graphs and uniform
// rows, 0.5 where those have few columns.
constexpr double STRUCTURED_NEAR = 0.85, GATHERED_NEAR = 0.6;

// Entries from which structured patterns of `steps` steps are looked at.  Launch without / with, us, and set, plan and launch
// without / with: dense tiles of 1.2 M entries K = 9 6.6 / 6.2, 83 / 105, K = 33 15.9 / 6.1, 92 / 105, K = 75 21.4 / 8.7, 98 / 108,
// K = 100 27.8 / 8.7, 103 / 109; 2.4 M K = 15 11.1 / 7.0, 89 / 118; 4 M K = 15 17.2 / 8.8, 96 / 129, K = 21 23.3 / 10.7, 103 /
// 131, K = 33 43.9 / 13.5, 123 / 134; 0.4 M K = 33 8.9 / 4.3, 83 / 95, K = 75 10.9 / 5.3, 85 / 96; banded blocks of 0.96 M K = 21
// 7.8 / 6.1, 82 / 96, K = 51 11.7 / 8.1, 86 / 99, K = 100 19.7 / 9.7, 93 / 100; 3.8 M K = 15 16 / 10, 96 / 98, K = 40 bf16 28 / 10,
// 106 / 98, K = 75 59 / 28, 139 / 113; 14 M K = 21 69 / 29.  At the lines of two to four steps, launch without / with and how much longer
// the plan takes: tiles of 0.38 M K = 40 8.8 / 4.9, 15, K = 60 8.0 / 5.2, 16, K = 72 bf16 9.7 / 4.5, 13; 0.65 M in 548 rows K = 45
// 9.4 / 4.3; 0.83 M K = 40 bf16 8.9 / 5.2, 19; 1.2 M 11.3 / 5.5, 25, K = 24 9.4 / 6.7, 24; bands of 0.48 M K = 40 8.0 / 6.5, 11, K = 60
// 7.4 / 6.7, 10, K = 72 bf16 8.9 / 5.2, 11; 0.96 M K = 24 7.7 / 5.6, 16, K = 40 bf16 8.8 / 5.8, 16.
constexpr int64_t ragged_entries(int steps) {
    return steps <= 1 ? 3 << 20 : steps <= 2 ? 1 << 20 : steps <= 4 ? 3 << 17 : steps <= 6 ? 5 << 16 : 1 << 16;
}

// Near-dense rows among others: their gathered strips are all there is to find.  The lines lie where four to six launches get the
// look back.  Launch without / with, set, plan and launch without / with: 2 M entries K = 33 30.4 / 21.4, 111 / 169, K = 60 49.4 / 25.0, 130 /
// 172, K = 75 69.6 / 36.7, 151 / 185, K = 100 67.8 / 55.9, 151 / 202, K = 133 117 / 75.7, 203 / 223, K = 120 bf16 48.5 / 21.3, 130 / 169,
// K = 200 bf16 88.7 / 31.7, 173 / 179; 1.3 M K = 60 30.3 / 17.0, 110 / 159, K = 75 41.4 / 26.9, 122 / 169, K = 72 bf16 23.0 / 12.1, 104 / 154,
// K = 120 bf16 28.7 / 14.7, 108 / 157, K = 160 fp16 36.8 / 18.6, 118 / 161; 0.78 M K = 60 16.6 / 9.8, 96 / 147, K = 75 24.2 / 18.6, 103 / 156, K = 120
// bf16 16.7 / 9.6, 96 / 147, K = 160 fp16 20.8 / 13.5, 100 / 151, K = 200 bf16 31.5 / 15.9, 111 / 153, K = 304 bf16 46.9 / 20.7, 126 / 158.  fp32 rows of
// more than twelve steps leave a wavefront per SIMD: K = 200 108 / 155.
constexpr int ragged_gathered_steps(bool half_width) { return half_width ? 16 : 12; }
constexpr int64_t ragged_gathered_entries(int steps, bool half_width) {
    return (half_width ? 5 << 20 : steps <= 6 ? 3 << 21 : 1 << 24) / steps;
}

// Rows of more than 1 KiB, which the tile and panel kernels take 512 bytes at a time.  Launch without / with: 0.27 M entries in
// 170 panels of 200 columns K = 260 26 / 23, K = 512 26 / 34, K = 1000 63 / 68; 0.48 M in 375 panels K = 300 32 / 26, K = 452 33 /
// 36, K = 700 77 / 57, K = 1024 bf16 34 / 44; 0.67 M in 300 panels K = 452 47 / 41; 0.96 M in 750 panels K = 512 100 / 53; dense
// tiles of 0.29 M K = 260 .. 512 28 / 11 .. 14, of 0.4 M K = 452 40 / 16, K = 1024 bf16 45 / 11.  (Rows of 1.5 to 2 KiB, which the
// gather kernels hold in registers, are four launches of the panel kernel: the only ones that lose.)
constexpr int64_t long_row_entries(int64_t row_bytes) { return row_bytes <= 1536 ? 1 << 18 : 17 << 14; }

// ---- 8-row panels ---------------------------------------------------------------------------
constexpr int PANEL_COLUMNS = 512;             // columns of a panel's work item, at the most

// Columns of a panel's work item, for rows of `steps` 64-byte steps: fewer than 512 where whole panels, of `average` columns,
// would leave most of the chip's wavefronts idle (the kernel's registers hold 5 per SIMD at 128-byte rows, 4 up to 512 bytes, 2
// beyond): as many items as half of the wavefronts, but two per panel for up to three eighths of them.
// 512 / this rule: 250 panels of 240 random columns K = 32 7.2 / 4.8 us, K = 256 30.5 / 13.4; 500 K = 128 16.2 / 10.2; 1 000
// K = 32 9.8 / 7.3, K = 64 12.7 / 11.0, K = 128 17.6 / 18.8, K = 64 fp16 7.1 / 6.5; 1 000 in 8x8 blocks K = 128 16.4 / 13.9;
// 1 500 K = 128 21.5 / 18.3, random 25.5 / 25.9.  Items for all of the wavefronts, and for up to half as many panels: 1 000 of
// 240 random columns K = 128 19.9, K = 64 fp16 7.55; 2 000 of 100 K = 128 19.0 (18.4 uncut), K = 64 fp16 7.3 (6.8); 2 000 of
// 160 K = 128 22.7 (20.7).  16-bit rows beyond 128 bytes, whose items are shorter in time, only where there are very few
// panels: 1 000 of 104 columns K = 128 bf16 6.0 / 6.8.
constexpr int panel_item_of(int64_t average, int64_t pieces) {          // columns, of a panel of average length
    const int64_t columns = pieces < 2 ? PANEL_COLUMNS : (average / pieces + 63) / 64 * 64;
    return columns < 64 ? 64 : columns < PANEL_COLUMNS ? (int)columns : PANEL_COLUMNS;
}
constexpr int panel_columns(int steps, bool half_width, int64_t panels, int64_t average) {
    const int64_t wavefronts = 1024 * (steps <= 2 ? 5 : steps <= 8 ? 4 : 2);
    int64_t pieces = steps <= 8 ? wavefronts / (2 * panels) : wavefronts / panels;
    if (pieces < 2 && 8 * panels <= 3 * wavefronts) pieces = 2;
    if (half_width && steps > 2 && 8 * panels > wavefronts) pieces = 1;
    const int columns = panel_item_of(average, pieces);
    if (half_width || steps > 8) return columns;
    // fp32: shorter items, for all of the wavefronts, where the steps of 64 columns go into them without a rest (four of five at
    // the least), of 64 columns only where they do not go into the longer ones; rows beyond 128 bytes only where panels are cut
    // anyway.  Without / with: 1 333 panels of 360 columns K = 24 14.8 / 11.9 us, K = 32 12.5 / 10.8, K = 64 17.2 / 15.7, K = 100
    // 27.4 / 24.6, K = 128 24.5 / 23.0, random K = 32 12.9 / 11.5, K = 128 30.2 / 32.7; 1 700 of 360 K = 24 15.9 / 13.9; 1 700 of 160
    // K = 24 8.5 / 8.0; 2 000 of 240 K = 24 12.9 / 12.1, K = 32 11.3 / 11.1; 2 523 of 288 K = 24 17.3 / 15.7.  (After a copy of 640 MB
    // K = 32 18.3 .. 26 us, 2 .. 9 % the other way; random columns, 1 700 of 360 K = 128 31.4 / 39.2 where panels are whole.)
    const int finer = panel_item_of(average, wavefronts / panels);
    if (finer >= columns || (steps > 2 && columns == PANEL_COLUMNS)) return columns;
    const int64_t blocks = (average + 63) / 64, per_item = finer / 64, items = (blocks + per_item - 1) / per_item;
    const bool even = items * per_item == blocks;
    if (finer == 64) return steps <= 2 && blocks * 64 > columns && blocks % (columns / 64) != 0 ? finer : columns;
    return even || (steps <= 2 && blocks >= 5 && 6 * blocks >= 5 * items * per_item) ? finer : columns;
}

// Entries per tile below which 16-row strips that are two panels of `panels` (as many as the matrix has groups of 8 rows) go to
// the panel kernel as panels, and from which they are strips of dense tiles: all of them together, by their average, since
// tiles and panels are two launches; for the same reason all of them are panels where others of the matrix are, up to
// PANELS_AMONG_PANELS entries per tile (4 000 banded rows, 120 entries, a few panels among the strips: K = 32 13.3 us, all panels
// 5.0, K = 512 bf16 37.7 and 15.6).
// Time of tiles / time of panels, strips of one fill, 112 .. 208 entries per tile:
//   rows of up to 128 bytes 0.92 .. 2.0, more with the size: 192, of fewer than 5 M entries 187 (a mixture of 205 and 125
//   entries that averages that is better as tiles).
//   256 bytes and more: from 176 entries on the launch splits K over a workgroup, 0.5 .. 1.0; below 0.85 .. 1.8.  Of 5 M entries
//   and more 176 .. 192 are 1.0 .. 1.4, with 1 KiB 0.8 .. 1.0.
//   the same, 600 .. 1 000 panels of up to 1.5 M entries, which whole panels do not fill the chip with and more items delay:
//   fp32 0.85 .. 1.05 from 144 entries on, 0.94 .. 1.14 below; 16 bits 0.62 .. 1.05 at any fill (2 000 panels: 1.0 .. 1.37).
//   16 bits, up to 1 000 panels: 512 bytes 0.76 .. 1.0 with up to 1.5 M entries, 1.1 .. 1.4 with more; 1 KiB 0.6 .. 1.0 up to 4 M
//   entries, then 1.0 .. 1.2.
//   3 000 and 6 000 panels of 28 .. 48 columns, a step of 64 half empty: 0.78 .. 0.96.
constexpr int PANELS_AMONG_PANELS = 192;
constexpr int panels_below(int steps, bool half_width, int64_t panels, int64_t nnz) {
    constexpr int never = 0;
    const bool few = panels <= 1280, some = few && panels > 512;
    if (panels > 2560 && nnz < 48 * 8 * panels) return never;
    const bool many = nnz >= (int64_t)5 << 20;
    if (steps <= 2) return many ? 192 : 187;
    if (half_width && nnz < (steps > 8 ? (int64_t)1 << 22 : (int64_t)3 << 19) && (steps > 4 ? few : some)) return never;
    if (!half_width && some && nnz < (int64_t)3 << 19) return 144;
    return many && steps <= 8 ? 192 : 176;
}

// The same for rows of more than 1 KiB, whose tiles always split K over a workgroup and whose panels take a launch per 512 bytes:
// 16 bits 0.24 .. 0.76 at 100 .. 224 entries per tile; fp32 0.38 .. 0.89 with 0.2 .. 0.8 M entries, 0.8 .. 1.3 with 0.8 .. 1.8 M (1.0
// from 144 entries per tile on), 1.2 .. 1.6 with 1.6 .. 2.6 M.
constexpr int long_panels_below(bool half_width, int64_t nnz) {
    return half_width || nnz < (int64_t)1 << 20 ? 0 : nnz < (int64_t)3 << 19 ? 144 : PANELS_AMONG_PANELS;
}

// Columns of a work item of the fused call: a panel of up to 1 024 columns is one item, or two where that leaves wavefronts
// of the chip something to do (halves_from: from more columns on; 0: not).  The items of a panel add their part of the
// output rows atomically to zeros: two sums come out the same in either order, three do not.
constexpr int fused_panel_columns(int len, int halves_from) {
    return halves_from && len > halves_from && len <= 2 * PANEL_COLUMNS ? ((len + 1) / 2 + 31) / 32 * 32 : PANEL_COLUMNS;
}
// Two items per panel as long as a wavefront takes one of them each (wavefronts_per_simd of the fused kernel: 3, 2 and 1 at
// 32, 64 and 128 components), of more than 64 columns, in 16 bits of more than 128.  Whole panels / halves: 250 panels of 240
// columns K = 32 15.8 / 12.8 us, K = 128 32.1 / 22.6; 500 K = 128 33.1 / 24.1, fp16 25.5 / 22.8; 1 000 K = 64 28.7 / 22.2,
// K = 128 fp16 29.6 / 37.2; 1 500 K = 32 21.3 / 19.5, K = 64 fp16 22.1 / 26.4; 1 000 of 104 K = 64 19.4 / 16.4, fp16 15.8 /
// 16.9.  (Items of 64 columns, which made O differ from run to run: 100 of 500 K = 32 12.1 where halves take 15.8, 1 000 of
// 240 K = 128 54.)
constexpr int fused_halves_from(int64_t panels, int wavefronts_per_simd, bool half_width) {
    return 2 * panels <= (int64_t)1024 * wavefronts_per_simd ? (half_width ? 128 : 64) : 0;
}

}  // namespace sddmm
