// The context behind sddmm_ctx, error and launch macros, and the dispatch over row layouts: what the
// planning code (sddmm_amd.hip) and the launchers (launch_*.hip) share.
#pragma once
#include "../../include/sddmm_amd.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "device_pool.h"
#include "kernels_gather.h"
#include "kernels_plan.h"
#include "kernels_tile.h"

using namespace sddmm;

// ---------------------------------------------------------------------------
struct sddmm_ctx {
    int device = 0;
    hipStream_t stream = nullptr;      // where work is enqueued: own_stream unless the caller lent one
    hipStream_t own_stream = nullptr;
    bool lent_stream = false;
    bool oversize = false;             // a launch was skipped because its grid does not fit one dispatch
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    ContextParts parts;                // owner of own_stream, the events and the counters

    char err[512] = {0};

    // dense operands
    int M = 0, N = 0, K = 0, dtype = SDDMM_F32;
    bool have_dense = false;
    void *dA = nullptr, *dB = nullptr;
    bool own_dense = false;

    // sparse operand
    bool have_sparse = false, have_rowptr = false, own_sparse = false, from_coo = false;
    int sM = 0, sN = 0;
    int64_t nnz = 0;
    int32_t *d_rowptr = nullptr, *d_col = nullptr, *d_rowidx = nullptr;
    float *d_sval = nullptr, *dP = nullptr;
    bool own_rowptr = false, own_rowidx = false;

    // plan
    bool planned = false;
    int strategy = SDDMM_AUTO;       // resolved
    int requested = SDDMM_AUTO;
    DevCounters *d_pc = nullptr;     // device counters
    DevTotals raw{};                 // what the device reported last
    DevCounters *h_pc = nullptr;     // pinned landing place of the reports and of copies
    PlanCounters pc{};               // its summary
    sddmm_stats stats{};
    // AUTO: rows shorter than ts go to the many-rows-per-wave kernel, the others
    // become wave-per-segment items of at most seg entries
    int ts = 0, seg = 0, rpw = 64;
    RowItem *d_items = nullptr;
    int64_t n_items = 0, items_cap = 0;
    unsigned int *d_block_sums = nullptr, *d_block_off = nullptr;     // items per block of the row scan, their exclusive scan
    unsigned int *d_scan_sums = nullptr;    // block sums of a long scan (device_scan)
    int64_t block_sums_cap = 0, scan_sums_cap = 0;
    int64_t rows_short = 0;
    int launches = 0;
    // dense-tile (MFMA) path
    unsigned int *d_strip_ntiles = nullptr, *d_strip_off = nullptr;
    int64_t strips_cap = 0;
    TileDesc *d_tiles = nullptr;
    int64_t n_tiles = 0, tiles_cap = 0, nnz_tiles = 0;
    int tile_steps = 0;
    bool ragged = false;             // tiles and panels of the plan are of ragged rows (ragged_steps)
    bool long_rows = false;          // and of more than 1 KiB each (rows_are_long)
    bool tiles_active = false;       // d_tiles describes the current pattern
    int32_t *d_win_order = nullptr;  // order in which the launch takes the windows (null: storage order)
    unsigned int *d_win_bins = nullptr;
    int64_t win_order_cap = 0;
    bool use_win_order = false;
    TileWindow *d_windows = nullptr; // one record per TILE_WINDOW consecutive descriptors
    int64_t n_windows = 0, windows_cap = 0;
    bool use_windows = false;        // tile kernels take windows as batches (else they walk them tile by tile)
    int64_t n_tiles_natural = 0;     // descriptors: 16-row strips first, then union strips, then gathered strips
    int64_t n_tiles_lead = 0;        // empty descriptors that fill the last window before the gathered strips
    int64_t n_win_single = 0;        // windows taken one per wavefront; the rest (gathered pairs) two per wavefront
    int64_t n_tile_units = 0;        // wavefronts of a tile launch
    int64_t n_tiles_union = 0, nnz_tiles_union = 0;
    unsigned int *d_ustrip_ntiles = nullptr, *d_ustrip_off = nullptr;
    int64_t ustrips_cap = 0;
    int32_t *d_tile_cols = nullptr;  // 16 B rows per descriptor
    bool union_counted = false;
    // gathered strips: candidate rows, sorted by first column, 16 per strip
    unsigned long long *d_cand_keys = nullptr, *d_sorted_keys = nullptr;   // (first column << 32) | row
    int32_t *d_vrows = nullptr;
    void *d_sort_tmp = nullptr;
    size_t sort_tmp_bytes = 0;
    int64_t cand_cap = 0, vstrips_cap = 0, n_cand = 0, n_vstrips = 0;
    int gathered_stride = 0;         // words of a pair's kept bitmap (k_gathered_count), 0: not kept
    unsigned int *d_vstrip_ntiles = nullptr, *d_vstrip_off = nullptr;
    // row ownership (one byte per row: 0 row kernels, 1 dense tiles, 2 row panels, 3 gathered strips, 4 union strips)
    unsigned char *d_owner = nullptr;
    int64_t owner_cap = 0;
    // every work array of the plan whose size follows from the number of rows lives in one
    // allocation (a first plan then pays for one hipMalloc instead of a dozen)
    char *d_arena = nullptr;
    int64_t arena_rows = -1;
    bool owner_active = false;
    // row-panel path
    unsigned int *d_panel_counts = nullptr, *d_panel_off = nullptr;
    int64_t panels_cap = 0;
    int2 *d_short_list = nullptr;    // {position, row} of the entries of the short rows nobody owns
    int64_t n_short_list = 0, short_list_cap = 0;
    ScanJobs scan_jobs{};            // short scans waiting for the next read-back of the counters
    int n_scan_jobs = 0;
    bool use_short_list = false;
    unsigned int *d_short_sums = nullptr, *d_short_off = nullptr;     // arena views: entries of short rows per block of the row scan
    RowItem *d_panel_items = nullptr;
    int64_t n_panel_items = 0, panel_items_cap = 0, n_panels = 0, nnz_panels = 0;
    int panel_columns = 0;           // of a work item
    RowItem *d_fused_panels = nullptr;       // the items of the fused call, where they are cut otherwise
    int64_t n_fused_panels = 0, fused_panels_cap = 0;
    bool fused_panels_valid = false;
    bool panel_mfma = false;         // panels run on k_panel_mfma (else on k_panel)
    bool panels_flagged = false;     // the panel detector ran in this plan
    // FLAT in slices of K (kernels_flat.h): partial products of a range of entries, [slice][entry]
    float *d_part = nullptr;
    int64_t part_floats = 0;
    bool use_slices = false;         // set by a plan of SDDMM_AUTO
    // FLAT with the long rows cut into column blocks (k_flat_blocks)
    char *d_blocks = nullptr;        // one allocation: lists and scans of the plan, item counts, items
    size_t blocks_bytes = 0;
    RowItem *d_block_segments = nullptr, *d_block_gaps = nullptr;
    int64_t block_segments_max = 0, block_gaps_max = 0;      // as the launch sizes its grid: the true numbers where the host has them
    bool use_blocks = false;         // set by a plan of SDDMM_AUTO
    unsigned int *d_long_sums = nullptr, *d_long_off = nullptr;       // arena views: long rows per block of the row scan
    // entries that came in no order, sorted by row and column block: row and column of each, the place every entry
    // went to, and the dot products in that order
    int32_t *d_order = nullptr;      // one allocation, kept until the sparse operand goes
    int32_t *d_order_row = nullptr, *d_order_col = nullptr, *d_order_place = nullptr;
    float *d_order_dots = nullptr;
    int64_t order_cap = 0;
    int64_t coo_jumps = 0;           // entries that share neither row nor column with the one before them
    double col_near = 1.0;           // share of the entries that lie in the same 16 columns as the one before them (a sample)
    bool use_order = false;          // set by a plan of SDDMM_AUTO
    // fused SDDMM + SpMM: items covering every non-empty row, output M x K
    RowItem *d_fused_items = nullptr;
    int64_t n_fused_items = 0, fused_items_cap = 0;
    bool fused_items_valid = false;
    bool fused_items_panels = false; // the fused items leave out the rows that the panel kernel owns
    double fused_short_avg = 0.0;    // entries per non-empty row of at most FUSED_ROW_MAX entries (panel rows apart)
    int fused_row_max = FUSED_ROW_MAX;   // rows beyond it are work items of their own
    int fused_seg = 0;               // of at most so many entries
    bool fused_rows_alike = false;   // most rows beyond fused_row_max look like the row after them (banded blocks, dense tiles)
    int fused_block_waves = WAVES_PER_BLOCK;   // wavefronts per workgroup of the fused gather kernels
    int64_t n_fused_cut = 0;         // rows that k_add_cut_rows completes, listed behind the items (0: the kernel of the short rows does)
    int fused_add_block = 0;         // its workgroup size
    float *d_fused_parts = nullptr;  // partial output rows of the pieces of the rows cut into several items
    int64_t n_fused_pieces = 0, fused_part_floats = 0;
    float *dO = nullptr;
    size_t o_cap = 0;
    bool have_fused = false;
};

inline int fail(sddmm_ctx *c, int code, const char *fmt, ...) {
    if (c) {
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(c->err, sizeof(c->err), fmt, ap);
        va_end(ap);
    }
    return code;
}

#define HIP_TRY(c, call)                                                                         \
    do {                                                                                         \
        hipError_t e_ = (call);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return fail((c), SDDMM_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                        __FILE__, __LINE__);                                                     \
    } while (0)

#define ALLOC_TRY(c, ptr, bytes)                                                                 \
    do {                                                                                         \
        hipError_t e_ = pool_alloc((void **)&(ptr), (bytes));                                    \
        if (e_ != hipSuccess) {                                                                  \
            (ptr) = nullptr;                                                                     \
            return fail((c), SDDMM_ERR_ALLOC, "hipMalloc(%zu bytes) failed: %s", (size_t)(bytes), \
                        hipGetErrorString(e_));                                                  \
        }                                                                                        \
    } while (0)

// A dispatch packet counts the work-items of a grid dimension in 32 bits: a launch of 2^32
// threads or more would run only part of its grid, without any error.  Such a launch is not
// made; launch_status() turns the skipped launch into an error of the entry point.
#define SDDMM_LAUNCH(c, kernel, grid, block, ...)                                                        \
    do {                                                                                                 \
        const int64_t g_ = (int64_t)(grid);                                                              \
        const int b_ = (int)(block);                                                                     \
        if (g_ * b_ >= ((int64_t)1 << 32)) (c)->oversize = true;                                         \
        else hipLaunchKernelGGL(kernel, dim3((unsigned)g_), dim3((unsigned)b_), 0, (c)->stream, __VA_ARGS__); \
    } while (0)

inline int launch_status(sddmm_ctx *c) {
    if (!c->oversize) return SDDMM_OK;
    c->oversize = false;
    return fail(c, SDDMM_ERR_UNSUPPORTED,
                "a kernel of this strategy needs 2^32 threads or more in one launch for this matrix "
                "(one wavefront per row or per work item): use SDDMM_AUTO or SDDMM_FLAT");
}

// after a group of launches: a failed launch, or one that was not made
#define LAUNCH_CHECK(c)                                \
    do {                                               \
        HIP_TRY(c, hipGetLastError());                 \
        const int ls_ = launch_status(c);              \
        if (ls_) return ls_;                           \
    } while (0)

// the entries as the flat kernels take them: in the caller's order, or sorted by the plan
inline const int32_t *entry_rows(const sddmm_ctx *c) { return c->use_order ? c->d_order_row : c->d_rowidx; }
inline const int32_t *entry_cols(const sddmm_ctx *c) { return c->use_order ? c->d_order_col : c->d_col; }

inline size_t elem_size(int dtype) { return dtype == SDDMM_F32 ? 4 : 2; }

inline int env_int(const char *name, int fallback) {
    const char *e = getenv(name);
    return e && *e ? atoi(e) : fallback;
}

// Memory that a plan can do without: nullptr where the device has none left, or where the array is larger than
// SDDMM_SPARE_BYTES allows (no limit by default).  The plan then takes the kernels that need no such array.
inline void *spare_alloc(size_t bytes) {
    const char *limit = getenv("SDDMM_SPARE_BYTES");
    if (limit && *limit && bytes > (size_t)strtoull(limit, nullptr, 10)) return nullptr;
    void *p = nullptr;
    if (pool_alloc(&p, bytes) == hipSuccess && p) return p;
    (void)hipGetLastError();                               // the failed allocation is not an error of the plan
    return nullptr;
}

// ---- kernel dispatch over the (unit type, lanes per entry, units per lane) layouts ----
struct Shape {
    int unit;    // 0: fp32 x4, 1: fp32 x1 (K < 4), 2: bf16 x8, 3: fp16 x8, 4: fp32 x4 in rows of no whole number of units
    int KU;      // units per row
    int len;     // length of a row as the kernels take it: KU, or K where rows hold no whole number of units
    int LPN;     // lanes per entry (0: row too long for the register layout)
    int UPL;     // units per lane
    bool fullk;  // KU == LPN*UPL
    bool wide;   // operands of 4 GiB or more: 64-bit byte offsets
    bool whole() const { return unit == 0 || unit == 2 || unit == 3; }     // 16-byte units only
};

inline int pow2ceil(int x) {
    int l = 1;
    while (l < x) l <<= 1;
    return l;
}

inline Shape shape_of(const sddmm_ctx *c) {
    Shape s{};
    if (c->dtype == SDDMM_BF16 || c->dtype == SDDMM_F16) { s.unit = c->dtype == SDDMM_BF16 ? 2 : 3; s.KU = s.len = c->K / 8; }
    else if (c->K % 4 == 0) { s.unit = 0; s.KU = s.len = c->K / 4; }
    else if (c->K > 4) { s.unit = 4; s.KU = (c->K + 3) / 4; s.len = c->K; }
    else { s.unit = 1; s.KU = s.len = c->K; }
    if (s.unit == 1) {
        s.LPN = 4; s.UPL = 1;
    } else {
        // 16-byte units: 8 lanes cover one whole 128-byte cache line per load
        // instruction (measured faster than 4 lanes x 64 bytes: half the lines per
        // instruction for the same bytes)
        if (s.KU <= 8) { s.LPN = pow2ceil(s.KU); s.UPL = 1; }
        else if (s.KU <= 64) {
            // units per lane: as few as hold the row, of those that have a kernel (a lane without a unit
            // of its own loads another one again: K = 96 31.9 us with four per lane, 25.5 with three)
            s.LPN = 8;
            const int upl = (s.KU + 7) / 8;
            s.UPL = upl <= 4 ? upl : upl <= 6 ? 6 : 8;
        }
        else if (s.KU <= 128) { s.LPN = 16; s.UPL = 8; }
        else { s.LPN = 0; s.UPL = 0; }
    }
    s.fullk = s.LPN > 0 && s.KU == s.LPN * s.UPL;
    const size_t rows = (size_t)std::max(c->M, c->N);
    s.wide = rows * (size_t)c->K * elem_size(c->dtype) >= ((size_t)1 << 32);
    return s;
}

// Calls f(Layout<...>{}) for the layout matching s.
template <class U, int LPN, int UPL, class F>
void with_mask_width(const Shape &s, F &&f) {
    if (s.wide) f(Layout<U, LPN, UPL, false, true>{});
    else if (s.fullk && U::WHOLE && U::ELEMS > 1 && UPL != 3 && UPL != 6) f(Layout<U, LPN, UPL, true, false>{});
    else f(Layout<U, LPN, UPL, false, false>{});
}

template <class U, class F>
void with_layout16(const Shape &s, F &&f) {
    if (s.LPN == 0) { f(Layout<U, 0, 1, false, true>{}); return; }
    if (s.LPN == 1) with_mask_width<U, 1, 1>(s, f);
    else if (s.LPN == 2) with_mask_width<U, 2, 1>(s, f);
    else if (s.LPN == 4) with_mask_width<U, 4, 1>(s, f);
    else if (s.LPN == 16) with_mask_width<U, 16, 8>(s, f);
    else if (s.UPL == 1) with_mask_width<U, 8, 1>(s, f);
    else if (s.UPL == 2) with_mask_width<U, 8, 2>(s, f);
    else if (s.UPL == 3) with_mask_width<U, 8, 3>(s, f);
    else if (s.UPL == 4) with_mask_width<U, 8, 4>(s, f);
    else if (s.UPL == 6) with_mask_width<U, 8, 6>(s, f);
    else with_mask_width<U, 8, 8>(s, f);
}

template <class F>
void with_layout(const Shape &s, F &&f) {
    if (s.unit == 0) with_layout16<UnitF32x4>(s, f);
    else if (s.unit == 2) with_layout16<UnitBF16x8>(s, f);
    else if (s.unit == 3) with_layout16<UnitF16x8>(s, f);
    else if (s.unit == 4) with_layout16<UnitF32x4u>(s, f);
    else with_mask_width<UnitF32x1, 4, 1>(s, f);
}

// wavefronts of the short-row part of the AUTO launches: 64 entries of the entry list each, or
// rpw consecutive rows each
inline int64_t short_row_waves(const sddmm_ctx *c) {
    if (c->rows_short <= 0) return 0;
    if (c->use_short_list) return (c->n_short_list + WAVE - 1) / WAVE;
    return ((int64_t)c->sM + c->rpw - 1) / c->rpw;
}

// Row-panel detector (8 consecutive rows, 8-aligned, same column list).  Two
// kernels can run the panels: the MFMA one (rows of 36 bytes and more, up to
// 1 KiB) and the VALU one (8-lanes-per-entry layouts whose 8 A rows fit in
// registers: fp32 K = 32 or 64, bf16 / fp16 K = 64, 32-bit offsets); the VALU kernel has
// the per-entry arithmetic of the gather kernels, the MFMA kernel is faster.
inline int panel_mfma_steps(const sddmm_ctx *c) {
    const size_t row_bytes = (size_t)c->K * elem_size(c->dtype);
    if (row_bytes % 64) return 0;
    const int steps = (int)(row_bytes / 64);
    return (steps == 1 || steps == 2 || steps == 4 || steps == 8 || steps == 16) ? steps : 0;
}

// Steps of 64 bytes that the tile and panel kernels take for rows of no whole power of two of them: as many as the row
// layout of the gather kernels holds; 0: no such kernel.
inline int ragged_steps(const sddmm_ctx *c) {
    const Shape s = shape_of(c);
    if (s.unit == 1 || s.wide || (s.LPN != 4 && s.LPN != 8) || panel_mfma_steps(c) != 0) return 0;
    return s.LPN * s.UPL / 4;
}

// Rows of more than 1 KiB, which the tile and panel kernels take LONG_STEPS at a time.  (As in ragged rows the length need
// be no whole number of units.)
constexpr int LONG_STEPS = 8;
inline bool rows_are_long(const sddmm_ctx *c) {
    const Shape s = shape_of(c);
    return s.unit != 1 && !s.wide && (size_t)c->K * elem_size(c->dtype) > 1024;
}

// The device code of a translation unit is loaded when something first asks for one of its kernels: 3 .. 13 ms, once per
// process.  A plan asks for the families that its launches take (load_*, one per launch_*.hip), so that no launch has to:
// launches may be captured, and they are what callers time.
inline hipError_t load_code(const void *kernel) {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, kernel);
}
hipError_t load_flat();
hipError_t load_rows();
hipError_t load_auto();
hipError_t load_tiles(bool ragged);
hipError_t load_ragged_tiles();
hipError_t load_panels(bool ragged);
hipError_t load_ragged_panels();
hipError_t load_fused();

// ---- launchers, one translation unit per family of kernels ----
void launch_flat(sddmm_ctx *c);                                                  // launch_flat.hip
int launch_flat_blocks(sddmm_ctx *c);                                            // number of launches
void launch_unsort(sddmm_ctx *c);
void block_items_max(const sddmm_ctx *c, bool cut_long_rows, int64_t *segments, int64_t *gaps);
bool blocks_pay(const sddmm_ctx *c);
bool order_pays(const sddmm_ctx *c);
bool slices_pay(const sddmm_ctx *c, double entries_per_row);
int64_t slice_workspace_floats(const sddmm_ctx *c);
int launch_flat_sliced(sddmm_ctx *c);                                            // number of launches
void launch_row_wave(sddmm_ctx *c, const RowItem *items, int64_t n_items);       // launch_rows.hip
void launch_short_rows(sddmm_ctx *c, int ts, int rpw);
void launch_auto(sddmm_ctx *c);                                                  // launch_auto.hip
bool launch_auto_with_tiles(sddmm_ctx *c);                                       // launch_tiles.hip
void launch_tiles(sddmm_ctx *c);
bool launch_ragged_auto_with_tiles(sddmm_ctx *c);                                // launch_tiles_ragged.hip
void launch_ragged_tiles(sddmm_ctx *c);
void launch_long_tiles(sddmm_ctx *c);
void launch_panels(sddmm_ctx *c);                                                // launch_panels.hip
void launch_ragged_panels(sddmm_ctx *c);                                         // launch_panels_ragged.hip
int launch_long_panels(sddmm_ctx *c);                                            // number of launches
void launch_panels_fused(sddmm_ctx *c);
// the list of the rows for k_add_cut_rows
inline int32_t *fused_cut_rows(const sddmm_ctx *c) {
    return c->n_fused_cut > 0 ? reinterpret_cast<int32_t *>(c->d_fused_items + c->n_fused_items) : nullptr;
}
inline int64_t blocks_of(int64_t waves, int per_block) { return (waves + per_block - 1) / per_block; }
bool fused_balanced(const sddmm_ctx *c);                                           // which kernel takes the short rows
int launch_fused_rows(sddmm_ctx *c, const unsigned char *panel_owner);           // launch_fused.hip: number of launches
