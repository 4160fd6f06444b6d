// C ABI of the gfx950 SDDMM engine: context, operand upload, plan, run.
// See include/sddmm_amd.h for the contract of every entry point.
#include "context.h"

#include <mutex>

#include <rocprim/device/device_radix_sort.hpp>

namespace {

// Gives a block back: to the pool if the caller has waited for the device, otherwise to hipFree.
template <class T>
void dfree(T *&p, bool idle = false) {
    pool_free((void *)p, idle);
    p = nullptr;
}

// Views into the plan arena: nothing here is freed on its own.
void release_arena(sddmm_ctx *c, bool idle = false) {
    dfree(c->d_arena, idle);
    c->arena_rows = -1;
    c->d_owner = nullptr;
    c->d_strip_ntiles = c->d_strip_off = c->d_ustrip_ntiles = c->d_ustrip_off = nullptr;
    c->d_panel_counts = c->d_panel_off = c->d_vstrip_ntiles = c->d_vstrip_off = nullptr;
    c->d_cand_keys = c->d_sorted_keys = nullptr;
    c->d_vrows = nullptr;
    c->d_block_sums = c->d_short_sums = c->d_long_sums = nullptr;
    c->d_block_off = c->d_short_off = c->d_long_off = c->d_scan_sums = nullptr;
    c->owner_cap = c->strips_cap = c->ustrips_cap = c->panels_cap = c->cand_cap = c->vstrips_cap = 0;
    c->block_sums_cap = 0;
}

int ensure_arena(sddmm_ctx *c) {
    const int64_t M = c->sM;
    if (c->d_arena && c->arena_rows == M) return SDDMM_OK;
    release_arena(c);
    const int64_t n_strips = (M + 15) / 16, n_panels = M / 8 + 1;
    const int64_t n_sums = M * COL_BLOCKS_MAX / SCAN_TILE + 8;  // the longest scan: a count per row and column block
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    };
    const size_t o_owner = take((size_t)M + 64);
    const size_t o_strip_n = take((size_t)n_strips * 4), o_strip_o = take((size_t)n_strips * 4);
    const size_t o_ustrip_n = take((size_t)n_strips * 4), o_ustrip_o = take((size_t)n_strips * 4);
    // (gathered strips come in pairs: up to two more than M / 16)
    const size_t o_vstrip_n = take((size_t)(n_strips + 2) * 4), o_vstrip_o = take((size_t)(n_strips + 2) * 4);
    const size_t o_vrows = take((size_t)(n_strips + 2) * 16 * 4);
    const size_t o_panel_n = take((size_t)n_panels * 4), o_panel_o = take((size_t)n_panels * 4);
    const size_t o_keys = take((size_t)(M + 1) * 8), o_sorted = take((size_t)(M + 1) * 8);
    const size_t n_blocks = (size_t)((M + SCAN_TILE - 1) / SCAN_TILE);
    const size_t o_scan = take((size_t)n_sums * 4), o_sums = take(n_blocks * 4), o_short_sums = take(n_blocks * 4), o_long_sums = take(n_blocks * 4);
    const size_t o_off = take(n_blocks * 4), o_short_off = take(n_blocks * 4), o_long_off = take(n_blocks * 4);
    ALLOC_TRY(c, c->d_arena, at);
    char *b = c->d_arena;
    c->d_owner = (unsigned char *)(b + o_owner);
    c->d_strip_ntiles = (unsigned int *)(b + o_strip_n); c->d_strip_off = (unsigned int *)(b + o_strip_o);
    c->d_ustrip_ntiles = (unsigned int *)(b + o_ustrip_n); c->d_ustrip_off = (unsigned int *)(b + o_ustrip_o);
    c->d_vstrip_ntiles = (unsigned int *)(b + o_vstrip_n); c->d_vstrip_off = (unsigned int *)(b + o_vstrip_o);
    c->d_vrows = (int32_t *)(b + o_vrows);
    c->d_panel_counts = (unsigned int *)(b + o_panel_n); c->d_panel_off = (unsigned int *)(b + o_panel_o);
    c->d_cand_keys = (unsigned long long *)(b + o_keys); c->d_sorted_keys = (unsigned long long *)(b + o_sorted);
    c->d_block_sums = (unsigned int *)(b + o_sums);
    c->d_short_sums = (unsigned int *)(b + o_short_sums);
    c->d_long_sums = (unsigned int *)(b + o_long_sums);
    c->d_block_off = (unsigned int *)(b + o_off);
    c->d_short_off = (unsigned int *)(b + o_short_off);
    c->d_long_off = (unsigned int *)(b + o_long_off);
    c->d_scan_sums = (unsigned int *)(b + o_scan);
    c->owner_cap = M + 64;
    c->strips_cap = c->ustrips_cap = n_strips;
    c->vstrips_cap = n_strips + 2;
    c->panels_cap = n_panels;
    c->cand_cap = M + 1;
    c->scan_sums_cap = n_sums;
    c->block_sums_cap = (int64_t)n_blocks;
    c->arena_rows = M;
    return SDDMM_OK;
}

// an arena view turned out too small: the sizes above are upper bounds, so this is a bug
#define ARENA_HOLDS(c, need, cap, what)                                                             \
    do {                                                                                            \
        if ((int64_t)(need) > (int64_t)(cap))                                                       \
            return fail((c), SDDMM_ERR_HIP, "internal: plan arena too small for %s (%lld > %lld)", what, \
                        (long long)(need), (long long)(cap));                                       \
    } while (0)

// Nothing that uses a block may be in flight when the block is handed on: release_* wait for the whole device (unless the
// caller has), since a caller may read the results on a stream of its own.
void release_dense(sddmm_ctx *c, bool idle = false) {
    idle = idle || (c->own_dense && pool_wait());
    if (c->own_dense) { dfree(c->dA, idle); dfree(c->dB, idle); }
    c->dA = c->dB = nullptr;
    c->have_fused = false;
    c->own_dense = false;
    c->have_dense = false;
    c->planned = false;
}

void release_sparse(sddmm_ctx *c, bool idle = false) {
    // (every pattern has its array of results, a context without one nothing to give back)
    idle = idle || (c->dP && pool_wait());
    if (c->own_sparse) { dfree(c->d_col, idle); dfree(c->d_sval, idle); }
    if (c->own_rowptr) dfree(c->d_rowptr, idle);
    if (c->own_rowidx) dfree(c->d_rowidx, idle);
    dfree(c->dP, idle);
    dfree(c->d_items, idle);
    dfree(c->d_tiles, idle);
    dfree(c->d_tile_cols, idle);
    dfree(c->d_windows, idle);
    dfree(c->d_win_order, idle);
    dfree(c->d_win_bins, idle);
    c->win_order_cap = 0;
    c->use_win_order = false;
    c->n_windows = c->windows_cap = 0;
    c->ustrips_cap = 0;
    dfree(c->d_sort_tmp, idle);
    release_arena(c, idle);
    c->sort_tmp_bytes = 0;
    c->cand_cap = c->vstrips_cap = c->n_cand = c->n_vstrips = 0;
    dfree(c->d_panel_items, idle);
    dfree(c->d_fused_panels, idle);
    c->n_fused_panels = c->fused_panels_cap = 0;
    c->fused_panels_valid = false;
    dfree(c->d_short_list, idle);
    c->short_list_cap = c->n_short_list = 0;
    c->use_short_list = false;
    dfree(c->d_order, idle);
    c->d_order_row = c->d_order_col = c->d_order_place = nullptr;
    c->d_order_dots = nullptr;
    c->order_cap = 0;
    c->use_order = false;
    dfree(c->d_fused_items, idle);
    c->n_fused_items = c->n_fused_cut = c->fused_items_cap = 0;
    dfree(c->d_fused_parts, idle);
    c->n_fused_pieces = c->fused_part_floats = 0;
    c->fused_items_valid = c->have_fused = false;
    c->owner_cap = c->panels_cap = c->panel_items_cap = 0;
    c->n_panel_items = c->n_panels = c->nnz_panels = 0;
    c->owner_active = false;
    c->items_cap = c->block_sums_cap = c->n_items = 0;
    c->strips_cap = c->tiles_cap = c->n_tiles = c->nnz_tiles = 0;
    c->tiles_active = false;
    c->d_col = nullptr; c->d_sval = nullptr; c->d_rowptr = nullptr; c->d_rowidx = nullptr;
    c->own_sparse = c->own_rowptr = c->own_rowidx = false;
    c->n_scan_jobs = 0;                       // (of a plan that failed: their arrays are gone)
    c->have_sparse = c->have_rowptr = false;
    c->from_coo = false;
    c->planned = false;
    c->nnz = 0;
}

int grid_for(int64_t n, int block) { return (int)std::max<int64_t>(1, (n + block - 1) / block); }
int grid_capped(int64_t n, int block, int cap = 16384) {
    return (int)std::min<int64_t>(cap, std::max<int64_t>(1, (n + block - 1) / block));
}

// The short scans of a plan (tiles per strip, items per panel, block sums of the row classes ...) feed
// nothing before the next read-back of the counters, so they are collected and run as ONE launch
// there instead of one launch each behind its producer.
int flush_scans(sddmm_ctx *c) {
    if (c->n_scan_jobs == 0) return SDDMM_OK;
    SDDMM_LAUNCH(c, k_scan_jobs, c->n_scan_jobs, SCAN_BLOCK, c->scan_jobs, c->n_scan_jobs, (const DevCounters *)c->d_pc, (DevTotals *)nullptr);
    c->n_scan_jobs = 0;
    LAUNCH_CHECK(c);
    return SDDMM_OK;
}
int queue_scan(sddmm_ctx *c, const unsigned int *in, unsigned int *out, int64_t n, unsigned long long *d_total) {
    if (c->n_scan_jobs == SCAN_JOBS_MAX) {
        const int rc = flush_scans(c);
        if (rc) return rc;
    }
    c->scan_jobs.job[c->n_scan_jobs++] = ScanJob{in, out, d_total, (int)n, 0};
    return SDDMM_OK;
}

// The scans that wait and a report of the counters; waits for it.
int read_totals(sddmm_ctx *c, DevTotals *out) {
    static_assert(sizeof(DevTotals) <= sizeof(DevCounters::k), "the slots' place in the pinned block");
    DevTotals *const totals = reinterpret_cast<DevTotals *>(&c->h_pc->k[0][0]);
    SDDMM_LAUNCH(c, k_scan_jobs, c->n_scan_jobs + 1, SCAN_BLOCK, c->scan_jobs, c->n_scan_jobs, (const DevCounters *)c->d_pc, totals);
    c->n_scan_jobs = 0;
    LAUNCH_CHECK(c);
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    *out = *totals;
    return SDDMM_OK;
}
int fetch_counters(sddmm_ctx *c) {
    const int rc = read_totals(c, &c->raw);
    if (rc) return rc;
    c->pc = summarize(c->raw);
    return SDDMM_OK;
}

// rows per wavefront of the many-rows body: about 256 short entries per wave, so
// that small matrices still produce enough waves to fill the chip
int rows_per_wave(double avg_short_len) {
    int rpw = 64;
    while (rpw > 8 && rpw * std::max(avg_short_len, 1.0) > 384.0) rpw >>= 1;
    return rpw;
}

// Row classifier: statistics, then the item list of the wave-per-segment kernel.
// Row classes and work items of the rows nobody owns, in two halves around a read-back of the
// counters: the count (launch only; it finds its counters cleared, begin_ownership), the scans of its sums (k_gathered_count
// takes the rows of the gathered strips out of the sums, which are then scanned once more) ...
int classify_rows_scan(sddmm_ctx *c) {
    const int64_t nb = ((int64_t)c->sM + SCAN_TILE - 1) / SCAN_TILE;
    if (nb == 0) return SDDMM_OK;
    if (nb <= SCAN_SMALL_MAX) {
        int rc = queue_scan(c, c->d_block_sums, c->d_block_off, nb, &c->d_pc->n_items);
        if (rc) return rc;
        rc = queue_scan(c, c->d_short_sums, c->d_short_off, nb, &c->d_pc->short_scanned);
        if (rc) return rc;
        return queue_scan(c, c->d_long_sums, c->d_long_off, nb, &c->d_pc->long_scanned);
    }
    SDDMM_LAUNCH(c, k_scan_block_sums, 1, SCAN_BLOCK, (const unsigned int *)c->d_block_sums, c->d_block_off, (int)nb, &c->d_pc->n_items);
    SDDMM_LAUNCH(c, k_scan_block_sums, 1, SCAN_BLOCK, (const unsigned int *)c->d_short_sums, c->d_short_off, (int)nb,
                 &c->d_pc->short_scanned);
    SDDMM_LAUNCH(c, k_scan_block_sums, 1, SCAN_BLOCK, (const unsigned int *)c->d_long_sums, c->d_long_off, (int)nb,
                 &c->d_pc->long_scanned);
    LAUNCH_CHECK(c);
    return SDDMM_OK;
}
int classify_rows_count(sddmm_ctx *c) {
    const int64_t nb = ((int64_t)c->sM + SCAN_TILE - 1) / SCAN_TILE;
    ARENA_HOLDS(c, nb, c->block_sums_cap, "block sums");
    if (nb > 0) {
        const unsigned char *owner = c->owner_active ? c->d_owner : nullptr;
        SDDMM_LAUNCH(c, k_classify_count, nb, SCAN_BLOCK, c->d_rowptr, owner,
                           c->sM, c->ts, c->seg, c->d_block_sums, c->d_pc, 0, c->d_short_sums, c->d_long_sums,
                           (const int32_t *)nullptr, 0);
        LAUNCH_CHECK(c);
    }
    return classify_rows_scan(c);
}
// ... and the items, once the counters are on the host (nothing may use the block sums in between)
int classify_rows_items(sddmm_ctx *c) {
    const int64_t nb = ((int64_t)c->sM + SCAN_TILE - 1) / SCAN_TILE;
    c->n_items = (int64_t)c->pc.n_items;
    c->rows_short = (int64_t)c->pc.rows_short;
    c->rpw = env_int("SDDMM_RPW", rows_per_wave(c->rows_short ? (double)c->pc.nnz_short / (double)c->rows_short : 0.0));
    c->rpw = std::min(64, std::max(1, c->rpw));
    if (c->n_items > c->items_cap) {
        dfree(c->d_items);
        ALLOC_TRY(c, c->d_items, (size_t)c->n_items * sizeof(RowItem));
        c->items_cap = c->n_items;
    }
    if (c->n_items > 0) {
        SDDMM_LAUNCH(c, k_classify_write, nb, SCAN_BLOCK, c->d_rowptr,
                           (const unsigned char *)(c->owner_active ? c->d_owner : nullptr), c->sM, c->ts, c->seg,
                           (const unsigned int *)c->d_block_off, c->d_items, 0);
        LAUNCH_CHECK(c);
    }
    // the entries of the short rows as a list, taken 64 at a time (entry_list_body)
    c->n_short_list = 0;
    c->use_short_list = env_int("SDDMM_SHORT_LIST", 1) != 0 && c->rows_short > 0;
    if (c->use_short_list) {
        c->n_short_list = (int64_t)c->pc.nnz_short;
        if ((int64_t)c->raw.short_scanned != c->n_short_list)
            return fail(c, SDDMM_ERR_HIP, "internal: scan of the short rows disagrees with their entry count");
        // The list is a convenience of 8 bytes per entry of a short row.  Above a cap
        // (SDDMM_SHORT_LIST_MAX entries, default 2^27 = 1 GiB), or when the device cannot
        // hold it, the launch walks the short rows themselves (short_rows_body) instead.
        const int64_t cap = (int64_t)env_int("SDDMM_SHORT_LIST_MAX", 1 << 27);
        if (c->n_short_list > cap) c->use_short_list = false;
        if (c->use_short_list && c->n_short_list > c->short_list_cap) {
            dfree(c->d_short_list);
            c->short_list_cap = 0;
            c->d_short_list = static_cast<int2 *>(spare_alloc((size_t)c->n_short_list * sizeof(int2)));
            if (c->d_short_list) c->short_list_cap = c->n_short_list;
            else c->use_short_list = false;
        }
        if (!c->use_short_list) c->n_short_list = 0;
    }
    if (c->use_short_list) {
        SDDMM_LAUNCH(c, k_short_list_write, nb * SHORT_LIST_SPLIT, SCAN_BLOCK, c->d_rowptr,
                           (const unsigned char *)(c->owner_active ? c->d_owner : nullptr), c->sM, c->ts,
                           (const unsigned int *)c->d_short_off, c->d_short_list);
        LAUNCH_CHECK(c);
    }
    return SDDMM_OK;
}

// Exclusive scan of n unsigned ints on the device (in != out), total to *d_total.
int device_scan(sddmm_ctx *c, const unsigned int *in, unsigned int *out, int64_t n, unsigned long long *d_total) {
    if (n <= SCAN_SMALL_MAX) return queue_scan(c, in, out, n, d_total);
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    ARENA_HOLDS(c, nb, c->scan_sums_cap, "block sums");
    SDDMM_LAUNCH(c, k_scan_sums, nb, SCAN_BLOCK, in, n, c->d_scan_sums);
    SDDMM_LAUNCH(c, k_scan_block_sums, 1, SCAN_BLOCK, (const unsigned int *)c->d_scan_sums, c->d_scan_sums, (int)nb, d_total);
    SDDMM_LAUNCH(c, k_scan_apply, nb, SCAN_BLOCK, in, n,
                       (const unsigned int *)c->d_scan_sums, out);
    LAUNCH_CHECK(c);
    return SDDMM_OK;
}

// Clears the row-ownership bytes (owners false: k_own_rows writes them all), the sums of the row classes and the counters
// before the classifiers run.
int begin_ownership(sddmm_ctx *c, bool owners) {
    const int64_t bytes = (int64_t)c->sM + 64;
    const int arc = ensure_arena(c);
    if (arc) return arc;
    ARENA_HOLDS(c, bytes, c->owner_cap, "row owners");
    const int64_t n_sums = c->d_block_off - c->d_block_sums;              // (the three arrays of sums lie next to each other)
    const int64_t threads = std::max(n_sums, owners ? (bytes + 15) / 16 : 0);
    SDDMM_LAUNCH(c, k_plan_reset, grid_for(threads, 256), 256, c->d_owner, owners ? bytes : (int64_t)0, c->d_block_sums, n_sums, c->d_pc);
    LAUNCH_CHECK(c);
    c->owner_active = true;
    c->tiles_active = false;
    c->n_tiles = c->nnz_tiles = c->n_tiles_natural = c->n_tiles_union = c->nnz_tiles_union = 0;
    c->n_tiles_lead = c->n_win_single = c->n_tile_units = 0;
    c->n_cand = c->n_vstrips = 0;
    c->union_counted = false;
    c->n_panel_items = c->n_panels = c->nnz_panels = 0;
    return SDDMM_OK;
}

// tile_steps stays 0 when the tile path does not apply (row length).
bool tile_path_applies(sddmm_ctx *c) {
    c->tile_steps = 0;
    if (c->nnz == 0) return false;
    c->tile_steps = c->long_rows ? LONG_STEPS : c->ragged ? ragged_steps(c) : panel_mfma_steps(c);
    return c->tile_steps != 0;
}

// Ragged rows on the tile and panel kernels instead of the gather kernels, and their gathered strips?
bool ragged_gathers(const sddmm_ctx *c) {
    const int steps = ragged_steps(c), mode = env_int("SDDMM_RAGGED", -1);       // -1: decide here, 0: never, 1: wherever it can
    if (c->long_rows || steps > ragged_gathered_steps(c->dtype != SDDMM_F32)) return false;
    return mode > 0 || c->nnz >= ragged_gathered_entries(steps, c->dtype != SDDMM_F32);
}
bool ragged_pays(const sddmm_ctx *c) {
    const int steps = ragged_steps(c), mode = env_int("SDDMM_RAGGED", -1);
    if (steps == 0 || mode >= 0) return steps != 0 && mode != 0;
    return c->col_near >= STRUCTURED_NEAR ? c->nnz >= ragged_entries(steps) : c->col_near >= GATHERED_NEAR && ragged_gathers(c);
}

// Rows of more than 1 KiB on the tile and panel kernels, if they own nearly all of the entries?
bool long_pays(const sddmm_ctx *c) {
    const int mode = env_int("SDDMM_LONG_TILES", -1);              // -1: decide here, 0: never, 1: wherever it can
    if (!rows_are_long(c) || mode == 0) return false;
    return mode > 0 || (c->nnz >= long_row_entries((int64_t)c->K * (int64_t)elem_size(c->dtype)) && c->col_near >= STRUCTURED_NEAR);
}

// A workgroup of 16 wavefronts per strip, not four strips to a workgroup of four wavefronts: where the chip holds them all at
// once and a strip is more than two round trips of a wavefront.  (k_own_rows four to a workgroup / one: 66 strips of 6 300
// entries 22.1 / 14.2 us, 130 of 4 000 22.0 / 16.7, 1 037 of 5 200 25.7 / 65.6.)
bool strips_are_wide(const sddmm_ctx *c) {
    const int64_t n_strips = ((int64_t)c->sM + 15) / 16;
    return n_strips <= 512 && c->nnz >= 2048 * n_strips;
}

// After the classifiers: panels of ragged fp32 rows of more than 512 bytes, and too few of them for kernels that occupy the chip
// with one or two wavefronts per SIMD.  (Gather kernels / panels: 117 panels of 224 columns K = 200 10.8 / 12.7 us; 577 k
// entries K = 196 22.3 / 15.4.)
bool too_few_panels(const sddmm_ctx *c) {
    if (!c->ragged || c->long_rows || (int64_t)c->pc.nnz_panels <= c->nnz / 2) return false;
    return env_int("SDDMM_RAGGED", -1) < 0 && c->dtype == SDDMM_F32 && ragged_steps(c) > 8 && c->nnz < 1 << 18;
}

// The rows' owners and, of the rows that are left, the candidates of the gathered strips and the row classes (launches
// only; fetch_counters brings the totals).  Rules that do not apply have been taken out.
int plan_owners(sddmm_ctx *c, const OwnRules &rules) {
    const int64_t M = c->sM, n_strips = (M + 15) / 16;
    ARENA_HOLDS(c, n_strips, c->strips_cap, "strips");
    ARENA_HOLDS(c, n_strips, c->ustrips_cap, "union strips");
    ARENA_HOLDS(c, M / 8, c->panels_cap, "panels");
    ARENA_HOLDS(c, M, c->cand_cap, "candidate rows");
    ARENA_HOLDS(c, (M + SCAN_TILE - 1) / SCAN_TILE, c->block_sums_cap, "block sums");
    const OwnArrays out{c->d_owner, c->d_strip_ntiles, c->d_panel_counts, c->d_ustrip_ntiles, c->d_cand_keys,
                        c->d_block_sums, c->d_short_sums, c->d_long_sums, c->d_vstrip_ntiles};
    // a group of four strips per workgroup, several one after the other where there are more than the chip holds at a time (five
    // per CU; a workgroup ends with atomics: graph of 200 000 rows, new pattern with every call 238 us with one group, 222 with two)
    const int64_t groups = (n_strips + STRIPS_PER_BLOCK - 1) / STRIPS_PER_BLOCK;
    const int each = (int)std::min<int64_t>(16, std::max<int64_t>(1, groups / 1280));
    if (strips_are_wide(c))
        SDDMM_LAUNCH(c, k_own_rows<true>, n_strips, WIDE_BLOCK, c->d_rowptr, c->d_col, c->sM, n_strips, 1, rules, out, c->d_pc);
    else
        SDDMM_LAUNCH(c, k_own_rows<false>, (groups + each - 1) / each, WAVE * STRIPS_PER_BLOCK, c->d_rowptr, c->d_col, c->sM, n_strips,
                     each, rules, out, c->d_pc);
    LAUNCH_CHECK(c);
    c->panels_flagged = rules.panel_min != 0;
    c->union_counted = rules.union_fill != 0;
    int rc = SDDMM_OK;
    if (rules.strip_fill) rc = device_scan(c, c->d_strip_ntiles, c->d_strip_off, n_strips, &c->d_pc->tiles_scanned);
    if (!rc && rules.panel_min) rc = device_scan(c, c->d_panel_counts, c->d_panel_off, M / 8, &c->d_pc->panel_items);
    if (!rc && rules.union_fill) rc = device_scan(c, c->d_ustrip_ntiles, c->d_ustrip_off, n_strips, &c->d_pc->utiles_scanned);
    return rc ? rc : classify_rows_scan(c);
}

// Strips of two panels that plan_owners sent either way go one way (launches only).
int settle_owners(sddmm_ctx *c, bool to_panels, int pseg) {
    const int64_t M = c->sM, n_strips = (M + 15) / 16;
    const OwnArrays out{c->d_owner, c->d_strip_ntiles, c->d_panel_counts, c->d_ustrip_ntiles, c->d_cand_keys,
                        c->d_block_sums, c->d_short_sums, c->d_long_sums, c->d_vstrip_ntiles};
    SDDMM_LAUNCH(c, k_settle_owners, (n_strips + 255) / 256, 256, c->d_rowptr, c->sM, n_strips, (int)to_panels, pseg, out, c->d_pc);
    LAUNCH_CHECK(c);
    const int rc = device_scan(c, c->d_strip_ntiles, c->d_strip_off, n_strips, &c->d_pc->tiles_scanned);
    return rc ? rc : device_scan(c, c->d_panel_counts, c->d_panel_off, M / 8, &c->d_pc->panel_items);
}

// after a fetch_counters that follows plan_owners (and precedes the gathered strips)
int take_tile_counts(sddmm_ctx *c) {
    c->n_tiles = c->n_tiles_natural = (int64_t)c->pc.n_tiles;
    c->nnz_tiles = (int64_t)c->pc.nnz_tiles;
    if (c->tile_steps != 0 && (int64_t)c->pc.tiles_scanned != c->n_tiles)
        return fail(c, SDDMM_ERR_HIP, "internal: tile scan disagrees with tile count");
    c->n_tiles_union = c->union_counted ? (int64_t)c->pc.n_utiles : 0;
    c->nnz_tiles_union = c->union_counted ? (int64_t)c->pc.nnz_utiles : 0;
    if (c->union_counted && (int64_t)c->pc.utiles_scanned != c->n_tiles_union)
        return fail(c, SDDMM_ERR_HIP, "internal: union tile scan disagrees with tile count");
    c->n_tiles += c->n_tiles_union;
    c->nnz_tiles += c->nnz_tiles_union;
    return SDDMM_OK;
}

// after the fetch_counters that follows plan_owners
int plan_gathered_count(sddmm_ctx *c, int min_fill, bool *launched) {
    *launched = false;
    if (c->tile_steps == 0 || c->sM < 2) return SDDMM_OK;
    c->n_cand = (int64_t)c->raw.n_candidates;
    // ragged rows: fewer tiles than the chip holds wavefronts do not pay (800 of 8 000 rows near-dense, 280 / 120 entries
    // each: fp32 K = 100 13.6 us without, 15.8 with them / 8.6 and 13.0, bf16 K = 72 9.8 and 7.3 / 6.0 and 7.3)
    if (c->n_cand < (c->ragged ? 1024 : 2)) { c->n_cand = 0; return SDDMM_OK; }
    int rc;
    // candidates ordered by (first column, row): a few thousand by their ranks in one launch (4 us against 23 us
    // for the radix sort on 3 000 keys), more by the library's radix sort
    if (c->n_cand <= RANK_SORT_MAX && env_int("SDDMM_RANK_SORT", 1) != 0) {
        constexpr int per_block = RANK_SORT_BLOCK / RANK_SORT_SPLIT;
        SDDMM_LAUNCH(c, k_rank_sort, (unsigned)((c->n_cand + per_block - 1) / per_block), RANK_SORT_BLOCK,
                           (const unsigned long long *)c->d_cand_keys, (unsigned long long *)c->d_sorted_keys, (int)c->n_cand);
        LAUNCH_CHECK(c);
    } else {
        size_t need = 0;
        HIP_TRY(c, rocprim::radix_sort_keys(nullptr, need, c->d_cand_keys, c->d_sorted_keys, (size_t)c->n_cand, 0, 64,
                                            c->stream));
        if (need > c->sort_tmp_bytes) {
            dfree(c->d_sort_tmp);
            ALLOC_TRY(c, c->d_sort_tmp, need);
            c->sort_tmp_bytes = need;
        }
        HIP_TRY(c, rocprim::radix_sort_keys(c->d_sort_tmp, need, c->d_cand_keys, c->d_sorted_keys, (size_t)c->n_cand, 0, 64,
                                            c->stream));
    }
    // pairs of strips: 32 consecutive candidates share one list of tile columns
    const int64_t M = c->sM;
    const int64_t n_vpairs = (c->n_cand + 31) / 32;
    c->n_vstrips = 2 * n_vpairs;
    ARENA_HOLDS(c, c->n_vstrips, c->vstrips_cap, "gathered strips");
    // the bitmaps of the pairs wait for k_gathered_tiles where the unsorted keys were, if they fit there
    c->gathered_stride = 2 + std::min(STRIP_BM_WORDS, (c->sN + 511) / 512);
    if (n_vpairs * c->gathered_stride * (int64_t)sizeof(unsigned int) > (M + 1) * (int64_t)sizeof(unsigned long long)) c->gathered_stride = 0;
    const RowClasses rows{c->d_block_sums, c->d_short_sums, c->d_long_sums, c->ts, c->seg};
    SDDMM_LAUNCH(c, k_gathered_count, n_vpairs, GATHERED_BLOCK, c->d_rowptr, c->d_col,
                       (const unsigned long long *)c->d_sorted_keys, c->n_cand, n_vpairs, min_fill, c->d_vstrip_ntiles,
                       c->d_vrows, c->d_owner, c->d_pc, rows, (unsigned int *)c->d_cand_keys, c->gathered_stride);
    LAUNCH_CHECK(c);
    rc = device_scan(c, c->d_vstrip_ntiles, c->d_vstrip_off, c->n_vstrips, &c->d_pc->tiles_scanned);
    if (rc) return rc;
    *launched = true;
    return SDDMM_OK;
}
// after the counters came back
int plan_gathered_take(sddmm_ctx *c) {
    const int64_t gathered = (int64_t)c->pc.n_tiles - c->n_tiles_natural;
    if ((int64_t)c->pc.tiles_scanned != gathered)
        return fail(c, SDDMM_ERR_HIP, "internal: gathered tile scan disagrees with tile count");
    // the gathered descriptors start a window of their own: the strips before them are padded
    // to a multiple of TILE_WINDOW with descriptors that stand for nothing
    const int64_t before = c->n_tiles_natural + c->n_tiles_union;
    c->n_tiles_lead = gathered > 0 ? (TILE_WINDOW - before % TILE_WINDOW) % TILE_WINDOW : 0;
    c->n_tiles = before + c->n_tiles_lead + gathered;
    c->nnz_tiles = (int64_t)c->pc.nnz_tiles + c->nnz_tiles_union;
    return SDDMM_OK;
}

// When the storage order of the windows (strip by strip) makes every XCD touch more of A and B
// than its L2 holds, the launch takes them block by block of a RB x CB grid over (strips, tile
// columns), one block per XCD (k_window_histogram and following).
int plan_window_order(sddmm_ctx *c) {
    c->use_win_order = false;
    const int mode = env_int("SDDMM_WINDOW_ORDER", -1);          // -1: decide here, 0: never, 1: always
    const double row_bytes = (double)c->K * (double)elem_size(c->dtype);
    const double a_bytes = (double)c->sM * row_bytes, b_bytes = (double)c->N * row_bytes;
    const double l2 = 4.0 * 1024 * 1024;
    // storage order: an XCD has an eighth of the strips and, over the launch, all of B
    if (mode == 0 || c->n_windows < 8 * NUM_XCD) return SDDMM_OK;
    // (gathered strips come sorted by column window already: reordering them measured 12 % slower)
    if (mode < 0 && c->n_tiles != c->n_tiles_natural) return SDDMM_OK;
    if (mode < 0 && a_bytes / NUM_XCD + b_bytes <= 0.75 * l2) return SDDMM_OK;
    // resident part of A per XCD within half an L2, then the least traffic A * CB + B * RB
    int RB = NUM_XCD, CB = 1;
    double best = -1.0;
    for (int rb = 1; rb <= NUM_XCD; rb *= 2) {
        const int cb = NUM_XCD / rb;
        const double traffic = a_bytes * cb + b_bytes * rb;
        const bool fits = a_bytes / rb <= 0.6 * l2;
        if (!fits && rb != NUM_XCD) continue;
        if (best < 0 || traffic < best) { best = traffic; RB = rb; CB = cb; }
    }
    if (c->n_windows > c->win_order_cap) {
        dfree(c->d_win_order);
        c->win_order_cap = 0;
        ALLOC_TRY(c, c->d_win_order, (size_t)c->n_windows * sizeof(int32_t));
        c->win_order_cap = c->n_windows;
    }
    const int64_t strip_span = std::max<int64_t>(1, std::max(((int64_t)c->sM + 15) / 16, c->n_vstrips));
    const int64_t tile_col_span = std::max<int64_t>(1, ((int64_t)c->N + 15) / 16);
    if (c->n_windows <= WINDOW_ORDER_BLOCK * WINDOW_ORDER_EACH) {
        SDDMM_LAUNCH(c, k_window_order, 1, WINDOW_ORDER_BLOCK, (const TileDesc *)c->d_tiles, (int)c->n_windows, strip_span, tile_col_span,
                     RB, CB, c->d_win_order);
        LAUNCH_CHECK(c);
        c->use_win_order = true;
        return SDDMM_OK;
    }
    if (!c->d_win_bins) ALLOC_TRY(c, c->d_win_bins, (size_t)WINDOW_BINS * sizeof(unsigned int));
    HIP_TRY(c, hipMemsetAsync(c->d_win_bins, 0, (size_t)WINDOW_BINS * sizeof(unsigned int), c->stream));
    const unsigned grid = (unsigned)((c->n_windows + 255) / 256);
    SDDMM_LAUNCH(c, k_window_histogram, grid, 256, (const TileDesc *)c->d_tiles, c->n_windows, strip_span, tile_col_span,
                       RB, CB, c->d_win_bins);
    SDDMM_LAUNCH(c, k_window_offsets, 1, WINDOW_BINS, c->d_win_bins);
    SDDMM_LAUNCH(c, k_window_scatter, grid, 256, (const TileDesc *)c->d_tiles, c->n_windows, strip_span, tile_col_span,
                       RB, CB, c->d_win_bins, c->d_win_order);
    LAUNCH_CHECK(c);
    c->use_win_order = true;
    return SDDMM_OK;
}

int plan_tiles_fill(sddmm_ctx *c) {
    if (c->n_tiles == 0) return SDDMM_OK;
    if (c->n_tiles > c->tiles_cap) {
        dfree(c->d_tiles);
        dfree(c->d_tile_cols);
        c->tiles_cap = 0;
        ALLOC_TRY(c, c->d_tiles, (size_t)c->n_tiles * sizeof(TileDesc));
        ALLOC_TRY(c, c->d_tile_cols, (size_t)c->n_tiles * 16 * sizeof(int32_t));
        c->tiles_cap = c->n_tiles;
    }
    // (1 037 strips, 33 000 tiles: k_strip_tiles and k_tile_rows 40 us, k_strip_tiles_wide 29; 35 strips 48 and 16.5.  Many more
    // strips than tiles: a workgroup that finds nothing costs 16 wavefronts)
    const bool strips_complete = ((int64_t)c->sM + 15) / 16 <= 8192;
    if (c->n_tiles_natural > 0) {
        const int64_t n_strips = ((int64_t)c->sM + 15) / 16;
        const unsigned strip_grid = (unsigned)((n_strips + STRIPS_PER_BLOCK - 1) / STRIPS_PER_BLOCK);
        if (strips_complete)
            SDDMM_LAUNCH(c, k_strip_tiles_wide, n_strips, WIDE_BLOCK, c->d_rowptr, c->d_col, c->sM, c->d_strip_ntiles, c->d_strip_off,
                         c->d_tiles, c->d_tile_cols);
        else
            SDDMM_LAUNCH(c, k_strip_tiles, strip_grid, WAVE * STRIPS_PER_BLOCK, c->d_rowptr, c->d_col, c->sM, n_strips,
                         c->d_strip_ntiles, c->d_strip_off, c->d_tiles, c->d_tile_cols);
        LAUNCH_CHECK(c);
    }
    if (c->n_tiles_union > 0) {
        const int64_t n_strips = ((int64_t)c->sM + 15) / 16;
        const unsigned strip_grid = (unsigned)((n_strips + STRIPS_PER_BLOCK - 1) / STRIPS_PER_BLOCK);
        SDDMM_LAUNCH(c, k_union_tiles, strip_grid, WAVE * STRIPS_PER_BLOCK, c->d_rowptr,
                           c->d_col, c->sM, n_strips, c->d_ustrip_ntiles, c->d_ustrip_off,
                           c->d_tiles + c->n_tiles_natural, c->d_tile_cols + c->n_tiles_natural * 16);
        LAUNCH_CHECK(c);
    }
    const int64_t gathered_lo = c->n_tiles_natural + c->n_tiles_union + c->n_tiles_lead;
    if (c->n_tiles > gathered_lo) {
        SDDMM_LAUNCH(c, k_gathered_tiles, c->n_vstrips / 2, GATHERED_BLOCK, c->d_rowptr,
                           c->d_col, (const unsigned long long *)c->d_sorted_keys, c->n_cand, c->n_vstrips / 2,
                           c->d_vstrip_ntiles, c->d_vstrip_off, c->d_tiles + gathered_lo,
                           c->d_tile_cols + gathered_lo * 16, (int)c->n_tiles_lead, (const unsigned int *)c->d_cand_keys,
                           c->gathered_stride);
        LAUNCH_CHECK(c);
    }
    const int64_t complete = strips_complete ? c->n_tiles_natural : 0;     // (and the gathered ones)
    const int64_t of_strips = c->n_tiles_natural + c->n_tiles_union - complete;
    if (of_strips > 0) {
        SDDMM_LAUNCH(c, k_tile_rows, ((of_strips * 16 + 255) / 256), 256, c->d_rowptr, c->d_col, c->sM,
                     (const int32_t *)(c->d_tile_cols + complete * 16), c->d_tiles + complete, of_strips, c->nnz);
        LAUNCH_CHECK(c);
    }
    // windows of TILE_WINDOW descriptors: what a wavefront of the tile kernels takes.  As a batch
    // (one access per run of a row's entries, which costs reading the column indices) where the
    // tiles are sparsely filled; tile by tile from the descriptors' masks where they are nearly
    // full (measured: 92 entries per tile 12.8 -> 11.3 us as batches, 256 per tile 8.5 -> 9.4 us)
    c->n_windows = (c->n_tiles + TILE_WINDOW - 1) / TILE_WINDOW;
    {
        const int rc = plan_window_order(c);
        if (rc) return rc;
    }
    c->use_windows = !c->long_rows && c->nnz_tiles < (int64_t)env_int("SDDMM_WINDOW_FILL", 176) * c->n_tiles;
    // wavefronts of a tile launch: one per window, and one per two windows of a pair of gathered strips
    // (their descriptors come last and fill whole windows, an even number of them)
    c->n_win_single = c->n_windows;
    // (rows of up to 256 bytes: beyond that the second A panel and the kept products do not fit the registers; a launch in
    // another order than the storage order takes every window alone)
    if (c->use_windows && !c->use_win_order && c->n_tiles > gathered_lo && tile_pairs(c->ragged, c->dtype == SDDMM_F32, c->tile_steps) && env_int("SDDMM_PAIRS", 1) != 0)
        c->n_win_single = gathered_lo / TILE_WINDOW;
    c->n_tile_units = c->n_win_single + (c->n_windows - c->n_win_single + 1) / 2;
    if (!c->use_windows) {
        c->tiles_active = true;
        return SDDMM_OK;
    }
    if (c->n_windows > c->windows_cap) {
        dfree(c->d_windows);
        c->windows_cap = 0;
        ALLOC_TRY(c, c->d_windows, (size_t)c->n_windows * sizeof(TileWindow));
        c->windows_cap = c->n_windows;
    }
    SDDMM_LAUNCH(c, k_tile_windows, ((c->n_windows * 16 + 255) / 256), 256, (const int32_t *)c->d_vrows, c->sM,
                       c->nnz, (const TileDesc *)c->d_tiles, c->n_tiles, c->n_tiles_natural,
                       c->n_tiles_natural + c->n_tiles_union, c->n_tiles > gathered_lo ? gathered_lo : c->n_tiles,
                       c->d_windows, c->n_windows);
    LAUNCH_CHECK(c);
    c->tiles_active = true;
    return SDDMM_OK;
}

bool panel_valu_applicable(const sddmm_ctx *c) {
    const Shape s = shape_of(c);
    if (!s.whole() || s.LPN != 8 || !s.fullk || s.wide) return false;
    return s.unit == 0 ? s.UPL <= 2 : s.UPL == 1;
}

int panel_steps(const sddmm_ctx *c) { return c->long_rows ? LONG_STEPS : c->ragged ? ragged_steps(c) : panel_mfma_steps(c); }

int panel_item_columns(const sddmm_ctx *c) {
    const int64_t M = std::max(1, c->sM);
    const int columns = panel_columns(panel_steps(c), c->dtype != SDDMM_F32, std::max<int64_t>(1, M / PANEL_ROWS), c->nnz / M);
    return std::max<int>(WAVE, env_int("SDDMM_PANEL_SEG", columns));
}

// whether the 8-row panels are looked for, and by which kernel they would be computed
bool panel_path_applies(sddmm_ctx *c) {
    if (c->nnz == 0 || c->sM < PANEL_ROWS) return false;
    c->panel_mfma = (c->ragged || panel_mfma_steps(c) != 0) && env_int("SDDMM_PANEL_MFMA", 1) != 0;
    return c->panel_mfma || panel_valu_applicable(c);
}

// after the fetch_counters that follows plan_owners
int plan_panels_items(sddmm_ctx *c, int pseg) {
    if (!c->panels_flagged) return SDDMM_OK;
    const int64_t n_panels = (int64_t)c->sM / 8;
    c->n_panels = (int64_t)c->pc.n_panels;
    c->nnz_panels = (int64_t)c->pc.nnz_panels;
    c->n_panel_items = (int64_t)c->pc.panel_items;
    c->panel_columns = pseg;
    if (c->n_panel_items == 0) return SDDMM_OK;
    if (c->n_panel_items > c->panel_items_cap) {
        dfree(c->d_panel_items);
        ALLOC_TRY(c, c->d_panel_items, (size_t)c->n_panel_items * sizeof(RowItem));
        c->panel_items_cap = c->n_panel_items;
    }
    SDDMM_LAUNCH(c, k_panel_items, ((n_panels + 255) / 256), 256, c->d_rowptr,
                       n_panels, pseg, 0, (const unsigned int *)c->d_panel_counts, (const unsigned int *)c->d_panel_off,
                       c->d_panel_items);
    LAUNCH_CHECK(c);
    return SDDMM_OK;
}

int ensure_rowidx(sddmm_ctx *c) {
    if (c->d_rowidx) return SDDMM_OK;
    ALLOC_TRY(c, c->d_rowidx, (size_t)c->nnz * sizeof(int32_t));
    c->own_rowidx = true;
    if (c->sM > 0 && c->nnz > 0)
        SDDMM_LAUNCH(c, k_expand_rows, grid_for(c->sM, 256), 256, c->d_rowptr, c->sM,
                           c->d_rowidx, c->nnz);
    LAUNCH_CHECK(c);
    return SDDMM_OK;
}

// Work items of k_flat_blocks: the segments of the long rows (more than `seg` entries) block by block, and
// the entries between those rows.  Nothing is read back: the arrays are sized for the most items there
// can be, the launch reads the true numbers (and sddmm_plan fetches them for its grid).  Leaves use_blocks false when the device has no room.
// cut_long_rows false: the entries 64 at a time and nothing else (the way to take a sorted order whose long rows
// need no cutting).
int plan_blocks(sddmm_ctx *c, bool cut_long_rows) {
    const int64_t n_long = cut_long_rows ? (int64_t)c->pc.rows_long : 0, nb = ((int64_t)c->sM + SCAN_TILE - 1) / SCAN_TILE;
    if (cut_long_rows && (int64_t)c->raw.long_scanned != n_long)
        return fail(c, SDDMM_ERR_HIP, "internal: scan of the long rows disagrees with their number");
    const int least = row_blocks_least(c->use_order), most = row_blocks_most(c->use_order, (int)c->pc.max_len);
    const int64_t n_seg = n_long * most, n_gap = n_long + 1;
    const int64_t piece = c->seg, gap_piece = WAVE;
    block_items_max(c, cut_long_rows, &c->block_segments_max, &c->block_gaps_max);
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    };
    const size_t o_rows = take((size_t)n_long * 4);
    const size_t o_seg[3] = {take((size_t)n_seg * 4), take((size_t)n_seg * 4), take((size_t)n_seg * 4)};
    const size_t o_gap[3] = {take((size_t)n_gap * 4), take((size_t)n_gap * 4), take((size_t)n_gap * 4)};
    const size_t o_segments = take((size_t)c->block_segments_max * sizeof(RowItem));
    const size_t o_gaps = take((size_t)c->block_gaps_max * sizeof(RowItem));
    if (at > c->blocks_bytes) {
        dfree(c->d_blocks);
        c->blocks_bytes = 0;
        c->d_blocks = static_cast<char *>(spare_alloc(at));
        if (!c->d_blocks) return SDDMM_OK;
        c->blocks_bytes = at;
    }
    char *b = c->d_blocks;
    c->d_block_segments = (RowItem *)(b + o_segments);
    c->d_block_gaps = (RowItem *)(b + o_gaps);
    int32_t *rows = (int32_t *)(b + o_rows), *seg_start = (int32_t *)(b + o_seg[0]), *gap_start = (int32_t *)(b + o_gap[0]);
    unsigned int *seg_items = (unsigned int *)(b + o_seg[1]), *seg_off = (unsigned int *)(b + o_seg[2]);
    unsigned int *gap_items = (unsigned int *)(b + o_gap[1]), *gap_off = (unsigned int *)(b + o_gap[2]);
    if (n_long > 0) {
        SDDMM_LAUNCH(c, k_long_rows, nb, SCAN_BLOCK, c->d_rowptr, c->sM, c->ts, c->seg, (const unsigned int *)c->d_long_off, rows);
        SDDMM_LAUNCH(c, k_long_segments, grid_for(n_seg, 256), 256, c->d_rowptr, entry_cols(c), c->sN, (const int32_t *)rows,
                     (int)n_long, (int)piece, least, most, seg_start, seg_items);
    }
    SDDMM_LAUNCH(c, k_long_gaps, grid_for(n_gap, 256), 256, c->d_rowptr, (const int32_t *)rows, (int)n_long, (int)c->nnz,
                 (int)gap_piece, gap_start, gap_items);
    LAUNCH_CHECK(c);
    int rc = device_scan(c, seg_items, seg_off, n_seg, &c->d_pc->block_items[0]);
    if (rc) return rc;
    rc = device_scan(c, gap_items, gap_off, n_gap, &c->d_pc->block_items[1]);
    if (rc) return rc;
    rc = flush_scans(c);
    if (rc) return rc;
    if (n_long > 0)
        SDDMM_LAUNCH(c, k_range_items, grid_for(c->block_segments_max, 256), 256, c->d_rowptr, (const int32_t *)rows, (int)n_long,
                     (int)c->nnz, 0, (int)piece, (const int32_t *)seg_start, (const unsigned int *)seg_off, (int)n_seg,
                     (const unsigned long long *)&c->d_pc->block_items[0], c->d_block_segments);
    SDDMM_LAUNCH(c, k_range_items, grid_for(c->block_gaps_max, 256), 256, c->d_rowptr, (const int32_t *)rows, (int)n_long,
                 (int)c->nnz, 1, (int)gap_piece, (const int32_t *)gap_start, (const unsigned int *)gap_off, (int)n_gap,
                 (const unsigned long long *)&c->d_pc->block_items[1], c->d_block_gaps);
    LAUNCH_CHECK(c);
    c->use_blocks = true;
    return SDDMM_OK;
}

// Room for the partial products of the slices of K; false when the device does not have it (the launch
// then takes the plain flat kernel).  Kept until the context goes.
bool ensure_slice_workspace(sddmm_ctx *c) {
    const int64_t need = slice_workspace_floats(c);
    if (need <= c->part_floats) return true;
    dfree(c->d_part);
    c->d_part = static_cast<float *>(spare_alloc((size_t)need * sizeof(float)));
    c->part_floats = c->d_part ? need : 0;
    return c->d_part != nullptr;
}

// Entries in no order: sort them by row and column block and plan the flat launch over that order.  Leaves use_order
// false when the device has no room.
template <class Key>
int sort_order(sddmm_ctx *c, bool *done) {
    const size_t n = (size_t)c->nnz, column = (n * 4 + 255) & ~(size_t)255;
    int bits = 1;
    while (bits < 36 && ((int64_t)c->sM * COL_BLOCKS_ORDER - 1) >> bits) ++bits;
    if (c->nnz > c->order_cap) {
        dfree(c->d_order);
        c->order_cap = 0;
        c->d_order = static_cast<int32_t *>(spare_alloc(4 * column));
        if (!c->d_order) return SDDMM_OK;
        c->order_cap = c->nnz;
    }
    int32_t *part[4];
    for (int i = 0; i < 4; ++i) part[i] = c->d_order + i * (column / 4);
    // The sort works in the arrays of the order itself, 16 bytes per entry: the keys it ends with are overwritten by the
    // rows, its values by the columns, the other buffer of either takes the places and the dot products.  64-bit keys
    // (2^28 rows and more) have buffers of their own.
    const size_t key_bytes = sizeof(Key) == 4 ? 0 : (n * sizeof(Key) + 255) & ~(size_t)255;
    rocprim::double_buffer<Key> keys((Key *)part[0], (Key *)part[2]);
    rocprim::double_buffer<int32_t> from(part[1], part[3]);
    size_t need = 0;
    HIP_TRY(c, rocprim::radix_sort_pairs(nullptr, need, keys, from, n, 0, bits, c->stream));
    if (2 * key_bytes + need > c->sort_tmp_bytes) {
        dfree(c->d_sort_tmp);
        c->sort_tmp_bytes = 0;
        c->d_sort_tmp = spare_alloc(2 * key_bytes + need);
        if (!c->d_sort_tmp) return SDDMM_OK;
        c->sort_tmp_bytes = 2 * key_bytes + need;
    }
    char *b = (char *)c->d_sort_tmp;
    if (key_bytes) keys = rocprim::double_buffer<Key>((Key *)b, (Key *)(b + key_bytes));
    const int64_t grid = (c->nnz + 255) / 256;
    SDDMM_LAUNCH(c, k_order_keys<Key>, grid, 256, (const int32_t *)c->d_rowidx, (const int32_t *)c->d_col, c->nnz, c->sN,
                 keys.current(), from.current());
    LAUNCH_CHECK(c);
    HIP_TRY(c, rocprim::radix_sort_pairs(b + 2 * key_bytes, need, keys, from, n, 0, bits, c->stream));
    c->d_order_row = key_bytes ? part[0] : (int32_t *)keys.current();
    c->d_order_place = key_bytes ? part[2] : (int32_t *)keys.alternate();
    c->d_order_col = from.current();
    c->d_order_dots = (float *)from.alternate();
    SDDMM_LAUNCH(c, k_order_entries<Key>, grid, 256, (const Key *)keys.current(), (const int32_t *)from.current(),
                 (const int32_t *)c->d_col, c->nnz, c->d_order_row, c->d_order_col, c->d_order_place);
    SDDMM_LAUNCH(c, k_rowptr_from_sorted_coo, grid_for(c->nnz + 1, 256), 256, (const int32_t *)c->d_order_row, c->nnz, c->sM,
                 c->d_rowptr);
    LAUNCH_CHECK(c);
    *done = true;
    return SDDMM_OK;
}

int plan_order(sddmm_ctx *c) {
    bool done = false;
    int rc = (int64_t)c->sM * COL_BLOCKS_ORDER <= ((int64_t)1 << 32) ? sort_order<uint32_t>(c, &done) : sort_order<uint64_t>(c, &done);
    if (rc || !done) return rc;
    rc = begin_ownership(c, true);
    if (rc) return rc;
    // row statistics of the sorted entries; no row has another owner
    c->ts = std::max(1, env_int("SDDMM_TS", 24));
    c->seg = std::max(WAVE, env_int("SDDMM_SEG", 256));
    HIP_TRY(c, hipMemsetAsync(&c->d_pc->k[K_ROWS_NONEMPTY][0], 0, sizeof(unsigned long long) * SPREAD, c->stream));
    SDDMM_LAUNCH(c, k_check_rowptr, grid_for(c->sM, 256), 256, (const int32_t *)c->d_rowptr, c->sM, c->nnz, c->d_pc);
    LAUNCH_CHECK(c);
    rc = classify_rows_count(c);
    if (rc) return rc;
    rc = fetch_counters(c);
    if (c->sort_tmp_bytes > ((size_t)16 << 20)) {          // (64-bit keys; the device is done with them)
        dfree(c->d_sort_tmp);
        c->sort_tmp_bytes = 0;
    }
    if (rc) return rc;
    if (c->pc.bad_pattern) return fail(c, SDDMM_ERR_HIP, "internal: row pointer built from sorted entries is inconsistent");
    const double avg_len = c->pc.rows_nonempty ? (double)c->nnz / (double)c->pc.rows_nonempty : 0.0;
    c->pc.rows_nonempty = 0;                               // (reported as unknown without a row pointer of the caller's order)
    c->use_order = true;
    // (the other kernel here is the flat one, whatever the rows hold)
    c->use_slices = slices_pay(c, std::min(avg_len, 31.0)) && ensure_slice_workspace(c);
    if (!c->use_slices) {
        // (rows beyond the register layout came here for the slices alone: without their workspace, the plain kernel)
        if (shape_of(c).LPN != 0) {
            rc = plan_blocks(c, blocks_pay(c));
            if (rc) return rc;
        }
        c->use_order = c->use_blocks;
    }
    return SDDMM_OK;
}

// Clears P and the counters of a new pattern.
int clear_pattern(sddmm_ctx *c, int64_t nnz) {
    SDDMM_LAUNCH(c, k_clear_pattern, grid_capped(nnz, 1024, 4096), 256, c->dP, nnz, (unsigned int *)c->d_pc);
    LAUNCH_CHECK(c);
    return SDDMM_OK;
}

// Checks the column indices and samples how near neighbours are to each other.
void check_columns(sddmm_ctx *c) {
    SDDMM_LAUNCH(c, k_check_index, grid_capped((c->nnz + 3) / 4, 256, 4096), 256, (const int32_t *)c->d_col, c->nnz, c->sN, 1, c->d_pc);
}
double columns_near(const PlanCounters &pc) { return pc.col_pairs ? (double)pc.col_near / (double)pc.col_pairs : 1.0; }

// Validate the device-resident CSR and gather row statistics.
int validate_csr(sddmm_ctx *c) {
    if (c->sM > 0)
        SDDMM_LAUNCH(c, k_check_rowptr, grid_for(c->sM, 256), 256, c->d_rowptr, c->sM,
                           c->nnz, c->d_pc);
    // (walks col[0..nnz) only behind a valid row pointer)
    if (c->nnz > 0)
        check_columns(c);
    LAUNCH_CHECK(c);
    const int rc = fetch_counters(c);
    if (rc) return rc;
    if (c->pc.bad_pattern & BAD_POINTER) return fail(c, SDDMM_ERR_PATTERN, "rowptr is not a valid CSR row pointer array");
    if (c->pc.bad_pattern) return fail(c, SDDMM_ERR_PATTERN, "column index outside [0,N)");
    c->col_near = columns_near(c->pc);
    return SDDMM_OK;
}

int check_dims(sddmm_ctx *c, int M, int N, int64_t nnz) {
    if (M < 0 || N < 0 || nnz < 0) return fail(c, SDDMM_ERR_INVALID, "negative dimension");
    if (nnz > 0 && (M == 0 || N == 0)) return fail(c, SDDMM_ERR_INVALID, "entries in an empty matrix");
    // positions are 32-bit like the reference's row pointers; the kernels look up to a few chunks
    // past a position before clamping, so the last 64 Ki values stay unused
    if (nnz > (int64_t)INT32_MAX - 65536) return fail(c, SDDMM_ERR_INVALID, "nnz exceeds 32-bit row pointers");
    return SDDMM_OK;
}

int enqueue_run(sddmm_ctx *c) {
    c->launches = 0;
    if (c->nnz == 0) return SDDMM_OK;
    c->launches = 1;
    switch (c->strategy) {
        case SDDMM_AUTO:
        case SDDMM_MFMA_TILE:
        case SDDMM_LDS_TILED: {
            // (a second stream for the first of these independent kernels was measured:
            // the fork/join events cost more than the overlap returns, 33 us against 23 us
            // on the mixed-density shape)
            c->launches = 0;
            const bool tiles = c->tiles_active && c->n_tiles > 0, rows = c->rows_short > 0 || c->n_items > 0;
            bool fused = false;
            if (tiles && rows && !c->long_rows && env_int("SDDMM_FUSE", 1) != 0) fused = launch_auto_with_tiles(c);
            if (fused) ++c->launches;
            if (tiles && !fused) {
                if (c->long_rows) launch_long_tiles(c);
                else launch_tiles(c);
                ++c->launches;
            }
            if (c->n_panel_items > 0) {
                if (c->long_rows) c->launches += launch_long_panels(c);
                else { launch_panels(c); ++c->launches; }
            }
            if (rows && !fused) { launch_auto(c); ++c->launches; }
            break;
        }
        case SDDMM_FLAT:
            if (c->use_slices) c->launches = launch_flat_sliced(c);
            else if (c->use_blocks) {
                if (launch_flat_blocks(c) == 0) return fail(c, SDDMM_ERR_UNSUPPORTED, "internal: no column blocks for this row layout");
            } else launch_flat(c);
            if (c->use_order) { launch_unsort(c); ++c->launches; }
            break;
        case SDDMM_ROW_WAVE: launch_row_wave(c, nullptr, c->sM); break;
        case SDDMM_SHORT_ROWS:
            launch_short_rows(c, INT32_MAX, rows_per_wave(c->sM ? (double)c->nnz / c->sM : 0.0));
            break;
        case SDDMM_EXACT:
            if (c->dtype == SDDMM_BF16)
                SDDMM_LAUNCH(c, k_exact<DT_BF16>, grid_for(c->nnz, BLOCK), BLOCK, c->dA,
                                   c->dB, c->K, c->d_rowidx, c->d_col, c->d_sval, c->dP, c->nnz);
            else if (c->dtype == SDDMM_F16)
                SDDMM_LAUNCH(c, k_exact<DT_F16>, grid_for(c->nnz, BLOCK), BLOCK, c->dA,
                                   c->dB, c->K, c->d_rowidx, c->d_col, c->d_sval, c->dP, c->nnz);
            else
                SDDMM_LAUNCH(c, k_exact<DT_F32>, grid_for(c->nnz, BLOCK), BLOCK, c->dA,
                                   c->dB, c->K, c->d_rowidx, c->d_col, c->d_sval, c->dP, c->nnz);
            break;
        default: return fail(c, SDDMM_ERR_STATE, "no kernel for strategy %d", c->strategy);
    }
    LAUNCH_CHECK(c);
    c->stats.kernels_launched = c->launches;
    return SDDMM_OK;
}

int do_plan(sddmm_ctx *c, int strategy) {
    // the plan state is rewritten in place: a plan that fails half way must not leave the
    // previous one looking valid (its items exclude rows that tiles and panels owned)
    c->planned = false;
    c->n_scan_jobs = 0;
    c->use_slices = c->use_blocks = c->use_order = false;
    c->fused_items_valid = false;    // they leave out the rows of this plan's panels
    c->fused_panels_valid = false;
    int resolved = strategy;
    const bool csr_ok = c->have_rowptr;
    // without a row pointer (unsorted COO) only the flat kernels apply
    if (strategy == SDDMM_AUTO && !csr_ok) resolved = SDDMM_FLAT;
    switch (resolved) {
        case SDDMM_AUTO:
        case SDDMM_MFMA_TILE:
        case SDDMM_LDS_TILED: {
            // Row ownership in this order: well-filled 16-row strips go to the MFMA tile
            // path, then 8-row panels with a common column list to the panel kernel, the
            // rest is split by length.  MFMA_TILE takes every sorted strip and no panel,
            // LDS_TILED every panel and no strip; AUTO applies the thresholds.
            if (!csr_ok) return fail(c, SDDMM_ERR_UNSUPPORTED, "strategy %d needs row-sorted entries", resolved);
            // entries per 16x16 tile from which the tile kernel beats the gather kernels,
            // measured on banded matrices of varying fill: 74 at 128-byte rows, 50 at 256
            // and 512 bytes; 64-byte rows keep the older, conservative figure
            const size_t row_bytes = (size_t)c->K * elem_size(c->dtype);
            const int tile_fill = std::max(1, env_int("SDDMM_TILE_FILL", row_bytes <= 64 ? 96 : row_bytes <= 128 ? 80 : 56));
            c->tile_steps = 0;
            c->long_rows = resolved == SDDMM_AUTO && long_pays(c);
            c->ragged = c->long_rows || (resolved == SDDMM_AUTO && ragged_pays(c));
            const bool gathered = resolved == SDDMM_AUTO && env_int("SDDMM_GATHERED", 1) != 0 && (!c->ragged || ragged_gathers(c));
            const bool tiles = resolved != SDDMM_LDS_TILED && tile_path_applies(c);
            OwnRules rules{};
            // 16-row strips must not take what the panel kernel does better (8x8-block rows reach ~80 entries per tile, in
            // narrow bands 190); the strips gathered after the panels use the measured break-even
            if (tiles) rules.strip_fill = resolved == SDDMM_MFMA_TILE ? 1 : std::max(96, tile_fill);
            if (resolved != SDDMM_MFMA_TILE && panel_path_applies(c)) {
                rules.panel_min = resolved == SDDMM_LDS_TILED ? 1 : std::max(1, env_int("SDDMM_PANEL_MIN", 16));
                if (c->panel_mfma) rules.panel_min = std::max(rules.panel_min, 4);       // 16-byte S/P accesses stay inside a row
            }
            if (tiles && resolved == SDDMM_AUTO && env_int("SDDMM_UNION", 1) != 0)
                rules.union_fill = std::max(1, env_int("SDDMM_UNION_FILL", tile_fill));
            if (tiles && gathered && c->sM >= 2) rules.cand_min = std::max(16, env_int("SDDMM_GATHERED_MIN", 64));
            const int pseg = panel_item_columns(c);
            rules.pseg = pseg;
            rules.panels_below = PANELS_AMONG_PANELS;                // (settled below)
            // the rows nobody owns so far are classified in the same launch: most matrices have
            // no gathered strips, and their plan then waits for the device once
            c->ts = rules.ts = std::max(1, env_int("SDDMM_TS", 24));
            // segment items of 256 entries: a wavefront walks its item chunk by chunk, one dependent
            // round trip each, so a few long items set the duration of a short launch (eight rows of
            // 554 entries as single items: 17.5 us on the mixed-density shape, 14.6 us in pieces of
            // 256); on a matrix of 36 M entries pieces of 128..2048 differ by 3 %
            c->seg = rules.seg = std::max(WAVE, env_int("SDDMM_SEG", 256));
            const bool looked = c->sM > 0 && (rules.strip_fill || rules.panel_min || rules.union_fill || rules.cand_min);
            int rc = begin_ownership(c, !looked);
            if (rc) return rc;
            c->panels_flagged = false;
            rc = looked ? plan_owners(c, rules) : classify_rows_count(c);
            if (rc) return rc;
            rc = fetch_counters(c);
            if (rc) return rc;
            // Strips that are two panels each: all of them go the way that their average says.  (Launch us, all strips / some /
            // all panels: 2 000 rows in a band, 155 entries per tile, K = 32 5.2 / 8.6 / 4.2, K = 512 bf16 8.9 / 13.9 / 10.4.)
            if (c->pc.either_tiles) {
                const uint64_t either = c->pc.nnz_either_strip + c->pc.nnz_either_panels;
                const bool among_panels = c->pc.nnz_panels - c->pc.nnz_either_panels > either / 16;
                const bool half_width = c->dtype != SDDMM_F32;
                const int line = among_panels ? PANELS_AMONG_PANELS
                               : c->long_rows ? long_panels_below(half_width, c->nnz)
                                              : panels_below(panel_steps(c), half_width, c->sM / PANEL_ROWS, c->nnz);
                const bool to_panels = either < (uint64_t)line * c->pc.either_tiles;
                if (to_panels ? c->pc.nnz_either_strip : c->pc.nnz_either_panels) {
                    rc = settle_owners(c, to_panels, pseg);
                    if (!rc) rc = fetch_counters(c);
                    if (rc) return rc;
                }
            }
            rc = take_tile_counts(c);
            if (rc) return rc;
            // The kernels of the other rows take a row of more than 1 KiB an entry at a time: the matrix goes in slices as a
            // whole where strips and panels do not own nearly all of it.
            if ((c->long_rows && (int64_t)(c->pc.nnz_tiles + c->pc.nnz_utiles + c->pc.nnz_panels) < c->nnz - c->nnz / 16) || too_few_panels(c)) {
                c->ragged = c->long_rows = c->panels_flagged = false;
                c->tile_steps = 0;
                if (c->pc.nnz_tiles + c->pc.nnz_utiles + c->pc.nnz_panels) {        // (else the rows are classified as if not looked at)
                    rc = begin_ownership(c, true);
                    if (!rc) rc = classify_rows_count(c);
                    if (!rc) rc = fetch_counters(c);
                    if (rc) return rc;
                }
            }
            rc = plan_panels_items(c, pseg);
            if (rc) return rc;
            if (gathered) {
                bool launched = false;
                // (gathered strips come in pairs that share every B tile they load: a tile pays for
                // itself at three quarters of the entries a tile of a lone strip needs)
                rc = plan_gathered_count(c, std::max(1, env_int("SDDMM_GATHERED_FILL", tile_fill * 3 / 4)), &launched);
                if (rc) return rc;
                if (launched) {
                    // gathered strips may have taken rows: the row classes without them, one more read-back
                    rc = classify_rows_scan(c);
                    if (rc) return rc;
                    rc = fetch_counters(c);
                    if (rc) return rc;
                    rc = plan_gathered_take(c);
                    if (rc) return rc;
                }
            }
            if (resolved != SDDMM_LDS_TILED) {
                rc = plan_tiles_fill(c);
                if (rc) return rc;
            }
            // A matrix whose rows are short on average (fewer than 32 entries per non-empty
            // row), with no strip or panel taken, is a flat stream of entries: the flat
            // kernel (row index per entry, perfectly balanced) measured 6 % faster there than
            // the row split (power-law shape, K=32: 634 us against 672 us).
            const double avg_len = c->pc.rows_nonempty ? (double)c->nnz / (double)c->pc.rows_nonempty : 0.0;
            const bool only_rows = resolved == SDDMM_AUTO && c->n_tiles == 0 && c->n_panel_items == 0;
            const bool sliced = only_rows && slices_pay(c, avg_len) && ensure_slice_workspace(c);
            const bool flat = only_rows && (sliced || avg_len < (double)env_int("SDDMM_FLAT_AVG", 32));
            if (flat) {                              // (which has no use for items, or for the entry list of the short rows)
                c->n_items = c->n_short_list = c->rows_short = 0;
                c->use_short_list = false;
                rc = ensure_rowidx(c);
                if (rc) return rc;
                resolved = SDDMM_FLAT;
                c->use_slices = sliced;
                if (!sliced && blocks_pay(c)) {
                    rc = plan_blocks(c, true);
                    if (rc) return rc;
                }
            } else {
                rc = classify_rows_items(c);
                if (rc) return rc;
            }
            break;
        }
        case SDDMM_FLAT:
        case SDDMM_EXACT: {
            int rc = ensure_rowidx(c);
            if (rc) return rc;
            // (asked for by name, FLAT stays the plain kernel; AUTO on unsorted entries gets here too)
            if (strategy == SDDMM_AUTO && c->nnz > 0) {
                if (order_pays(c)) rc = plan_order(c);
                if (rc) return rc;
                if (!c->use_blocks && !c->use_slices) c->use_slices = slices_pay(c, 1.0) && ensure_slice_workspace(c);
            }
            break;
        }
        case SDDMM_ROW_WAVE:
        case SDDMM_SHORT_ROWS:
            if (!csr_ok) return fail(c, SDDMM_ERR_UNSUPPORTED, "strategy %d needs row-sorted entries", resolved);
            break;
        default: return fail(c, SDDMM_ERR_INVALID, "unknown strategy %d", strategy);
    }
    c->requested = strategy;
    c->strategy = resolved;
    c->planned = true;
    return SDDMM_OK;
}

// Device code of every kernel that enqueue_run may launch under this plan.
int load_planned(sddmm_ctx *c) {
    switch (c->strategy) {
        case SDDMM_FLAT: HIP_TRY(c, load_flat()); break;
        case SDDMM_ROW_WAVE:
        case SDDMM_SHORT_ROWS: HIP_TRY(c, load_rows()); break;
        case SDDMM_EXACT: break;                           // (k_exact comes with the plan kernels)
        default:
            if (c->tiles_active && c->n_tiles > 0) HIP_TRY(c, load_tiles(c->ragged));
            if (c->n_panel_items > 0) HIP_TRY(c, load_panels(c->ragged));
            if (c->rows_short > 0 || c->n_items > 0) HIP_TRY(c, load_auto());
    }
    return SDDMM_OK;
}

void fill_model(sddmm_ctx *c) {
    sddmm_stats &s = c->stats;
    s.strategy_used = c->strategy;
    s.nnz = c->nnz;
    s.rows_nonempty = (int64_t)c->pc.rows_nonempty;
    if (c->strategy == SDDMM_AUTO || c->strategy == SDDMM_MFMA_TILE || c->strategy == SDDMM_LDS_TILED) {
        s.mfma_tiles = c->tiles_active ? c->n_tiles : 0;
        s.nnz_mfma = c->tiles_active ? c->nnz_tiles : 0;
        s.panels = c->n_panels;
        s.nnz_panel = c->nnz_panels;
        s.rows_short = (int64_t)c->pc.rows_short; s.rows_medium = (int64_t)c->pc.rows_medium;
        s.rows_long = (int64_t)c->pc.rows_long;
        s.nnz_short = (int64_t)c->pc.nnz_short; s.nnz_medium = (int64_t)c->pc.nnz_medium;
        s.nnz_long = (int64_t)c->pc.nnz_long;
    }
    const double e = (double)elem_size(c->dtype);
    s.flops = 2.0 * (double)c->nnz * (double)c->K;
    s.bytes_gathered = 4.0 * ((double)c->sM + 1.0) + 12.0 * (double)c->nnz +
                       e * (double)c->K * (double)s.rows_nonempty + e * (double)c->K * (double)c->nnz;
}

}  // namespace

// ===========================================================================
extern "C" {

const char *sddmm_version(void) { return "sddmm_amd 0.1 (gfx950, wave64)"; }

const char *sddmm_strerror(int code) {
    switch (code) {
        case SDDMM_OK: return "ok";
        case SDDMM_ERR_INVALID: return "invalid argument";
        case SDDMM_ERR_NULL: return "null pointer";
        case SDDMM_ERR_STATE: return "operands or plan missing";
        case SDDMM_ERR_ALLOC: return "allocation failed";
        case SDDMM_ERR_HIP: return "HIP runtime error";
        case SDDMM_ERR_UNSUPPORTED: return "strategy not applicable";
        case SDDMM_ERR_NO_DEVICE: return "no usable HIP device";
        case SDDMM_ERR_PATTERN: return "malformed sparse structure";
        case SDDMM_ERR_TOO_LARGE:
            return "more stored entries than the static scratch buffer of sddmm_launch_noalloc holds "
                   "(SDDMM_NOALLOC_MAX_NNZ)";
        default: return "unknown error";
    }
}

const char *sddmm_last_error(const sddmm_ctx *ctx) { return ctx ? ctx->err : ""; }

int sddmm_create(sddmm_ctx **out, int device) {
    if (!out) return SDDMM_ERR_NULL;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return SDDMM_ERR_NO_DEVICE;
    if (device < 0 || device >= count) return SDDMM_ERR_INVALID;
    if (hipSetDevice(device) != hipSuccess) return SDDMM_ERR_NO_DEVICE;
    sddmm_ctx *c = new (std::nothrow) sddmm_ctx();
    if (!c) return SDDMM_ERR_ALLOC;
    c->device = device;
    if (take_parts(&c->parts, device, sizeof(DevCounters)) != hipSuccess) {
        delete c;
        return SDDMM_ERR_HIP;
    }
    c->stream = c->own_stream = c->parts.stream;
    c->ev0 = c->parts.ev0; c->ev1 = c->parts.ev1;
    c->d_pc = (DevCounters *)c->parts.counters;
    c->h_pc = (DevCounters *)c->parts.host_counters;
    *out = c;
    return SDDMM_OK;
}

int sddmm_set_stream(sddmm_ctx *c, void *stream, int lent) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    // nothing of this context may still be in flight on the stream it leaves
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    c->lent_stream = lent != 0;
    c->stream = c->lent_stream ? (hipStream_t)stream : c->own_stream;
    return SDDMM_OK;
}

int sddmm_get_stream(const sddmm_ctx *c, void **stream) {
    if (!c || !stream) return SDDMM_ERR_NULL;
    *stream = (void *)c->stream;
    return SDDMM_OK;
}

void sddmm_destroy(sddmm_ctx *c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    const bool idle = pool_wait();
    release_dense(c, idle);
    release_sparse(c, idle);
    dfree(c->dO, idle);
    dfree(c->d_part, idle);
    dfree(c->d_blocks, idle);
    give_parts(c->parts, idle);
    delete c;
}

int sddmm_trim(void) {
    pool_trim();
    return SDDMM_OK;
}

static int set_dense_common(sddmm_ctx *c, int M, int N, int K, const void *A, const void *B, int dtype,
                            bool on_device) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    if (M < 0 || N < 0 || K < 1) return fail(c, SDDMM_ERR_INVALID, "need M,N >= 0 and K >= 1 (got %d,%d,%d)", M, N, K);
    if (dtype != SDDMM_F32 && dtype != SDDMM_BF16 && dtype != SDDMM_F16)
        return fail(c, SDDMM_ERR_INVALID, "unknown dtype %d", dtype);
    if (dtype != SDDMM_F32 && K % 8) return fail(c, SDDMM_ERR_INVALID, "16-bit operands need K %% 8 == 0 (got %d)", K);
    if ((M > 0 && !A) || (N > 0 && !B)) return fail(c, SDDMM_ERR_NULL, "A or B is NULL");
    // a plan depends on the pattern and on the shape and type of the dense operands, not on their
    // values: new A and B of the same shape (the next iteration of a solver) keep it
    const bool keep_plan = c->planned && c->have_dense && c->M == M && c->N == N && c->K == K && c->dtype == dtype;
    release_dense(c);
    const size_t es = elem_size(dtype);
    const size_t a_bytes = (size_t)M * K * es, b_bytes = (size_t)N * K * es;
    if (on_device) {
        if (((uintptr_t)A | (uintptr_t)B) & 15) return fail(c, SDDMM_ERR_INVALID, "device A/B must be 16-byte aligned");
        c->dA = const_cast<void *>(A);
        c->dB = const_cast<void *>(B);
        c->own_dense = false;
    } else {
        c->own_dense = true;
        ALLOC_TRY(c, c->dA, a_bytes);
        ALLOC_TRY(c, c->dB, b_bytes);
        if (a_bytes) HIP_TRY(c, hipMemcpyAsync(c->dA, A, a_bytes, hipMemcpyHostToDevice, c->stream));
        if (b_bytes) HIP_TRY(c, hipMemcpyAsync(c->dB, B, b_bytes, hipMemcpyHostToDevice, c->stream));
        HIP_TRY(c, hipStreamSynchronize(c->stream));
    }
    c->M = M; c->N = N; c->K = K; c->dtype = dtype;
    c->have_dense = true;
    c->planned = keep_plan;
    return SDDMM_OK;
}

int sddmm_set_dense(sddmm_ctx *c, int M, int N, int K, const void *A, const void *B, int dtype) {
    return set_dense_common(c, M, N, K, A, B, dtype, false);
}
int sddmm_set_dense_device(sddmm_ctx *c, int M, int N, int K, const void *dA, const void *dB, int dtype) {
    return set_dense_common(c, M, N, K, dA, dB, dtype, true);
}

int sddmm_set_csr(sddmm_ctx *c, int M, int N, int64_t nnz, const int32_t *rowptr, const int32_t *col,
                  const float *sval) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_dims(c, M, N, nnz);
    if (rc) return rc;
    if (!rowptr || (nnz > 0 && (!col || !sval))) return fail(c, SDDMM_ERR_NULL, "rowptr, col or values is NULL");
    release_sparse(c);
    c->own_sparse = c->own_rowptr = true;
    ALLOC_TRY(c, c->d_rowptr, (size_t)(M + 1) * sizeof(int32_t));
    ALLOC_TRY(c, c->d_col, (size_t)nnz * sizeof(int32_t));
    ALLOC_TRY(c, c->d_sval, (size_t)nnz * sizeof(float));
    ALLOC_TRY(c, c->dP, (size_t)nnz * sizeof(float));
    HIP_TRY(c, hipMemcpyAsync(c->d_rowptr, rowptr, (size_t)(M + 1) * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    if (nnz) {
        HIP_TRY(c, hipMemcpyAsync(c->d_col, col, (size_t)nnz * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
        HIP_TRY(c, hipMemcpyAsync(c->d_sval, sval, (size_t)nnz * sizeof(float), hipMemcpyHostToDevice, c->stream));
    }
    rc = clear_pattern(c, nnz);
    if (rc) return rc;
    c->sM = M; c->sN = N; c->nnz = nnz;
    rc = validate_csr(c);
    if (rc) { release_sparse(c); return rc; }
    c->have_sparse = c->have_rowptr = true;
    return SDDMM_OK;
}

int sddmm_set_csr_device(sddmm_ctx *c, int M, int N, int64_t nnz, const int32_t *d_rowptr, const int32_t *d_col,
                         const float *d_sval) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_dims(c, M, N, nnz);
    if (rc) return rc;
    if (!d_rowptr || (nnz > 0 && (!d_col || !d_sval))) return fail(c, SDDMM_ERR_NULL, "rowptr, col or values is NULL");
    release_sparse(c);
    c->own_sparse = c->own_rowptr = false;
    c->d_rowptr = const_cast<int32_t *>(d_rowptr);
    c->d_col = const_cast<int32_t *>(d_col);
    c->d_sval = const_cast<float *>(d_sval);
    ALLOC_TRY(c, c->dP, (size_t)nnz * sizeof(float));
    rc = clear_pattern(c, nnz);
    if (rc) return rc;
    c->sM = M; c->sN = N; c->nnz = nnz;
    rc = validate_csr(c);
    if (rc) { release_sparse(c); return rc; }
    c->have_sparse = c->have_rowptr = true;
    return SDDMM_OK;
}

static int set_coo_common(sddmm_ctx *c, int M, int N, int64_t nnz, const int32_t *row, const int32_t *col,
                          const float *sval, bool on_device) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_dims(c, M, N, nnz);
    if (rc) return rc;
    if (nnz > 0 && (!row || !col || !sval)) return fail(c, SDDMM_ERR_NULL, "row, col or values is NULL");
    release_sparse(c);
    c->own_sparse = c->own_rowidx = !on_device;
    c->own_rowptr = true;                 // the row pointer is always built here
    c->from_coo = true;
    if (on_device) {
        c->d_rowidx = const_cast<int32_t *>(row);
        c->d_col = const_cast<int32_t *>(col);
        c->d_sval = const_cast<float *>(sval);
    } else {
        ALLOC_TRY(c, c->d_rowidx, (size_t)nnz * sizeof(int32_t));
        ALLOC_TRY(c, c->d_col, (size_t)nnz * sizeof(int32_t));
        ALLOC_TRY(c, c->d_sval, (size_t)nnz * sizeof(float));
    }
    ALLOC_TRY(c, c->dP, (size_t)nnz * sizeof(float));
    ALLOC_TRY(c, c->d_rowptr, (size_t)(M + 1) * sizeof(int32_t));
    c->sM = M; c->sN = N; c->nnz = nnz;
    rc = clear_pattern(c, nnz);
    if (rc) return rc;
    if (nnz) {
        if (!on_device) {
            HIP_TRY(c, hipMemcpyAsync(c->d_rowidx, row, (size_t)nnz * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
            HIP_TRY(c, hipMemcpyAsync(c->d_col, col, (size_t)nnz * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
            HIP_TRY(c, hipMemcpyAsync(c->d_sval, sval, (size_t)nnz * sizeof(float), hipMemcpyHostToDevice, c->stream));
        }
        SDDMM_LAUNCH(c, k_check_index, grid_capped((nnz + 3) / 4, 256, 4096), 256, (const int32_t *)c->d_rowidx, nnz, M, 0, c->d_pc);
        check_columns(c);
        SDDMM_LAUNCH(c, k_check_coo_sorted, grid_capped(nnz, 256, 1024), 256, (const int32_t *)c->d_rowidx,
                           (const int32_t *)c->d_col, nnz, c->d_pc);
        LAUNCH_CHECK(c);
    }
    rc = fetch_counters(c);
    if (rc) { release_sparse(c); return rc; }
    if (c->pc.bad_pattern) {
        release_sparse(c);
        return fail(c, SDDMM_ERR_PATTERN, "COO row or column index out of range");
    }
    const bool sorted = c->pc.coo_unsorted == 0;
    c->coo_jumps = (int64_t)c->pc.coo_jumps;
    c->col_near = columns_near(c->pc);                     // (of entries in no order: of no use, they have no rows to look at)
    if (sorted) {
        SDDMM_LAUNCH(c, k_rowptr_from_sorted_coo, grid_for(nnz + 1, 256), 256,
                           c->d_rowidx, nnz, M, c->d_rowptr);
        LAUNCH_CHECK(c);
        HIP_TRY(c, hipMemsetAsync(c->d_pc, 0, sizeof(DevCounters), c->stream));
        if (M > 0)
            SDDMM_LAUNCH(c, k_check_rowptr, grid_for(M, 256), 256, c->d_rowptr, M, nnz,
                               c->d_pc);
        LAUNCH_CHECK(c);
        rc = fetch_counters(c);
        if (rc) { release_sparse(c); return rc; }
        if (c->pc.bad_pattern) {
            release_sparse(c);
            return fail(c, SDDMM_ERR_HIP, "internal: row pointer built from COO is inconsistent");
        }
        c->have_rowptr = true;
    } else {
        // row statistics are not available without a row pointer; count distinct rows as unknown
        c->have_rowptr = false;
        c->pc.rows_nonempty = 0;
    }
    c->have_sparse = true;
    return SDDMM_OK;
}

int sddmm_set_coo(sddmm_ctx *c, int M, int N, int64_t nnz, const int32_t *row, const int32_t *col,
                  const float *sval) {
    return set_coo_common(c, M, N, nnz, row, col, sval, false);
}
int sddmm_set_coo_device(sddmm_ctx *c, int M, int N, int64_t nnz, const int32_t *d_row, const int32_t *d_col,
                         const float *d_sval) {
    return set_coo_common(c, M, N, nnz, d_row, d_col, d_sval, true);
}

int sddmm_update_values(sddmm_ctx *c, const float *sval) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    if (!c->have_sparse) return fail(c, SDDMM_ERR_STATE, "no sparse operand set");
    if (!c->own_sparse) return fail(c, SDDMM_ERR_STATE, "values are caller-owned device memory");
    if (c->nnz > 0 && !sval) return fail(c, SDDMM_ERR_NULL, "values is NULL");
    if (c->nnz) HIP_TRY(c, hipMemcpyAsync(c->d_sval, sval, (size_t)c->nnz * sizeof(float), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return SDDMM_OK;
}

static int check_ready(sddmm_ctx *c) {
    if (!c->have_dense || !c->have_sparse) return fail(c, SDDMM_ERR_STATE, "set dense and sparse operands first");
    if (c->sM > c->M || c->sN > c->N)
        return fail(c, SDDMM_ERR_INVALID, "S is %dx%d but A has %d rows and B has %d rows", c->sM, c->sN, c->M, c->N);
    return SDDMM_OK;
}

int sddmm_plan(sddmm_ctx *c, int strategy) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_ready(c);
    if (rc) return rc;
    HIP_TRY(c, hipEventRecord(c->ev0, c->stream));
    rc = do_plan(c, strategy);
    if (rc) return rc;
    if (c->use_blocks)
        HIP_TRY(c, hipMemcpyAsync(c->h_pc->block_items, c->d_pc->block_items, sizeof(c->h_pc->block_items), hipMemcpyDeviceToHost,
                                  c->stream));
    HIP_TRY(c, hipEventRecord(c->ev1, c->stream));
    HIP_TRY(c, hipEventSynchronize(c->ev1));
    if (c->use_blocks) {
        // A workgroup without an item costs the launch 0.2 ns (of 92 000 more than needed, 2.6 M rows K = 32: 530 us, 521 without)
        c->block_segments_max = (int64_t)c->h_pc->block_items[0];
        c->block_gaps_max = (int64_t)c->h_pc->block_items[1];
    }
    float ms = 0.f;
    HIP_TRY(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->stats = sddmm_stats{};
    c->stats.plan_ms = ms;
    fill_model(c);
    if (c->nnz > 0) {
        rc = load_planned(c);
        if (rc) c->planned = false;
    }
    return rc;
}

int sddmm_launch(sddmm_ctx *c) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_ready(c);
    if (rc) return rc;
    if (!c->planned) {
        // operands were replaced since the last plan: plan again as last asked (AUTO on a new context)
        rc = sddmm_plan(c, c->requested);
        if (rc) return rc;
    }
    return enqueue_run(c);
}

int sddmm_synchronize(sddmm_ctx *c) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return SDDMM_OK;
}

int sddmm_run(sddmm_ctx *c) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_ready(c);
    if (rc) return rc;
    if (!c->planned) {
        // operands were replaced since the last plan: plan again as last asked (AUTO on a new context)
        rc = sddmm_plan(c, c->requested);
        if (rc) return rc;
    }
    HIP_TRY(c, hipEventRecord(c->ev0, c->stream));
    rc = enqueue_run(c);
    if (rc) return rc;
    HIP_TRY(c, hipEventRecord(c->ev1, c->stream));
    HIP_TRY(c, hipEventSynchronize(c->ev1));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    float ms = 0.f;
    HIP_TRY(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->stats.run_ms = ms;
    c->stats.kernels_launched = c->launches;
    return SDDMM_OK;
}

// Room for the partial output rows of the pieces of at most seg entries (K floats each); false when the device does not
// have it.  256 entries a piece can take K / 64 bytes per stored entry: beyond SDDMM_FUSED_PARTS_MAX MiB (1 024 by default)
// they have to be longer.
static bool fused_parts(sddmm_ctx *c, int seg) {
    const int64_t need = c->n_fused_pieces * c->K;
    const int64_t most = ((int64_t)env_int("SDDMM_FUSED_PARTS_MAX", 1024) << 20) / (int64_t)sizeof(float);
    if (seg < 1024 && need > most && !getenv("SDDMM_FUSED_SEG")) return false;
    if (need <= c->fused_part_floats) return true;
    dfree(c->d_fused_parts);
    c->d_fused_parts = static_cast<float *>(spare_alloc((size_t)need * sizeof(float)));
    c->fused_part_floats = c->d_fused_parts ? need : 0;
    return c->d_fused_parts != nullptr;
}

// items of the fused kernel: the rows of more than fused_row_max entries, cut into segments of
// SDDMM_FUSED_SEG entries (by default 256, and up to 1024 where most rows are about as long)
static int plan_fused_items(sddmm_ctx *c, const unsigned char *panel_owner) {
    if (c->fused_items_valid && c->fused_items_panels == (panel_owner != nullptr) && fused_parts(c, c->fused_seg)) return SDDMM_OK;
    int seg = std::max(WAVE, env_int("SDDMM_FUSED_SEG", 1024));
    const int64_t nb = ((int64_t)c->sM + SCAN_TILE - 1) / SCAN_TILE;
    int row_max = FUSED_ROW_MAX;
    const int arc = ensure_arena(c);
    if (arc) return arc;
    ARENA_HOLDS(c, nb, c->block_sums_cap, "block sums");
    c->n_fused_items = c->n_fused_pieces = c->n_fused_cut = 0;
    if (nb > 0) {
        DevTotals tmp;
        PlanCounters counted;
        int window = WAVE / shape_of(c).LPN;               // rows of a wavefront of the kernel of the short rows
        const int32_t *look_at = c->d_col;                 // (which rows are alike: the first count tells)
        auto count = [&]() -> int {
            HIP_TRY(c, hipMemsetAsync(&c->d_pc->k[K_ROWS_SHORT][0], 0,
                                      sizeof(unsigned long long) * SPREAD * (K_WINDOW - K_ROWS_SHORT + 1), c->stream));
            HIP_TRY(c, hipMemsetAsync(&c->d_pc->n_items, 0, sizeof(unsigned long long), c->stream));
            SDDMM_LAUNCH(c, k_classify_count, nb, SCAN_BLOCK, c->d_rowptr,
                               panel_owner, c->sM, row_max + 1, seg, c->d_block_sums, c->d_pc, 2,
                               (unsigned int *)nullptr, (unsigned int *)nullptr, look_at, window);
            SDDMM_LAUNCH(c, k_scan_block_sums, 1, SCAN_BLOCK, (const unsigned int *)c->d_block_sums, c->d_block_off, (int)nb,
                               &c->d_pc->n_items);
            LAUNCH_CHECK(c);
            const int trc = read_totals(c, &tmp);
            counted = summarize(tmp);
            return trc;
        };
        int rc = count();
        if (rc) return rc;
        const PlanCounters first = counted;
        look_at = nullptr;
        const int64_t item_entries = (int64_t)(first.nnz_medium + first.nnz_long);
        c->fused_rows_alike = 2 * SCAN_ITEMS * first.rows_alike >= first.rows_medium + first.rows_long;
        c->fused_short_avg = first.rows_short ? (double)first.nnz_short / (double)first.rows_short : 0.0;
        if (fused_balanced(c)) window = WAVE;              // (those rows are so short that they are counted again, below)
        // A wavefront walks its item chunk by chunk and the launch waits for the longest one: the long rows are cut into
        // pieces of 256 entries (1024 / 512 / 256: 200 k rows, 128 bytes 85.3 / 84.3 / 81.2 us, 256 bytes 122 / 119 / 116,
        // 512 bytes 228 / 223 / 218; 1 M rows of 128 bytes 289 / 284 / 281; 2.6 M rows 800 / 793 / 787).  Rows that are all
        // about as long as what 3 072 wavefronts would take stay whole: 3 000 rows of 554 entries of 1 KiB 264 us, in
        // pieces of 512 280.
        const int64_t even = ((item_entries / 3072 + WAVE - 1) / WAVE) * WAVE;
        const int longer = (int)std::max<int64_t>(256, std::min<int64_t>(seg, even));
        bool uneven = (int64_t)first.fused_longest > 2 * (int64_t)longer;
        const bool choose_seg = uneven && !getenv("SDDMM_FUSED_SEG");
        const int best_seg = choose_seg ? 256 : seg;
        // Where most of the short rows are very short, one of 17 .. 64 entries among them holds up the rows of its
        // wavefront: those become items too (graphs of 2.8 .. 4 entries per short row, 64 against 16: 50 k rows K=64
        // 46 -> 35 us; 200 k rows K=8 60 -> 44 us, K=64 fp16 92 -> 77, K=128 251 -> 218; 1 M rows K=64 606 -> 566;
        // 2.6 M rows K=32 868 -> 780).  Rows of about one length stay: 42 .. 48 entries each, K=128 54 us, as items 84;
        // 17 .. 23 entries 10.5 and 20 us.
        const int best_row_max = first.rows_short && c->fused_short_avg < 8.0 ? FUSED_ROW_MAX / 4 : FUSED_ROW_MAX;
        if (best_seg != seg || best_row_max != row_max) {
            seg = best_seg;
            row_max = best_row_max;
            rc = count();
            if (rc) return rc;
            // Where that would cut more than a third of the items, most rows are about one length and a few are longer: only
            // those are cut.  (The share is a fifth to a quarter in graphs.  256 / this rule: 36 000 rows of 392 entries and
            // one of 3 365, K=256 766 / 552 us, K=16 92 / 65; 20 000 rows of 390 and 500 of 4 000, K=64 245 / 243, K=16 85 / 78;
            // no row cut that stays whole now, 20 000 rows of 100 and 100 of 4 000: K=64 78 us with 256, 93 without.)
            if (choose_seg && longer > seg && 3 * (counted.rows_long - first.rows_long) > first.rows_medium + first.rows_long) {
                uneven = false;
                seg = longer;
                rc = count();
                if (rc) return rc;
            }
        }
        // Workgroups of one wavefront only where lengths differ: the place on the CU is then free as soon as an item ends
        // (four / one: graphs of 200 k rows, K=64 fp16 78.3 / 74.3 us, K=8 bf16 54.6 / 51.4, K=16 42.6 / 40.5).  Rows of about
        // one length end together, and neighbours share B rows in the vector L1 (banded blocks of 36 k rows K=256 499 / 522,
        // K=16 67.7 / 71.0; uniform rows of 45 entries K=8 bf16 222 / 232).
        c->fused_block_waves = uneven ? 1 : WAVES_PER_BLOCK;
        if (row_max != FUSED_ROW_MAX) {
            // (a launch takes fewer than 2^32 threads: 2^26 items, which rows of more than 64 entries cannot reach)
            if (xcd_grid(blocks_of((int64_t)tmp.n_items, c->fused_block_waves)) * c->fused_block_waves * WAVE >= (int64_t)1 << 32) {
                row_max = FUSED_ROW_MAX;
                rc = count();
                if (rc) return rc;
            }
        }
        // the pieces of the rows that are cut, at the most; without room for them fewer and longer ones, and at last every
        // row stays whole
        const auto pieces = [&]() { return c->n_fused_pieces = (int64_t)counted.rows_long + (int64_t)counted.nnz_long / seg; };
        for (pieces(); !fused_parts(c, seg); pieces()) {
            seg = seg < 1024 ? 1024 : INT_MAX;
            rc = count();
            if (rc) return rc;
        }
        c->n_fused_items = (int64_t)tmp.n_items;
        // (a launch takes fewer than 2^32 threads, a workgroup per cut row)
        const int apart = env_int("SDDMM_FUSED_ADD_APART", -1);
        if ((apart >= 0 ? apart != 0 : counted.fused_window > FUSED_APART_PIECES) && counted.rows_long < (1u << 24))
            c->n_fused_cut = (int64_t)counted.rows_long;
        c->fused_add_block = counted.fused_longest / (unsigned int)seg > 512 && c->n_fused_cut < 65536 ? FUSED_APART_BLOCK : 256;
        const int64_t room = c->n_fused_items + (c->n_fused_cut + 3) / 4;           // a list of rows behind the items
        if (room > c->fused_items_cap) {
            dfree(c->d_fused_items);
            c->fused_items_cap = 0;
            ALLOC_TRY(c, c->d_fused_items, (size_t)room * sizeof(RowItem));
            c->fused_items_cap = room;
        }
        if (c->n_fused_items > 0) {
            SDDMM_LAUNCH(c, k_classify_write, nb, SCAN_BLOCK, c->d_rowptr,
                               panel_owner, c->sM, row_max + 1, seg, (const unsigned int *)c->d_block_off, c->d_fused_items, 2);
            if (c->n_fused_pieces > 0) {
                HIP_TRY(c, hipMemsetAsync(&c->d_pc->fused_pieces, 0, 2 * sizeof(unsigned long long), c->stream));
                SDDMM_LAUNCH(c, k_piece_places, grid_for(c->n_fused_items, 256), 256, (const int32_t *)c->d_rowptr,
                             c->d_fused_items, c->n_fused_items, fused_cut_rows(c), c->d_pc);
            }
            LAUNCH_CHECK(c);
        }
    }
    c->fused_row_max = row_max;
    c->fused_seg = seg;
    c->fused_items_valid = true;
    c->fused_items_panels = panel_owner != nullptr;
    return SDDMM_OK;
}

// items of the fused panel kernel: those of the plan, or a list of its own
static int plan_fused_panels(sddmm_ctx *c) {
    if (c->fused_panels_valid) return SDDMM_OK;
    c->n_fused_panels = 0;
    const bool half_width = c->dtype != SDDMM_F32;
    const int halves_from = fused_halves_from(c->n_panels, panel_mfma_min_waves(panel_mfma_steps(c), true, half_width), half_width);
    if (!getenv("SDDMM_PANEL_SEG") && (halves_from || c->panel_columns != PANEL_COLUMNS)) {
        const int64_t n_panels = (int64_t)c->sM / 8;
        SDDMM_LAUNCH(c, k_fused_panel_counts, (n_panels + 255) / 256, 256, (const int32_t *)c->d_rowptr, n_panels, halves_from,
                     c->d_panel_counts);
        LAUNCH_CHECK(c);
        int rc = device_scan(c, c->d_panel_counts, c->d_panel_off, n_panels, &c->d_pc->panel_items);
        if (rc) return rc;
        DevTotals totals;
        rc = read_totals(c, &totals);
        if (rc) return rc;
        const int64_t n = (int64_t)totals.panel_items;
        if (n > c->fused_panels_cap) {
            dfree(c->d_fused_panels);
            c->fused_panels_cap = 0;
            ALLOC_TRY(c, c->d_fused_panels, (size_t)n * sizeof(RowItem));
            c->fused_panels_cap = n;
        }
        SDDMM_LAUNCH(c, k_panel_items, (n_panels + 255) / 256, 256, (const int32_t *)c->d_rowptr, n_panels, 0, halves_from,
                     (const unsigned int *)c->d_panel_counts, (const unsigned int *)c->d_panel_off, c->d_fused_panels);
        LAUNCH_CHECK(c);
        c->n_fused_panels = n;
    }
    c->fused_panels_valid = true;
    return SDDMM_OK;
}

int sddmm_run_fused(sddmm_ctx *c) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_ready(c);
    if (rc) return rc;
    const Shape s = shape_of(c);
    // 16-byte units, at most 8 lanes per entry and 32 fp32 accumulators of the output row per lane
    if (!s.whole() || s.LPN == 0 || s.LPN > 8 || c->K > 256)
        return fail(c, SDDMM_ERR_UNSUPPORTED,
                    "the fused SDDMM+SpMM needs K <= 256, a multiple of 4 (fp32) or 8 (bf16, fp16)");
    if (!c->have_rowptr) return fail(c, SDDMM_ERR_UNSUPPORTED, "the fused SDDMM+SpMM needs row-sorted entries");
    // rows of 32, 64 or 128 components: the 8-row panels of the current plan (AUTO if there is none
    // yet) take the matrix-core kernel, which shares every gathered B row between 8 rows and both
    // products; the other rows take the gather kernels
    bool panels = (c->K == 32 || c->K == 64 || c->K == 128) && env_int("SDDMM_FUSED_PANELS", 1) != 0;
    if (panels && !c->planned) {
        rc = sddmm_plan(c, c->requested);
        if (rc) return rc;
    }
    panels = panels && c->planned && c->panel_mfma && c->n_panel_items > 0 && c->owner_active &&
             (c->strategy == SDDMM_AUTO || c->strategy == SDDMM_LDS_TILED || c->strategy == SDDMM_MFMA_TILE);
    const unsigned char *panel_owner = panels ? (const unsigned char *)c->d_owner : nullptr;
    rc = plan_fused_items(c, panel_owner);
    if (rc) return rc;
    if (panels) {
        rc = plan_fused_panels(c);
        if (rc) return rc;
    }
    const size_t o_bytes = (size_t)c->M * (size_t)c->K * sizeof(float);
    if (o_bytes > c->o_cap) {
        dfree(c->dO);
        c->o_cap = 0;
        ALLOC_TRY(c, c->dO, o_bytes);
        c->o_cap = o_bytes;
    }
    if (c->nnz > 0) {
        HIP_TRY(c, load_fused());
        if (panels) HIP_TRY(c, load_panels(false));
    }
    HIP_TRY(c, hipEventRecord(c->ev0, c->stream));
    // (when the panels own every row that has entries, O is complete after a memset and the panel kernel;
    // otherwise the kernels of the other rows write every row of O below sM, zeros for the panels' rows,
    // and only the rows of A beyond S are cleared here)
    const bool others = c->sM > 0 && c->nnz > 0 && (!panels || c->n_tiles > 0 || c->rows_short > 0 || c->n_items > 0);
    if (o_bytes) {
        const size_t written = others ? (size_t)c->sM * (size_t)c->K * sizeof(float) : 0;
        if (written < o_bytes) HIP_TRY(c, hipMemsetAsync((char *)c->dO + written, 0, o_bytes - written, c->stream));
    }
    int launches = 0;
    if (c->sM > 0 && c->nnz > 0) {
        if (others) {
            launches = launch_fused_rows(c, panel_owner);
            if (launches == 0) return fail(c, SDDMM_ERR_UNSUPPORTED, "internal: no fused kernel for this row layout");
        }
        if (panels) {
            launch_panels_fused(c);
            ++launches;
        }
        LAUNCH_CHECK(c);
    }
    HIP_TRY(c, hipEventRecord(c->ev1, c->stream));
    HIP_TRY(c, hipEventSynchronize(c->ev1));
    float ms = 0.f;
    HIP_TRY(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->stats.run_ms = ms;
    c->stats.kernels_launched = launches;
    c->have_fused = true;
    return SDDMM_OK;
}

int sddmm_get_fused(sddmm_ctx *c, float *O) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    if (!c->have_fused) return fail(c, SDDMM_ERR_STATE, "no fused result: call sddmm_run_fused first");
    const size_t o_bytes = (size_t)c->M * (size_t)c->K * sizeof(float);
    if (o_bytes > 0 && !O) return fail(c, SDDMM_ERR_NULL, "O is NULL");
    if (o_bytes) HIP_TRY(c, hipMemcpyAsync(O, c->dO, o_bytes, hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return SDDMM_OK;
}

int sddmm_get_fused_device(sddmm_ctx *c, const float **dO) {
    if (!c || !dO) return SDDMM_ERR_NULL;
    if (!c->have_fused) return fail(c, SDDMM_ERR_STATE, "no fused result: call sddmm_run_fused first");
    *dO = c->dO;
    return SDDMM_OK;
}

int sddmm_time_runs(sddmm_ctx *c, int warmup, int reps, int include_plan, float *ms_each) {
    if (!c) return SDDMM_ERR_NULL;
    if (reps < 0 || warmup < 0) return fail(c, SDDMM_ERR_INVALID, "negative repetition count");
    if (reps > 0 && !ms_each) return fail(c, SDDMM_ERR_NULL, "ms_each is NULL");
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_ready(c);
    if (rc) return rc;
    if (!c->planned) {
        // operands were replaced since the last plan: plan again as last asked (AUTO on a new context)
        rc = sddmm_plan(c, c->requested);
        if (rc) return rc;
    }
    const int requested = c->requested;
    for (int i = 0; i < warmup + reps; ++i) {
        HIP_TRY(c, hipEventRecord(c->ev0, c->stream));
        if (include_plan) {
            rc = do_plan(c, requested);
            if (rc) return rc;
        }
        rc = enqueue_run(c);
        if (rc) return rc;
        HIP_TRY(c, hipEventRecord(c->ev1, c->stream));
        HIP_TRY(c, hipEventSynchronize(c->ev1));
        if (i >= warmup) HIP_TRY(c, hipEventElapsedTime(&ms_each[i - warmup], c->ev0, c->ev1));
    }
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return SDDMM_OK;
}

int sddmm_time_region(sddmm_ctx *c, int reps, int include_plan, float *total_ms) {
    if (!c) return SDDMM_ERR_NULL;
    if (reps < 1) return fail(c, SDDMM_ERR_INVALID, "repetition count must be positive");
    if (!total_ms) return fail(c, SDDMM_ERR_NULL, "total_ms is NULL");
    HIP_TRY(c, hipSetDevice(c->device));
    int rc = check_ready(c);
    if (rc) return rc;
    if (!c->planned) {
        // operands were replaced since the last plan: plan again as last asked (AUTO on a new context)
        rc = sddmm_plan(c, c->requested);
        if (rc) return rc;
    }
    const int requested = c->requested;
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    HIP_TRY(c, hipEventRecord(c->ev0, c->stream));
    for (int i = 0; i < reps; ++i) {
        if (include_plan) {
            rc = do_plan(c, requested);
            if (rc) return rc;
        }
        rc = enqueue_run(c);
        if (rc) return rc;
    }
    HIP_TRY(c, hipEventRecord(c->ev1, c->stream));
    HIP_TRY(c, hipEventSynchronize(c->ev1));
    HIP_TRY(c, hipEventElapsedTime(total_ms, c->ev0, c->ev1));
    return SDDMM_OK;
}

int sddmm_get_values(sddmm_ctx *c, float *P_values) {
    if (!c) return SDDMM_ERR_NULL;
    HIP_TRY(c, hipSetDevice(c->device));
    if (!c->have_sparse) return fail(c, SDDMM_ERR_STATE, "no sparse operand set");
    if (c->nnz > 0 && !P_values) return fail(c, SDDMM_ERR_NULL, "P_values is NULL");
    if (c->nnz) HIP_TRY(c, hipMemcpyAsync(P_values, c->dP, (size_t)c->nnz * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return SDDMM_OK;
}

int sddmm_get_values_device(sddmm_ctx *c, const float **dP) {
    if (!c || !dP) return SDDMM_ERR_NULL;
    if (!c->have_sparse) return fail(c, SDDMM_ERR_STATE, "no sparse operand set");
    *dP = c->dP;
    return SDDMM_OK;
}

int sddmm_last_stats(const sddmm_ctx *c, sddmm_stats *out) {
    if (!c || !out) return SDDMM_ERR_NULL;
    *out = c->stats;
    return SDDMM_OK;
}

int sddmm_flat_variant(const sddmm_ctx *c, int *variant) {
    if (!c || !variant) return SDDMM_ERR_NULL;
    const bool flat = c->planned && c->strategy == SDDMM_FLAT;
    *variant = !flat ? 0 : (c->use_slices ? SDDMM_FLAT_SLICES : 0) | (c->use_blocks ? SDDMM_FLAT_BLOCKS : 0) |
                               (c->use_order ? SDDMM_FLAT_SORTED : 0);
    return SDDMM_OK;
}

// ---- the entry point that allocates nothing ---------------------------------------
// The row index per stored entry that the flat kernel reads (k_expand_rows writes it,
// k_flat reads it) lives in a static device array instead of a hipMalloc'ed buffer.
// Every device the library runs on holds its own copy of the array at its own address
// until the process ends; in host code the array's name is only a handle for
// hipGetSymbolAddress, never an address to hand to a kernel.
}  // extern "C"

static __device__ __align__(256) int32_t scratch[SDDMM_NOALLOC_MAX_NNZ];

namespace {
constexpr int NOALLOC_MAX_DEVICES = 64;
int32_t *g_scratch_ptr[NOALLOC_MAX_DEVICES] = {nullptr};   // device address of `scratch`, per device
std::mutex g_scratch_mu;

// Device address of the current device's copy of `scratch` (looked up once per device, when the flat kernels are loaded too).
int scratch_of_current_device(int *device, int32_t **ptr) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) return SDDMM_ERR_NO_DEVICE;
    if (dev >= NOALLOC_MAX_DEVICES) return SDDMM_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> guard(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p || load_flat() != hipSuccess) return SDDMM_ERR_HIP;
        g_scratch_ptr[dev] = static_cast<int32_t *>(p);
    }
    *device = dev;
    *ptr = g_scratch_ptr[dev];
    return SDDMM_OK;
}
}  // namespace

extern "C" {

int sddmm_launch_noalloc(int M, int N, int K, int64_t nnz, const float *dA, const float *dB,
                         const int32_t *d_rowptr, const int32_t *d_col, const float *d_sval, float *dP,
                         void *stream) {
    if (M < 0 || N < 0 || K < 1 || nnz < 0) return SDDMM_ERR_INVALID;
    if (nnz > 0 && (M == 0 || N == 0)) return SDDMM_ERR_INVALID;
    if (nnz > (int64_t)SDDMM_NOALLOC_MAX_NNZ) return SDDMM_ERR_TOO_LARGE;
    if (!d_rowptr || (nnz > 0 && (!dA || !dB || !d_col || !d_sval || !dP))) return SDDMM_ERR_NULL;
    if (((uintptr_t)dA | (uintptr_t)dB) & 15) return SDDMM_ERR_INVALID;
    int device = -1;
    int32_t *rowidx = nullptr;
    const int rc = scratch_of_current_device(&device, &rowidx);
    if (rc) return rc;
    if (nnz == 0) return SDDMM_OK;
    // a context on the stack: nothing is allocated for it, it only carries the launch arguments
    sddmm_ctx c;
    c.device = device;
    c.stream = static_cast<hipStream_t>(stream);
    c.M = M; c.N = N; c.K = K; c.dtype = SDDMM_F32;
    c.dA = const_cast<float *>(dA);
    c.dB = const_cast<float *>(dB);
    c.sM = M; c.sN = N; c.nnz = nnz;
    c.d_rowptr = const_cast<int32_t *>(d_rowptr);
    c.d_col = const_cast<int32_t *>(d_col);
    c.d_sval = const_cast<float *>(d_sval);
    c.dP = dP;
    c.d_rowidx = rowidx;                       // every position below nnz is rewritten: nothing to clear
    // (bounded by nnz: a row pointer that runs past it cannot make the kernel leave the array)
    SDDMM_LAUNCH(&c, k_expand_rows, grid_for(M, 256), 256, c.d_rowptr, M, rowidx, nnz);
    launch_flat(&c);
    if (hipGetLastError() != hipSuccess) return SDDMM_ERR_HIP;
    if (c.oversize) return SDDMM_ERR_UNSUPPORTED;
    return SDDMM_OK;
}

// Smallest feasible maximum load by bisection, then a greedy left-to-right fill
// with that load: the contract of CSR<T>::_dispatch (src/matrices/CSR.hpp:196-264).
int sddmm_partition_rows(int M, const int32_t *rowptr, int parts, int stride, int32_t *start_idx) {
    if (!rowptr || !start_idx) return SDDMM_ERR_NULL;
    if (M <= 0 || parts <= 0 || stride <= 0 || M % stride) return SDDMM_ERR_INVALID;
    const int64_t groups = M / stride;
    auto load = [&](int64_t g) { return (int64_t)rowptr[(g + 1) * stride] - (int64_t)rowptr[g * stride]; };
    int64_t heaviest = 0;
    for (int64_t g = 0; g < groups; ++g) heaviest = std::max(heaviest, load(g));
    auto parts_needed = [&](int64_t cap) {
        int64_t used = 1, acc = 0;
        for (int64_t g = 0; g < groups; ++g) {
            acc += load(g);
            if (acc > cap) { ++used; acc = load(g); }
        }
        return used;
    };
    int64_t lo = std::max<int64_t>(1, heaviest), hi = std::max<int64_t>(lo, rowptr[M]);
    int64_t cap = 0;                       // stays 0 when even cap == nnz needs too many parts
    if (parts_needed(hi) <= parts) {
        while (lo < hi) {
            const int64_t mid = lo + (hi - lo) / 2;
            if (parts_needed(mid) <= parts) hi = mid; else lo = mid + 1;
        }
        cap = lo;
    }
    int w = 0;
    int64_t acc = 0;
    start_idx[w++] = 0;
    for (int64_t g = 0; g < groups; ++g) {
        acc += load(g);
        if (acc > cap) {
            if (w > parts) return SDDMM_ERR_INVALID;
            start_idx[w++] = (int32_t)(g * stride);
            acc = load(g);
        }
    }
    while (w <= parts) start_idx[w++] = M;
    return SDDMM_OK;
}

}  // extern "C"
