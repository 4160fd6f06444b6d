// Launches of the gather kernels that work by rows.
#include "context.h"

void launch_row_wave(sddmm_ctx *c, const RowItem *items, int64_t n_items) {
    const Shape s = shape_of(c);
    const int64_t nblocks = (n_items + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        SDDMM_LAUNCH(c, (k_row_wave<LT>), xcd_grid(nblocks), BLOCK, nblocks, n_items, items, c->d_rowptr, c->d_col,
                     (const void *)c->dA, (const void *)c->dB, s.len, c->d_sval, c->dP);
    });
}

void launch_short_rows(sddmm_ctx *c, int ts, int rpw) {
    const Shape s = shape_of(c);
    const int64_t waves = ((int64_t)c->sM + rpw - 1) / rpw;
    const int64_t nblocks = (waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        SDDMM_LAUNCH(c, (k_short_rows<LT>), xcd_grid(nblocks), BLOCK,
                           (const void *)c->dA, (const void *)c->dB, s.len, c->d_rowptr, c->d_col, c->d_sval, c->dP,
                           c->sM, ts, rpw, nblocks);
    });
}

hipError_t load_rows() { return load_code(reinterpret_cast<const void *>(k_row_wave<Layout<UnitF32x1, 4, 1, false, false>>)); }
