// Launch of the kernel that takes short rows and row segments together.
#include "context.h"

void launch_auto(sddmm_ctx *c) {
    const Shape s = shape_of(c);
    const int64_t waves = short_row_waves(c);
    const int64_t short_blocks = (waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    const int64_t item_blocks = (c->n_items + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    const int64_t nblocks = short_blocks + item_blocks;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        SDDMM_LAUNCH(c, (k_auto<LT>), xcd_grid(nblocks), BLOCK, nblocks, short_blocks, c->d_items, c->n_items,
                     (const int2 *)(c->use_short_list ? c->d_short_list : nullptr), (const void *)c->dA, (const void *)c->dB,
                     s.len, c->d_rowptr, (const unsigned char *)(c->owner_active ? c->d_owner : nullptr), c->d_col, c->d_sval,
                     c->dP, c->sM, c->ts, c->rpw, c->n_short_list);
    });
}

hipError_t load_auto() { return load_code(reinterpret_cast<const void *>(k_auto<Layout<UnitF32x1, 4, 1, false, false>>)); }
