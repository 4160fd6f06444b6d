// Launches of the dense-tile kernels: rows of no whole number of steps of 64 bytes.
#include "launch_tiles.h"

template <int DT, class U>
void launch_ragged_tile_steps(sddmm_ctx *c, int len) {
    switch (c->tile_steps) {
        case 1: launch_tile_t<DT, 1, RaggedRows<U, 1>>(c, len); break;
        case 2: launch_tile_t<DT, 2, RaggedRows<U, 2>>(c, len); break;
        case 4: launch_tile_t<DT, 4, RaggedRows<U, 4>>(c, len); break;
        case 6: launch_tile_t<DT, 6, RaggedRows<U, 6>, 8, RaggedRows<U, 8>>(c, len); break;
        case 8: launch_tile_t<DT, 8, RaggedRows<U, 8>>(c, len); break;
        case 12: launch_tile_t<DT, 12, RaggedRows<U, 12>>(c, len); break;
        default: launch_tile_t<DT, 16, RaggedRows<U, 16>>(c, len); break;
    }
}

// rows of more than 1 KiB: LONG_STEPS at a time
template <int DT, class U>
void launch_long_tile_steps(sddmm_ctx *c, int len) {
    SDDMM_LAUNCH(c, (k_tile_ksplit<DT, LONG_STEPS, RaggedRows<U, LONG_STEPS>, true>), xcd_grid(c->n_windows), BLOCK, c->n_windows,
                 (const int32_t *)(c->use_win_order ? c->d_win_order : nullptr), (const TileDesc *)c->d_tiles, c->n_tiles,
                 (const int32_t *)c->d_tile_cols, (const void *)c->dA, (const void *)c->dB, len, c->M, c->N,
                 (const int32_t *)c->d_vrows, (const float *)c->d_sval, c->dP);
}
void launch_long_tiles(sddmm_ctx *c) {
    if (c->dtype == SDDMM_BF16) launch_long_tile_steps<DT_BF16, UnitBF16x8>(c, c->K / 8);
    else if (c->dtype == SDDMM_F16) launch_long_tile_steps<DT_F16, UnitF16x8>(c, c->K / 8);
    else launch_long_tile_steps<DT_F32, UnitF32x4u>(c, c->K);
}

bool launch_ragged_auto_with_tiles(sddmm_ctx *c) { return launch_auto_with_tiles_t<true>(c); }
void launch_ragged_tiles(sddmm_ctx *c) {
    if (c->dtype == SDDMM_BF16) launch_ragged_tile_steps<DT_BF16, UnitBF16x8>(c, c->K / 8);
    else if (c->dtype == SDDMM_F16) launch_ragged_tile_steps<DT_F16, UnitF16x8>(c, c->K / 8);
    else launch_ragged_tile_steps<DT_F32, UnitF32x4u>(c, c->K);
}

hipError_t load_ragged_tiles() { return load_code(reinterpret_cast<const void *>(k_tile<DT_F32, 1, RaggedRows<UnitF32x4u, 1>>)); }
