// Launches of the dense-tile kernels, alone and together with the rows, for rows of whole steps (launch_tiles.hip) and
// ragged ones (launch_tiles_ragged.hip).
#pragma once
#include "context.h"

// Tiles and rows in one launch (k_auto_tiles); measured faster than two launches at
// every row size the tile path takes (mixed-density shape: 23 -> 20 us at 128-byte
// rows, 107 -> 92 us at 1 KiB rows).  Returns false when the layout has no fused
// kernel; the caller then launches the two kernels in turn.
// RAGGED: the layouts of rows that are no STEPS * 64 bytes.
template <bool RAGGED>
bool launch_auto_with_tiles_t(sddmm_ctx *c) {
    const Shape s = shape_of(c);
    if (c->tile_steps < 1 || c->tile_steps > env_int("SDDMM_FUSE_STEPS", 16) || s.wide || s.LPN * s.UPL != 4 * c->tile_steps) return false;
    const int64_t waves = short_row_waves(c);
    const int64_t short_blocks = (waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    const int64_t item_blocks = (c->n_items + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    const int64_t tile_blocks = (c->n_tile_units + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    const int64_t nblocks = short_blocks + item_blocks + tile_blocks;
    // Order of the blocks on every XCD.  Rows of up to 256 bytes: the tile windows (the wavefronts that
    // live longest) start first, then the items, then the chunks of the entry list -- measured
    // 14.7 -> 13.5 us on the mixed-density shape at 128 bytes, 21.3 -> 21.1 us (cold 29.7 -> 27.8) at
    // 256; at 1 KiB, where the gathers of the short rows are the longer half, the even deal is 3 % faster.
    const int longest_first = env_int("SDDMM_LONGEST_FIRST", c->tile_steps <= 4 ? 1 : 0);
    auto eighth = [](int64_t n) { return (n + NUM_XCD - 1) / NUM_XCD; };
    const int64_t grid = longest_first ? NUM_XCD * (eighth(short_blocks) + eighth(item_blocks) + eighth(tile_blocks))
                                       : xcd_grid(nblocks);
    bool launched = false;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        constexpr int KU_ = LT::LPN * LT::UPL;
        if constexpr (!LT::LONG && LT::FULLK != RAGGED && !LT::WIDE && LT::U::ELEMS > 1 && (LT::LPN == 4 || LT::LPN == 8) &&
                      (RAGGED || (LT::U::WHOLE && LT::UPL != 3 && LT::UPL != 6))) {
            SDDMM_LAUNCH(c, (k_auto_tiles<LT, KU_ / 4>), grid, BLOCK, (int)tile_blocks, (int)nblocks, (int)short_blocks,
                         longest_first, (int)c->n_windows, (int)c->n_win_single,
                         (const TileWindow *)(c->use_windows ? c->d_windows : nullptr),
                         (const int2 *)(c->use_short_list ? c->d_short_list : nullptr), (const void *)c->dA,
                         (const void *)c->dB, c->d_col, c->d_sval, c->dP, c->nnz, c->sM, c->N, s.len, c->ts, c->rpw,
                         c->d_rowptr, (const unsigned char *)(c->owner_active ? c->d_owner : nullptr), c->d_items, c->n_items,
                         (const int32_t *)c->d_vrows, (const int32_t *)c->d_tile_cols, (const TileDesc *)c->d_tiles,
                         c->n_tiles, c->n_short_list, (const int32_t *)(c->use_win_order ? c->d_win_order : nullptr));
            launched = true;
        }
    });
    return launched;
}

// KSTEPS, KR: what the kernel that splits K takes (a multiple of KSPLIT steps)
template <int DT, int STEPS, class R, int KSTEPS = STEPS, class KR = R>
void launch_tile_t(sddmm_ctx *c, int len) {
    // Well-filled tiles (walked from the descriptors' masks) of rows of 256 bytes and more, fewer
    // windows than keep the chip busy on their own: one workgroup per window, K in four parts.
    if constexpr (KSTEPS % KSPLIT == 0) {
        if (!c->use_windows && c->n_windows <= (int64_t)env_int("SDDMM_KSPLIT_MAX", 32768) && env_int("SDDMM_KSPLIT", 1) != 0) {
            const int64_t nb = c->n_windows;
            SDDMM_LAUNCH(c, (k_tile_ksplit<DT, KSTEPS, KR>), xcd_grid(nb), BLOCK, nb,
                         (const int32_t *)(c->use_win_order ? c->d_win_order : nullptr), (const TileDesc *)c->d_tiles,
                         c->n_tiles, (const int32_t *)c->d_tile_cols, (const void *)c->dA, (const void *)c->dB, len, c->M,
                         c->N, (const int32_t *)c->d_vrows, (const float *)c->d_sval, c->dP);
            return;
        }
    }
    const int64_t nblocks = (c->n_tile_units + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    SDDMM_LAUNCH(c, (k_tile<DT, STEPS, R>), xcd_grid(nblocks), BLOCK, nblocks,
                 (const TileWindow *)(c->use_windows ? c->d_windows : nullptr), c->n_windows, c->n_win_single,
                 (const int32_t *)(c->use_win_order ? c->d_win_order : nullptr), (const void *)c->dA, (const void *)c->dB,
                 len, c->M, c->N, (const int32_t *)c->d_vrows, (const int32_t *)c->d_tile_cols, (const TileDesc *)c->d_tiles,
                 c->n_tiles, (const int32_t *)c->d_col, (const float *)c->d_sval, c->dP, c->nnz);
}
