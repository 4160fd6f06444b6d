// Launches of the gather kernels of the fused SDDMM + SpMM.
#include "context.h"
#include "kernels_fused.h"

// Short rows of fewer entries, on average, than half of what a lane group takes per step (a power-law
// graph: 2.8 against 8 lanes per entry) leave most lanes of a group idle in one row per lane group: the
// wavefronts deal whole rows out to their groups by entry count instead.  That takes 64 rows per wavefront,
// so it needs enough rows to fill the chip: graphs of 2.6 M rows, 128 bytes 935 -> 781 us, 1 M rows 337 -> 287 us
// (256 bytes 593 -> 569), 500 k rows 169 -> 152 us; 200 k rows 66 -> 63 us (128 bytes), 217 -> 235 us (512
// bytes); 50 k rows 25 -> 32 us, 8 k rows 14 -> 23 us.  With longer rows, or fewer lanes per entry, the extra
// gathers of the A rows and the longer walks cost more than the idle lanes (12.5 entries per short row: 31 -> 64 us;
// 1 M rows of 64 bytes 249 -> 281 us).
bool fused_balanced(const sddmm_ctx *c) {
    const int mode = env_int("SDDMM_FUSED_BALANCED", -1);
    if (mode >= 0) return mode != 0;
    return c->sM >= 400000 && c->fused_short_avg > 0.0 && 2.0 * c->fused_short_avg < (double)shape_of(c).LPN;
}

// k_fusedmm in steps (its comment has both sides): items of about one length (they were not cut to 256 entries), more of
// them than the chip holds wavefronts (256 CUs x 32), and neighbouring rows do not share their columns.  Lanes with four
// bf16 units lose half of their places to the batches: steps whatever the number and the columns (steps / batches: 3 000
// rows of 300 .. 700 entries 77 / 88 us, near-dense rows 141 / 147, banded rows 390 / 405), batches in graphs (73 / 71).
// SDDMM_FUSED_STEPS 0 / 1 overrides it.
template <class L>
bool fused_in_steps(const sddmm_ctx *c) {
    const int mode = env_int("SDDMM_FUSED_STEPS", -1);
    if (mode >= 0) return mode != 0;
    if (c->fused_block_waves == 1) return false;
    return (L::U::DT == DT_BF16 && L::UPL >= 4) || (c->n_fused_items > 256 * 32 && !c->fused_rows_alike);
}

// The work items of the rows of more than fused_row_max entries, then the other rows; 0: no kernel for this row layout.
int launch_fused_rows(sddmm_ctx *c, const unsigned char *panel_owner) {
    const Shape s = shape_of(c);
    const bool balanced = fused_balanced(c);
    int launches = 0;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        if constexpr (!LT::LONG && LT::LPN <= 8 && LT::U::ELEMS > 1 && LT::U::WHOLE && LT::UPL * LT::U::ELEMS <= 32) {
            const int64_t rows_per_wave = WAVE / LT::LPN;
            const int64_t waves = ((int64_t)c->sM + rows_per_wave - 1) / rows_per_wave;
            const int64_t rblocks = blocks_of(waves, c->fused_block_waves);
            if (c->n_fused_items > 0) {
                const int64_t nblocks = blocks_of(c->n_fused_items, c->fused_block_waves);
                auto launch = [&](auto kernel) {
                    SDDMM_LAUNCH(c, kernel, xcd_grid(nblocks), c->fused_block_waves * WAVE, nblocks, c->n_fused_items,
                                 (const RowItem *)c->d_fused_items, c->d_col, c->d_sval, (const void *)c->dA,
                                 (const void *)c->dB, s.len, c->d_rowptr, c->dP, c->dO, c->d_fused_parts);
                };
                if constexpr (LT::UPL == 1) launch(k_fusedmm<LT, false>);
                else if (fused_in_steps<LT>(c)) launch(k_fusedmm<LT, true>);
                else launch(k_fusedmm<LT, false>);
                ++launches;
            }
            if (c->n_fused_cut > 0) {
                SDDMM_LAUNCH(c, k_add_cut_rows, c->n_fused_cut, c->fused_add_block, (const float *)c->d_fused_parts, c->dO, c->K,
                             c->fused_seg, (const int32_t *)c->d_rowptr, (const int32_t *)fused_cut_rows(c));
                ++launches;
            }
            const int seg = c->n_fused_cut > 0 ? INT_MAX : c->fused_seg;      // the pieces are added by the kernel of the other rows
            if (balanced) {
                const int64_t bwaves = ((int64_t)c->sM + WAVE - 1) / WAVE;
                const int64_t bblocks = blocks_of(bwaves, c->fused_block_waves);
                SDDMM_LAUNCH(c, (k_fusedmm_rows_balanced<LT>), xcd_grid(bblocks), c->fused_block_waves * WAVE, bblocks,
                             c->d_rowptr, panel_owner, c->d_col, c->d_sval, (const void *)c->dA, (const void *)c->dB, s.len,
                             c->dP, c->dO, (const float *)c->d_fused_parts, c->sM, c->fused_row_max, seg);
            } else {
                SDDMM_LAUNCH(c, (k_fusedmm_rows<LT>), xcd_grid(rblocks), c->fused_block_waves * WAVE, rblocks, c->d_rowptr,
                             panel_owner, c->d_col, c->d_sval, (const void *)c->dA, (const void *)c->dB, s.len, c->dP, c->dO,
                             (const float *)c->d_fused_parts, c->sM, c->fused_row_max, seg);
            }
            ++launches;
        }
    });
    return launches;
}

hipError_t load_fused() { return load_code(reinterpret_cast<const void *>(k_fusedmm<Layout<UnitF32x4, 8, 1, true, false>, false>)); }
