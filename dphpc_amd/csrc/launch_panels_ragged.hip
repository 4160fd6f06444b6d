// Launches of the matrix-core panel kernel: rows of no whole number of steps of 64 bytes.
#include "launch_panels.h"

template <int DT, class U>
void launch_ragged_panel_steps(sddmm_ctx *c, int len) {
    switch (ragged_steps(c)) {
        case 1: launch_panel_mfma_t<DT, 1, RaggedRows<U, 1>>(c, len); break;
        case 2: launch_panel_mfma_t<DT, 2, RaggedRows<U, 2>>(c, len); break;
        case 4: launch_panel_mfma_t<DT, 4, RaggedRows<U, 4>>(c, len); break;
        case 6: launch_panel_mfma_t<DT, 6, RaggedRows<U, 6>>(c, len); break;
        case 8: launch_panel_mfma_t<DT, 8, RaggedRows<U, 8>>(c, len); break;
        case 12: launch_panel_mfma_t<DT, 12, RaggedRows<U, 12>>(c, len); break;
        default: launch_panel_mfma_t<DT, 16, RaggedRows<U, 16>>(c, len); break;
    }
}

// rows of more than 1 KiB: LONG_STEPS at a time
template <int DT, class U>
int launch_long_panel_steps(sddmm_ctx *c, int len, int units) {
    constexpr int PW = panel_mfma_waves(LONG_STEPS);
    const int64_t nblocks = (c->n_panel_items + PW - 1) / PW;
    int launches = 0;
    for (int unit0 = 0; unit0 < units; unit0 += 4 * LONG_STEPS, ++launches)
        SDDMM_LAUNCH(c, (k_panel_mfma<DT, LONG_STEPS, false, RaggedRows<U, LONG_STEPS>, true>), xcd_grid(nblocks), PW * WAVE,
                     (const RowItem *)c->d_panel_items, c->n_panel_items, nblocks, c->d_rowptr, c->d_col, (const void *)c->dA,
                     (const void *)c->dB, len, (const float *)c->d_sval, c->dP, (float *)nullptr, unit0);
    return launches;
}

int launch_long_panels(sddmm_ctx *c) {
    if (c->dtype == SDDMM_BF16) return launch_long_panel_steps<DT_BF16, UnitBF16x8>(c, c->K / 8, c->K / 8);
    if (c->dtype == SDDMM_F16) return launch_long_panel_steps<DT_F16, UnitF16x8>(c, c->K / 8, c->K / 8);
    return launch_long_panel_steps<DT_F32, UnitF32x4u>(c, c->K, (c->K + 3) / 4);
}

void launch_ragged_panels(sddmm_ctx *c) {
    if (c->dtype == SDDMM_BF16) launch_ragged_panel_steps<DT_BF16, UnitBF16x8>(c, c->K / 8);
    else if (c->dtype == SDDMM_F16) launch_ragged_panel_steps<DT_F16, UnitF16x8>(c, c->K / 8);
    else launch_ragged_panel_steps<DT_F32, UnitF32x4u>(c, c->K);
}

hipError_t load_ragged_panels() { return load_code(reinterpret_cast<const void *>(k_panel_mfma<DT_F32, 2, false, RaggedRows<UnitF32x4u, 2>>)); }
