// Launch of the matrix-core panel kernel, for rows of whole steps (launch_panels.hip) and ragged ones
// (launch_panels_ragged.hip).
#pragma once
#include "context.h"

template <int DT, int STEPS, class R>
void launch_panel_mfma_t(sddmm_ctx *c, int len) {
    constexpr int PW = panel_mfma_waves(STEPS);
    const int64_t nblocks = (c->n_panel_items + PW - 1) / PW;
    SDDMM_LAUNCH(c, (k_panel_mfma<DT, STEPS, false, R>), xcd_grid(nblocks), PW * WAVE,
                 (const RowItem *)c->d_panel_items, c->n_panel_items, nblocks, c->d_rowptr, c->d_col, (const void *)c->dA,
                 (const void *)c->dB, len, (const float *)c->d_sval, c->dP, (float *)nullptr, 0);
}
