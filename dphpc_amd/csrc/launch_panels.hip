// Launches of the row-panel kernels.
#include "launch_panels.h"

template <class U, int UPL>
void launch_panel_t(sddmm_ctx *c, int KU) {
    using LT = Layout<U, 8, UPL, true, false>;
    const int64_t nblocks = (c->n_panel_items + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    SDDMM_LAUNCH(c, (k_panel<LT>), xcd_grid(nblocks), BLOCK,
                       (const void *)c->dA, (const void *)c->dB, KU, c->d_rowptr, c->d_col, c->d_sval, c->dP,
                       (const RowItem *)c->d_panel_items, c->n_panel_items, nblocks);
}
template <class U>
void launch_panel_u(sddmm_ctx *c, const Shape &s) {
    if (s.UPL == 1) launch_panel_t<U, 1>(c, s.KU);
    else launch_panel_t<U, 2>(c, s.KU);
}
// the panels of the fused SDDMM+SpMM: P and the panels' part of O
template <int DT, int STEPS>
void launch_panel_fused_t(sddmm_ctx *c) {
    constexpr int PW = panel_mfma_waves(STEPS);
    const int64_t n_items = c->n_fused_panels ? c->n_fused_panels : c->n_panel_items;
    const int64_t nblocks = (n_items + PW - 1) / PW;
    SDDMM_LAUNCH(c, (k_panel_mfma<DT, STEPS, true>), xcd_grid(nblocks), PW * WAVE,
                 (const RowItem *)(c->n_fused_panels ? c->d_fused_panels : c->d_panel_items), n_items, nblocks, c->d_rowptr, c->d_col, (const void *)c->dA,
                 (const void *)c->dB, 0, (const float *)c->d_sval, c->dP, c->dO, 0);
}
template <int DT>
void launch_panel_mfma_steps(sddmm_ctx *c) {
    switch (panel_mfma_steps(c)) {
        case 1: launch_panel_mfma_t<DT, 1, WholeRows<1>>(c, 0); break;
        case 2: launch_panel_mfma_t<DT, 2, WholeRows<2>>(c, 0); break;
        case 4: launch_panel_mfma_t<DT, 4, WholeRows<4>>(c, 0); break;
        case 8: launch_panel_mfma_t<DT, 8, WholeRows<8>>(c, 0); break;
        default: launch_panel_mfma_t<DT, 16, WholeRows<16>>(c, 0); break;
    }
}

void launch_panels(sddmm_ctx *c) {
    if (c->panel_mfma && c->ragged) {
        launch_ragged_panels(c);
        return;
    }
    if (c->panel_mfma) {
        if (c->dtype == SDDMM_BF16) launch_panel_mfma_steps<DT_BF16>(c);
        else if (c->dtype == SDDMM_F16) launch_panel_mfma_steps<DT_F16>(c);
        else launch_panel_mfma_steps<DT_F32>(c);
        return;
    }
    const Shape s = shape_of(c);
    if (s.unit == 0) launch_panel_u<UnitF32x4>(c, s);
    else if (s.unit == 2) launch_panel_t<UnitBF16x8, 1>(c, s.KU);
    else launch_panel_t<UnitF16x8, 1>(c, s.KU);
}

void launch_panels_fused(sddmm_ctx *c) {
    if (c->dtype == SDDMM_F32) {
        if (c->K == 32) launch_panel_fused_t<DT_F32, 2>(c);
        else if (c->K == 64) launch_panel_fused_t<DT_F32, 4>(c);
        else launch_panel_fused_t<DT_F32, 8>(c);
    } else if (c->dtype == SDDMM_BF16) {
        if (c->K == 32) launch_panel_fused_t<DT_BF16, 1>(c);
        else if (c->K == 64) launch_panel_fused_t<DT_BF16, 2>(c);
        else launch_panel_fused_t<DT_BF16, 4>(c);
    } else {
        if (c->K == 32) launch_panel_fused_t<DT_F16, 1>(c);
        else if (c->K == 64) launch_panel_fused_t<DT_F16, 2>(c);
        else launch_panel_fused_t<DT_F16, 4>(c);
    }
}

hipError_t load_panels(bool ragged) {
    return ragged ? load_ragged_panels() : load_code(reinterpret_cast<const void *>(k_panel_mfma<DT_F32, 2>));
}
