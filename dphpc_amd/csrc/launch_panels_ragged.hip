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

void launch_ragged_panels(sddmm_ctx *c) {
    if (c->dtype == SDDMM_BF16) launch_ragged_panel_steps<DT_BF16, UnitBF16x8>(c, c->K / 8);
    else if (c->dtype == SDDMM_F16) launch_ragged_panel_steps<DT_F16, UnitF16x8>(c, c->K / 8);
    else launch_ragged_panel_steps<DT_F32, UnitF32x4u>(c, c->K);
}

hipError_t load_ragged_panels() { return load_code(reinterpret_cast<const void *>(k_panel_mfma<DT_F32, 2, false, RaggedRows<UnitF32x4u, 2>>)); }
