// Launches of the dense-tile kernels: rows of whole steps of 64 bytes.
#include "launch_tiles.h"

template <int DT>
void launch_tile_steps(sddmm_ctx *c) {
    switch (c->tile_steps) {
        case 1: launch_tile_t<DT, 1, WholeRows<1>>(c, 0); break;
        case 2: launch_tile_t<DT, 2, WholeRows<2>>(c, 0); break;
        case 4: launch_tile_t<DT, 4, WholeRows<4>>(c, 0); break;
        case 8: launch_tile_t<DT, 8, WholeRows<8>>(c, 0); break;
        default: launch_tile_t<DT, 16, WholeRows<16>>(c, 0); break;
    }
}

bool launch_auto_with_tiles(sddmm_ctx *c) {
    return c->ragged ? launch_ragged_auto_with_tiles(c) : launch_auto_with_tiles_t<false>(c);
}
void launch_tiles(sddmm_ctx *c) {
    if (c->ragged) launch_ragged_tiles(c);
    else if (c->dtype == SDDMM_BF16) launch_tile_steps<DT_BF16>(c);
    else if (c->dtype == SDDMM_F16) launch_tile_steps<DT_F16>(c);
    else launch_tile_steps<DT_F32>(c);
}

hipError_t load_tiles(bool ragged) {
    return ragged ? load_ragged_tiles() : load_code(reinterpret_cast<const void *>(k_tile<DT_F32, 1, WholeRows<1>>));
}
