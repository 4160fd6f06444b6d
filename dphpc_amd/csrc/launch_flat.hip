// Launch of the flat gather kernel.
#include "context.h"

void launch_flat(sddmm_ctx *c) {
    const Shape s = shape_of(c);
    const int64_t chunks = (c->nnz + WAVE - 1) / WAVE;
    const int cpw = (int)std::min<int64_t>(8, std::max<int64_t>(1, chunks / (WAVES_PER_BLOCK * 4096)));
    const int64_t waves = (chunks + cpw - 1) / cpw;
    const int64_t nblocks = (waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    with_layout(s, [&](auto L) {
        using LT = decltype(L);
        SDDMM_LAUNCH(c, (k_flat<LT>), xcd_grid(nblocks), BLOCK,
                           (const void *)c->dA, (const void *)c->dB, s.KU, c->d_rowidx, c->d_col, c->d_sval, c->dP,
                           c->nnz, cpw, nblocks);
    });
}
