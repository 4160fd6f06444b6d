// Rules of the plan that are arithmetic alone: no HIP, so that a host program can check them (tests/host/test_plan_rules.cpp).
// constexpr functions run on the device as well.
#pragma once
#include <cstdint>

namespace sddmm {

// ---- 8-row panels ---------------------------------------------------------------------------
constexpr int PANEL_COLUMNS = 512;             // columns of a panel's work item, at the most

// Columns of a work item of the fused call: a panel of up to 1 024 columns is one item, or two where that leaves wavefronts
// of the chip something to do (halves_from: from more columns on; 0: not).  The items of a panel add their part of the
// output rows atomically to zeros: two sums come out the same in either order, three do not.
constexpr int fused_panel_columns(int len, int halves_from) {
    return halves_from && len > halves_from && len <= 2 * PANEL_COLUMNS ? ((len + 1) / 2 + 31) / 32 * 32 : PANEL_COLUMNS;
}
// Two items per panel as long as a wavefront takes one of them each (wavefronts_per_simd of the fused kernel: 3, 2 and 1 at
// 32, 64 and 128 components), of more than 64 columns, in 16 bits of more than 128.  Whole panels / halves: 250 panels of 240
// columns K = 32 15.8 / 12.8 us, K = 128 32.1 / 22.6; 500 K = 128 33.1 / 24.1, fp16 25.5 / 22.8; 1 000 K = 64 28.7 / 22.2,
// K = 128 fp16 29.6 / 37.2; 1 500 K = 32 21.3 / 19.5, K = 64 fp16 22.1 / 26.4; 1 000 of 104 K = 64 19.4 / 16.4, fp16 15.8 /
// 16.9.  (Items of 64 columns, which made O differ from run to run: 100 of 500 K = 32 12.1 where halves take 15.8, 1 000 of
// 240 K = 128 54.)
constexpr int fused_halves_from(int64_t panels, int wavefronts_per_simd, bool half_width) {
    return 2 * panels <= (int64_t)1024 * wavefronts_per_simd ? (half_width ? 128 : 64) : 0;
}

}  // namespace sddmm
