// The rules of csrc/plan_rules.h: what the kernels and the launches rely on.  No GPU, no HIP.
#include "plan_rules.h"

#include <cstdio>
#include <initializer_list>

using namespace sddmm;

static int failures = 0;
#define CHECK(cond, ...)                                                        \
    do {                                                                        \
        if (!(cond)) {                                                          \
            ++failures;                                                         \
            std::printf("FAILED %s:%d: %s: ", __FILE__, __LINE__, #cond);       \
            std::printf(__VA_ARGS__);                                           \
            std::printf("\n");                                                  \
        }                                                                       \
    } while (0)

static void panels() {
    for (int steps : {1, 2, 4, 6, 8, 12, 16})
        for (bool half : {false, true})
            for (int64_t n : {1, 7, 100, 255, 256, 257, 512, 513, 1000, 1024, 1025, 1280, 1281, 1536, 1537, 4500, 1000000})
                for (int64_t average : {0, 1, 16, 63, 64, 65, 104, 127, 128, 160, 240, 480, 481, 5000}) {
                    const int columns = panel_columns(steps, half, n, average);
                    CHECK(columns >= 64 && columns <= PANEL_COLUMNS, "%d columns", columns);
                    CHECK(columns % 64 == 0, "%d columns", columns);
                    if (n > (steps <= 2 && !half ? 2560 : 1920)) CHECK(columns == PANEL_COLUMNS, "%d panels fill the chip", (int)n);
                    // no more items than wavefronts
                    const int64_t items = n * ((average + columns - 1) / columns), whole = n * ((average + PANEL_COLUMNS - 1) / PANEL_COLUMNS);
                    CHECK(items <= 5120 || items <= whole, "%d items of %d panels of %d columns", (int)items, (int)n, (int)average);
                }
    CHECK(panel_columns(8, false, 1000, 240) == 128 && panel_columns(2, true, 1000, 240) == 128, "1 000 panels of 240");
    for (int steps : {2, 4, 8}) CHECK(panel_columns(steps, false, 2000, 160) == PANEL_COLUMNS, "2 000 panels");
    // steps of 64 columns that go into the items without a rest
    for (int steps : {1, 2, 4, 8}) CHECK(panel_columns(steps, false, 1333, 360) == 128, "%d steps, 1 333 panels of 360", steps);
    CHECK(panel_columns(2, false, 2000, 240) == 128 && panel_columns(8, false, 2000, 240) == PANEL_COLUMNS, "2 000 of 240");
    CHECK(panel_columns(2, false, 1700, 160) == 64 && panel_columns(2, false, 1000, 240) == 128, "items of 64 columns");
    CHECK(panel_columns(2, true, 1333, 360) == 192 && panel_columns(12, false, 1333, 360) == PANEL_COLUMNS, "16 bits, long rows");
    CHECK(panel_columns(2, false, 2523, 288) == 192 && panel_columns(2, false, 1555, 448) == 256, "a rest of one step");
}

// A matrix whose strips all hold the same number of entries per tile, on either side of the line.
static void tiles_or_panels() {
    CHECK(panels_below(4, false, 250, 200000) == 176 && panels_below(16, false, 4000, 11000000) == 176, "split K");
    CHECK(panels_below(4, false, 4000, 11000000) == 192 && panels_below(2, false, 250, 200000) == 187, "many entries, short rows");
    CHECK(panels_below(4, false, 1000, 1200000) == 144 && panels_below(4, false, 2000, 1200000) == 176, "a chip that whole panels do not fill");
    CHECK(panels_below(16, true, 250, 200000) == 0 && panels_below(16, true, 1000, 4100000) == 0, "16 bits, 1 KiB");
    CHECK(panels_below(16, true, 4000, 11000000) == 176 && panels_below(8, true, 1000, 1200000) == 0, "16 bits");
    CHECK(panels_below(4, true, 250, 200000) == 176 && panels_below(4, true, 600, 500000) == 0, "16 bits, 256 bytes");
    CHECK(long_panels_below(true, 100000000) == 0 && long_panels_below(false, 700000) == 0, "long rows");
    CHECK(long_panels_below(false, 1200000) == 144 && long_panels_below(false, 1800000) == 192, "long rows, many entries");
    CHECK(panels_below(1, false, 6000, 6000 * 8 * 47) == 0 && panels_below(1, false, 6000, 6000 * 8 * 48) == 187, "short lists");
}

static void fused_panels() {
    for (int from : {0, 64, 128})
        for (int len = 1; len <= 5000; ++len) {
            const int columns = fused_panel_columns(len, from), items = (len + columns - 1) / columns;
            CHECK(columns >= 32 && columns % 32 == 0 && columns <= PANEL_COLUMNS, "%d columns, %d", len, columns);
            if (len <= 1024) CHECK(items <= 2, "%d columns in %d items", len, items);
            if (len <= 1024 && from && len > from) CHECK(items == 2, "%d columns in %d items", len, items);
        }
    CHECK(fused_halves_from(1536, 3, false) == 64 && fused_halves_from(1537, 3, false) == 0, "three wavefronts per SIMD");
    CHECK(fused_halves_from(512, 1, true) == 128 && fused_halves_from(513, 1, true) == 0, "one wavefront per SIMD");
}

// A launch of few short steps never pays for a longer plan; longer rows and more entries do.
static void rows_of_any_length() {
    int64_t before = INT64_MAX;
    for (int steps : {1, 2, 4, 6, 8, 12, 16}) {
        CHECK(ragged_entries(steps) <= before, "%d steps", steps);
        before = ragged_entries(steps);
        for (bool half : {false, true}) CHECK(ragged_gathered_entries(steps, half) * steps <= 1 << 24, "%d steps", steps);
    }
    CHECK(ragged_entries(1) > 5 << 19 && ragged_entries(2) > 825600 && ragged_entries(4) > 338688, "rows of up to 256 bytes");
    CHECK(ragged_entries(1) <= 3840000 && ragged_entries(2) <= 1199872 && ragged_entries(4) <= 480000, "where few launches gain what the look costs");
    CHECK(ragged_entries(6) <= 331264 && ragged_entries(8) <= 96000, "longer rows");
    CHECK(ragged_gathered_entries(6, false) <= 1960000 && ragged_gathered_entries(8, false) > 1960000, "near-dense rows");
    CHECK(ragged_gathered_entries(4, true) <= 1960000 && ragged_gathered_entries(4, false) > 1306340, "near-dense rows, 16 bits");
    CHECK(long_row_entries(1200) == 1 << 18 && long_row_entries(2048) > 272000 && long_row_entries(4000) <= 287744, "beyond 1 KiB");
}

// Rows of every length: a power of two that divides `most` (the lanes of a row), the bound that sizes the list of segments.
static void column_blocks() {
    for (bool sorted : {false, true})
        for (int longest : {257, 1023, 1024, 4096, 100000}) {
            const int least = row_blocks_least(sorted), most = row_blocks_most(sorted, longest);
            CHECK(most >= least && most <= COL_BLOCKS_MAX && most % least == 0, "%d", longest);
            for (int len = 257; len <= longest; len += len / 50 + 1) {
                const int n = row_blocks(len, least, most);
                CHECK(n >= least && most % n == 0, "%d blocks of a row of %d", n, len);
                CHECK(n == least || len >= n * COL_BLOCK_ENTRIES, "%d blocks of a row of %d", n, len);
                CHECK(row_block_segments(7, 7 * (int64_t)len, 256, sorted, longest) >= 7 * (len / 256 + n), "row of %d", len);
                if (sorted) CHECK(n == 16, "sorted entries, %d blocks of a row of %d", n, len);
            }
        }
}

// A total outside of the reported ones (those of the column blocks lie behind them) has no place in the report.
static void reported_totals() {
    unsigned long long counters[16];
    for (int i = 0; i < 16; ++i) CHECK(scan_total_slot(&counters[i], &counters[2], 7) == (i >= 2 && i < 9 ? i - 2 : -1), "%d", i);
}

int main() {
    reported_totals();
    rows_of_any_length();
    tiles_or_panels();
    panels();
    column_blocks();
    fused_panels();
    std::printf("%d failed\n", failures);
    return failures != 0;
}
