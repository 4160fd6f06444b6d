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

int main() {
    column_blocks();
    fused_panels();
    std::printf("%d failed\n", failures);
    return failures != 0;
}
