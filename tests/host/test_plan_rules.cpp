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

int main() {
    fused_panels();
    std::printf("%d failed\n", failures);
    return failures != 0;
}
