// CPU checks of the projections' plan (linear_plan.hpp).
#include <cstdio>

#include "linear_plan.hpp"

static int failures = 0;
#define CHECK(c, ...)                              \
    do {                                           \
        if (!(c) && failures++ < 20) {             \
            std::printf("FAIL %s: ", #c);          \
            std::printf(__VA_ARGS__);              \
            std::printf("\n");                     \
        }                                          \
    } while (0)

int main() {
    using namespace mx;
    // K an odd multiple of 32 runs on the tiles of 256 rows wherever the next multiple of 64 does and no 128-column shape
    // is in question
    for (int M : {300, 1024, 1500, 2048, 4096})
        for (int N : {1280, 4096, 6144, 14336})
            for (int K = 32; K <= 16384; K += 64) {
                const int a = linear_plan(M, N, K, 1, SIZE_MAX).cfg, b = linear_plan(M, N, K + 32, 1, SIZE_MAX).cfg;
                CHECK(kGemmCfgs[b].bm != 256 || kGemmCfgs[a].bm == 256, "%d x %d x %d: shape %d, with K + 32 %d", M, N, K, a, b);
            }
    // some shape takes every K, and none whose loads reach past 32 bits of a tile's first row without 64-bit offsets
    for (int64_t K = 32; K <= INT32_MAX; K = K < 4096 ? K + 32 : K + K / 64 / 32 * 32 + 32) {
        const int i = linear_plan(9, 64, (int32_t)K, 1, SIZE_MAX).cfg;
        CHECK(i >= 0, "K %lld: no shape", (long long)K);
        if (i >= 0 && !kGemmCfgs[i].wide)
            CHECK((std::max(kGemmCfgs[i].bm, kGemmCfgs[i].bn) - 1) * (K + 63) / 64 * 128 + 2 * kGemmCfgs[i].bk <= UINT32_MAX, "K %lld: shape %d",
                  (long long)K, i);
    }
    std::printf("%d failures\n", failures);
    return failures != 0;
}
