// CPU check of the GEMMs' operand loads (mx_kernels.hpp: gemm_block_row, gemm_block_chunk, gemm_load_offset, gemm_half_back),
// from which every tile shape forms its addresses: over operands of 1 to 600 rows and several K, each load of each tile and
// step stays inside the row that it is for (rows past the last repeat it), reads that row's columns of its step, or for
// columns past K columns of the same row, and the lanes' loads fill every chunk of the tile once, where the swizzled
// operand reads look for it. Offsets are formed in 32 bits and compared with 64.
#include <cstdio>
#include <set>

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

// One operand's tiles of `tile` rows: weights (columns past K go back) or staged rows (zero-padded to kp columns).
template <int BK>
static void operand(int tile, int rows, int K, bool weights) {
    const int kp = (K + BK - 1) / BK * BK, stride = weights ? K : kp, blocks = tile * BK / 512;
    for (int first = 0; first < rows; first += tile) {
        std::set<int> filled;
        for (int block = 0; block < blocks; block++)
            for (int lane = 0; lane < 64; lane++) {
                const int row = mx::gemm_block_row<BK>(block, lane), chunk = mx::gemm_block_chunk<BK>(block, lane);
                CHECK(row >= 0 && row < tile && chunk >= 0 && chunk < BK / 8, "tile %d BK %d block %d lane %d", tile, BK, block, lane);
                // 16-byte slot in LDS of the lane, and where the operand reads look for (row, chunk)
                CHECK(block * 64 + lane == row * (BK / 8) + (chunk ^ mx::gemm_swizzle<BK>(row % 32)), "tile %d BK %d row %d chunk %d", tile, BK, row, chunk);
                filled.insert(row * 1000 + chunk);
                const int r = first + row < rows ? first + row : rows - 1;
                for (int step = 0; step < kp / BK; step++) {
                    const bool past = weights && step * BK + 8 * chunk >= K;
                    const uint32_t off = mx::gemm_load_offset<uint32_t>(first, row, rows, stride, chunk) -
                                         (weights && step * BK + BK > K ? mx::gemm_half_back(chunk) : 0);
                    const int64_t at = (int64_t)first * stride * 2 + (int64_t)step * BK * 2 + off - (int64_t)r * stride * 2;
                    const int64_t want = 2 * (step * BK + 8 * chunk);
                    CHECK(past ? at >= 0 && at + 16 <= 2 * K : at == want, "tile %d BK %d rows %d K %d weights %d: row %d chunk %d step %d reads byte %lld of row %d",
                          tile, BK, rows, K, weights, row, chunk, step, (long long)at, r);
                }
                CHECK(mx::gemm_load_offset<uint32_t>(first, row, rows, stride, chunk) == mx::gemm_load_offset<uint64_t>(first, row, rows, stride, chunk), "32 bits");
            }
        CHECK((int)filled.size() == tile * BK / 8, "tile %d BK %d: %zu chunks filled", tile, BK, filled.size());
    }
}

int main() {
    using namespace mx;
    for (const GemmCfg & c : kGemmCfgs)
        for (int rows = 1; rows <= 600; rows += rows < 40 ? 1 : 7)
            for (int K : {32, 64, 96, 128, 160, 384}) {
                if (!gemm_takes(c, K)) continue;
                for (bool weights : {false, true}) {
                    const int tile = weights ? c.bn : c.bm;
                    if (c.bk == 128) operand<128>(tile, rows, K, weights);
                    else operand<64>(tile, rows, K, weights);
                }
            }
    // the shapes with 32-bit offsets at the largest K that they take: the last chunk of a full tile's last row
    for (const GemmCfg & c : kGemmCfgs) {
        if (c.wide) continue;
        int32_t K = 0;
        for (int32_t step = 1 << 30; step >= c.bk; step /= 2)
            if (K + (int64_t)step <= INT32_MAX / 128 * 128 && gemm_takes(c, K + step)) K += step;
        const int tile = c.bm > c.bn ? c.bm : c.bn;
        CHECK(gemm_load_offset<uint32_t>(0, tile - 1, tile, K, c.bk / 8 - 1) == gemm_load_offset<uint64_t>(0, tile - 1, tile, K, c.bk / 8 - 1),
              "%d x %d at K %d", c.bm, c.bn, K);
    }
    std::printf("%d failures\n", failures);
    return failures != 0;
}
