// How a projection of more than kLinearGemvMaxRows rows runs: the GEMM's tile shapes, their costs, and the choice among
// them. Host code only, apart from linear.hip so that CPU tests can evaluate it.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "mx_kernels.hpp"

namespace mx {

// The GEMM's tile shapes and what a product costs on each, in microseconds, fitted (least relative squares, 8 % rms) to
// 4700 measured launches: 9 to 4096 rows of the decoders' projections, every shape with 1 to 12 parts of K.
//   t = 4.5 + 0.2 M K / 1e6 (staging) + 1.06 M N / 1e6 (output)                       the same for every shape
//     + rounds * (tile + steps * step)     steps of 64 columns per part; a round is one workgroup per CU, or two where
//                                          per_cu is 2 (a part round of at most one per CU takes step1, else step2)
//     + (parts > 1) * (merge * (1 + parts * tile bytes / 64 KB) + part_mb * partial MB)
// Picking the cheapest is within 1.1 % of the measured best on average over those products (the worst 19 %). What the
// split buys, against the 128 x 128 tiles with whole K that took every product of few tiles (us, staging included):
// 24 x 4096 x 4096 47.9 -> 12.9, 64 x 4096 x 4096 49.0 -> 15.3, 256 x 4096 x 4096 51.0 -> 24.6, 24 x 4096 x 14336
// 147 -> 29.4, 512 x 1152 x 896 19.1 -> 10.0, 1024 x 3584 x 3584 50.2 -> 46.
struct GemmCfg {
    int bm, bn, bk, per_cu;
    float step1, step2, tile, merge, part_mb;
    bool wide = false;  // 64-bit offsets within a tile
};
constexpr int kGemmCUs = 256;
constexpr int kGemmBigRows = 256;  // rows of the tiles of 8 waves, which take whole K only
constexpr int kMaxParts = 12, kMaxSplitGrid = 1024;  // the fitted range
constexpr GemmCfg kGemmCfgs[] = {
    {16, 64, 128, 1, 0.219f, 0.f, 0.315f, 0.539f, 1.588f},
    {32, 64, 128, 2, 0.250f, 0.402f, 0.f, 0.899f, 0.522f},
    {64, 64, 64, 2, 0.340f, 0.553f, 0.f, 0.920f, 0.415f},
    {128, 64, 128, 1, 0.421f, 0.f, 1.094f, 0.765f, 0.348f},
    {128, 128, 64, 1, 0.640f, 0.f, 2.207f, 0.930f, 0.203f},
    {128, 128, 64, 2, 0.887f, 1.078f, 0.f, 1.092f, 0.306f},
    {256, 192, 64, 1, 1.243f, 0.f, 5.946f, 0.f, 0.f},
    {256, 256, 64, 1, 1.426f, 0.f, 8.941f, 0.f, 0.f},
    {64, 64, 64, 2, 0.340f, 0.553f, 0.f, 0.920f, 0.415f, true},
};
constexpr int kNumGemmCfgs = sizeof kGemmCfgs / sizeof *kGemmCfgs;

// Whether the bytes from a tile's first row to any of its loads fit 32 bits.
inline bool gemm_offsets_fit(const GemmCfg & c, int32_t K) {
    return ((uint64_t)std::max(c.bm, c.bn) - 1) * (((uint64_t)K + 63) / 64 * 128) + 2 * c.bk <= UINT32_MAX;
}
// Whether shape c takes a K (a multiple of 32): the 64-column shapes take any that its offsets allow, and the wide one the
// rest (K above 34 million), so that some shape always applies.
inline bool gemm_takes(const GemmCfg & c, int32_t K) {
    return K % (c.bk == 128 ? 128 : 32) == 0 && gemm_offsets_fit(c, K) != c.wide;
}

// counters of a split GEMM, each on a 256-byte line of its own
inline size_t linear_counter_bytes(const LinearPlan & l) { return l.splits > 1 ? (size_t)l.tiles * kCounterStride * 4 : 0; }

// The plan of tile shape cfg with K in the given number of parts.
inline LinearPlan linear_plan_of(int cfg, int splits, int32_t M, int32_t N, int32_t count) {
    const GemmCfg & c = kGemmCfgs[cfg];
    const int64_t tiles = count * (((int64_t)N + c.bn - 1) / c.bn) * (((int64_t)M + c.bm - 1) / c.bm);
    LinearPlan l{cfg, splits, (int32_t)tiles, 0};
    if (splits > 1) l.bytes = (size_t)l.tiles * splits * c.bm * c.bn * 4 + linear_counter_bytes(l);
    return l;
}

// avail: workspace bytes behind the staged rows that the plan may use
inline LinearPlan linear_plan(int32_t M, int32_t N, int32_t K, int32_t count, size_t avail) {
    LinearPlan best{-1, 1, 0, 0};
    float best_t = 0.f;
    for (int i = 0; i < kNumGemmCfgs; i++) {
        const GemmCfg & c = kGemmCfgs[i];
        if (!gemm_takes(c, K)) continue;
        const int ksteps = (K + c.bk - 1) / c.bk;
        const int64_t tiles = linear_plan_of(i, 1, M, N, count).tiles;
        const int most = c.merge > 0.f ? (int)std::min<int64_t>(std::min(kMaxParts, ksteps), kMaxSplitGrid / tiles) : 1;
        for (int s = 1; s <= std::max(most, 1); s++) {
            const LinearPlan l = linear_plan_of(i, s, M, N, count);
            if (l.bytes > avail) break;
            const int64_t wgs = tiles * s, slots = (int64_t)kGemmCUs * c.per_cu, full = wgs / slots, rem = wgs % slots;
            const float steps = (float)((ksteps + s - 1) / s) * (float)(c.bk / 64);
            const float n1 = (float)((c.per_cu == 1 ? full : 0) + (rem > 0 && rem <= kGemmCUs ? 1 : 0));
            const float n2 = (float)((c.per_cu == 1 ? 0 : full) + (rem > kGemmCUs ? 1 : 0));
            float t = (n1 + n2) * c.tile + steps * (n1 * c.step1 + n2 * c.step2);
            if (s > 1) {
                const int64_t part = (int64_t)c.bm * c.bn * 4;
                t += c.merge * (1.f + (float)(s * part) / 65536.f) + c.part_mb * (float)(tiles * s * part) * 1e-6f;
            }
            if (best.cfg < 0 || t < best_t) {
                best = l;
                best_t = t;
            }
        }
    }
    return best;
}

// The most that linear_plan takes behind the staged rows of a product of up to M rows. It does not grow with M (a product of
// few rows has more parts), and depends on M through the tiles alone, so every 16th row count is looked at, up to the
// last one at which some shape could be split.
inline size_t linear_plan_room(int32_t M, int32_t N, int32_t K, int32_t count) {
    int64_t top = 0;
    for (const GemmCfg & c : kGemmCfgs)
        if (c.merge > 0.f) top = std::max(top, c.bm * (kMaxSplitGrid / 2 / (count * (((int64_t)N + c.bn - 1) / c.bn))));
    size_t room = 0;
    for (int32_t m = (int32_t)std::min<int64_t>(M, top); m > kLinearGemvMaxRows; m = (m - 1) / 16 * 16)
        room = std::max(room, linear_plan(m, N, K, count, SIZE_MAX).bytes);
    return room;
}

}  // namespace mx
