// Launch shapes of the f32-faithful matrix-core GEMV (gemv_f32mma.hip): host
// arithmetic only.
#pragma once

#include <algorithm>
#include <cstddef>

namespace ribn_amd {

// Launch shape of one product: compute waves per workgroup, the K split and
// the row groups. The split comes from the weight shape alone (row tiles,
// super-blocks and the partial room a 64-member launch needs), never from the
// member count, so a member's sums are added in the same order whatever the
// batch: among the one-tile-per-wave shapes whose grid fits the CUs in one
// round (all workgroups resident at once), the one with the fewest (row tile
// x super-block) units per workgroup sets it (ties: more compute waves, which
// share the LDS fragments, then fewer splits). Measured on MI355X at the
// Qwen3-8B FFN shapes, two row tiles per wave (halving the LDS fragment
// reads) ran M = 64 slower: 96.0 against 80.3 us per FFN.
struct F32MmaShape {
    int waves, splits, split_blocks, groups;
};
constexpr int kF32MmaMaxComputeWaves = 7;  // plus the loader: eight waves, two per SIMD
inline F32MmaShape f32mma_split(int tiles, int nb, int max_splits, int cu_count) {
    constexpr int kMaxWaves = kF32MmaMaxComputeWaves;
    F32MmaShape best{kMaxWaves, 1, nb, (tiles + kMaxWaves - 1) / kMaxWaves};
    long best_cost = -1;
    for (int s = 1; s <= std::min(nb, std::max(1, max_splits)); ++s) {
        const int sbk = (nb + s - 1) / s;
        if ((nb + sbk - 1) / sbk != s) continue;  // the same split as a smaller s
        for (int w = 1; w <= kMaxWaves; ++w) {
            const int groups = (tiles + w - 1) / w;
            if ((long)groups * s > cu_count) continue;
            const long cost = (long)w * sbk;
            const bool better = best_cost < 0 || cost < best_cost ||
                                (cost == best_cost && (w > best.waves || (w == best.waves && s < best.splits)));
            if (better) {
                best = {w, s, sbk, groups};
                best_cost = cost;
            }
        }
    }
    return best;
}
// The same split with R row tiles per wave (gate/up pairs: 2): the fewest
// compute waves that still fit the grid in one round.
inline F32MmaShape f32mma_shape_r(const F32MmaShape& one, int tiles, int R, int cu_count) {
    const int units = (tiles + R - 1) / R;
    const int max_groups = std::max(1, cu_count / one.splits);
    const int w = std::min(kF32MmaMaxComputeWaves, std::max(1, (units + max_groups - 1) / max_groups));
    return {w, one.splits, one.split_blocks, (units + w - 1) / w};
}

// K splits whose sums of one launch's members the partial room holds (at most 16).
inline int f32mma_max_splits(int launch_members, int rows, size_t partial_bytes) {
    return (int)std::min<size_t>(16, partial_bytes / ((size_t)launch_members * (size_t)rows * 4));
}

// Whether two waves share a unit of a gate/up pair of two or four member tiles:
// where a workgroup holds one unit, and for Q4_K at four tiles. Measured, gate/up
// at 24 / 64 members, us, one wave a unit / two: 4096 -> 2 x 4096 (one unit) Q4_K
// 21.9 / 20.7 and 31.0 / 26.9, Q6_K 42.9 / 40.4 and 82.5 / 77.7; 4096 -> 2 x 12288
// (three) Q4_K 32.7 / 37.0 and 48.4 / 46.7, Q5_K 38.2 / 45.4 and 54.2 / 55.7. (Single
// products were slower with two at every shape tried.)
inline bool f32mma_two_waves(bool q4_k, int member_tiles, const F32MmaShape& sh) {
    return sh.waves == 1 || (q4_k && member_tiles == 4 && 2 * sh.waves + 1 <= kF32MmaMaxComputeWaves + 1);
}

}  // namespace ribn_amd
