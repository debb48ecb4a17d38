// Prints "units a workgroup, K splits, waves a unit" of a gate/up pair on the f32-faithful
// matrix-core GEMV: f32mma_shape_print TYPE K N MEMBERS CUS PARTIAL_BYTES (member counts of one launch).
#include "f32mma_shape.hpp"

#include <cstdio>
#include <cstdlib>

int main(int argc, char** argv) {
    if (argc != 7) return 2;
    const int type = std::atoi(argv[1]), k = std::atoi(argv[2]), n = std::atoi(argv[3]), members = std::atoi(argv[4]);
    const int cus = std::atoi(argv[5]);
    const int step = type == 14 ? 32 : 64;  // Q6_K: two member tiles a launch
    const int mt = ((members > step ? step : members) + 15) / 16;
    const int tiles = 2 * ((n + 15) / 16);
    const int splits = ribn_amd::f32mma_max_splits(step, 2 * n, std::strtoull(argv[6], nullptr, 10));
    const auto sh = ribn_amd::f32mma_shape_r(ribn_amd::f32mma_split(tiles, k / 256, splits, cus), tiles, 2, cus);
    std::printf("%d %d %d\n", sh.waves, sh.splits, mt % 2 == 0 && ribn_amd::f32mma_two_waves(type == 12, mt, sh) ? 2 : 1);
    return 0;
}
