// Launch shape of the three-way fills (poyg_cube.hip).  Plain C++ (no HIP), so
// that a CPU test can check it.
#pragma once

#include <algorithm>

namespace poyg {

constexpr int kCubeWaves = 8;   // waves of a block kernel's workgroup (one triple)

// Workgroups of a plan: `rows` of the block kernels (kCubeWaves waves each),
// `fill` of the chunked kernel, whose workgroup is one wave with a triple of its
// own.  waves_per_cu: resident waves per compute unit, 0 or less for the
// defaults: 16 for the block kernels (cube_packed_kernel<16> holds one workgroup
// a compute unit), 8 for the chunked one.  4,096 triples of 30 x 30 x 1,100 in
// the chunked kernel take 32 ms with 8 waves a compute unit, 82 with 2; 600 of
// them 11 and 20.
struct CubeGrid {
  int rows, fill;
};

inline CubeGrid cube_grid(int n, int cus, int waves_per_cu, bool one_per_cu) {
  const int waves = waves_per_cu > 0 ? waves_per_cu : 2 * kCubeWaves;
  const int groups = std::max(1, waves / kCubeWaves);
  const int chunked = waves_per_cu > 0 ? waves_per_cu : 8;
  return CubeGrid{std::max(1, std::min(n, cus * (one_per_cu ? 1 : groups))),
                  std::max(1, std::min(n, cus * chunked))};
}

}  // namespace poyg
