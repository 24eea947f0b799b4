// Launch shape of the three-way fills (poyg_cube.hip).  Plain C++ (no HIP), so
// that a CPU test can check it.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <vector>

namespace poyg {

constexpr int kCubeWaves = 8;   // waves of a block kernel's workgroup (one triple) ...
constexpr int kCubeFew = 2;     // ... for batches of small triples

// Waves per compute unit of the block kernels: the asked ones, or 16;
// cube_packed_kernel<16> has registers for 8.
inline int cube_block_waves(int waves_per_cu, bool one_per_cu) {
  return one_per_cu ? kCubeWaves : waves_per_cu > 0 ? waves_per_cu : 2 * kCubeWaves;
}

// Planes and lines of a triple, and the chunks of lines (one barrier each) that
// a workgroup of `waves` waves takes them in: the lines of plane 0 one by one,
// those of plane p min(p + 1, 2 waves) at a time.
struct CubeRows {
  int planes, lines;
};
inline int64_t cube_chunks(const CubeRows &r, int waves) {
  const int most = 2 * waves;
  int64_t c = r.lines;
  for (int p = 1; p < std::min(r.planes, most); ++p) c += (r.lines + p) / (p + 1);
  if (r.planes > most) c += (int64_t)(r.planes - most) * ((r.lines + most - 1) / most);
  return c;
}

// Waves of a block kernel's workgroup.  Eight finish a triple soonest; but the
// first planes, and planes of few lines, leave most of them idle, and two waves
// let four times as many triples run.  A launch lasts as long as its longest
// triple or as all chunks shared out over the resident workgroups, whichever is
// longer; a chunk takes about 1.2 us with the one and 1.6 with the other while
// they fill the chip.  Two against eight waves, ms: 20,000 triples of 6 x 6 x 6
// 0.29 against 0.58 (one wave per triple: 0.34), 4,096 of 20 0.43 / 0.65, of 40
// 1.39 / 1.85, 2,048 of 100 4.1 / 4.8; 1,024 of 100 whose costs leave the packed
// kernel's range 4.06 / 3.78.
inline int cube_group_waves(const std::vector<CubeRows> &rows, int cus, int waves_per_cu, bool one_per_cu) {
  int64_t time[2];
  for (int few = 0; few < 2; ++few) {
    const int waves = few ? kCubeFew : kCubeWaves;
    const int64_t groups = (int64_t)cus * std::max(1, cube_block_waves(waves_per_cu, one_per_cu) / waves);
    int64_t longest = 0, all = 0;
    for (const CubeRows &r : rows) {
      const int64_t c = cube_chunks(r, waves);
      longest = std::max(longest, c);
      all += c;
    }
    time[few] = std::max(longest, all / groups);
  }
  return 4 * time[1] < 3 * time[0] ? kCubeFew : kCubeWaves;
}

// Workgroups of a plan: `rows` of the block kernels (group_waves waves each),
// `fill` of the chunked kernel, whose workgroup is one wave with a triple of its
// own.  waves_per_cu: resident waves per compute unit, 0 or less for the
// defaults: cube_block_waves for the block kernels, 8 for the chunked one.  4,096
// triples of 30 x 30 x 1,100 in the chunked kernel take 32 ms with 8 waves a
// compute unit, 82 with 2; 600 of them 11 and 20.
struct CubeGrid {
  int rows, fill;
};

inline CubeGrid cube_grid(int n, int cus, int waves_per_cu, bool one_per_cu, int group_waves) {
  const int groups = std::max(1, cube_block_waves(waves_per_cu, one_per_cu) / group_waves);
  const int chunked = waves_per_cu > 0 ? waves_per_cu : 8;
  return CubeGrid{std::max(1, std::min(n, cus * groups)), std::max(1, std::min(n, cus * chunked))};
}

}  // namespace poyg
