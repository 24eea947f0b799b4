"""Launch shapes of the three-way plans (poyd_amd/csrc/poyg_cube.h): the block
kernels count workgroups of eight waves, or of two for batches of small triples;
the chunked kernel, whose workgroup is one wave, waves.  The header is plain
C++; the test compiles a small checker with g++."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "poyd_amd", "csrc")

CHECKER = r'''
#include <cstdio>
#include "poyg_cube.h"
using namespace poyg;
// lines: triples, compute units, asked waves, one workgroup a unit, group waves -> rows, fill; or, with 0 group
// waves, kinds and then count, planes, lines of each -> waves of a workgroup
int main() {
  int n, cus, waves, one, group;
  while (scanf("%d %d %d %d %d", &n, &cus, &waves, &one, &group) == 5) {
    if (group) {
      const CubeGrid g = cube_grid(n, cus, waves, one != 0, group);
      printf("%d %d\n", g.rows, g.fill);
      continue;
    }
    std::vector<CubeRows> r;
    int kinds, count, planes, lines;
    if (scanf("%d", &kinds) != 1) return 1;
    while (kinds-- && scanf("%d %d %d", &count, &planes, &lines) == 3) r.insert(r.end(), count, CubeRows{planes, lines});
    printf("%d\n", cube_group_waves(r, cus, waves, one != 0));
  }
  return 0;
}
'''

STEPS = r'''
#include <cstdio>
#include "poyg_cube.h"
using namespace poyg;
int main() {
  long bad = 0, tot = 0;
  for (int waves = 1; waves <= 8; waves *= 2)
    for (int n1 = 1; n1 < 60; ++n1)
      for (int n2 = 1; n2 < 60; ++n2) {
        long c = n2;   // plane by plane, chunk by chunk
        for (int p = 1; p < n1; ++p)
          for (int r = 0; r < n2; r += std::min(p + 1, 2 * waves)) ++c;
        bad += c != cube_chunks(CubeRows{n1, n2}, waves);
        ++tot;
      }
  printf("%ld %ld\n", tot, bad);
  return 0;
}
'''


def build(tmp_path, name, text):
    src, exe = tmp_path / (name + ".cpp"), tmp_path / name
    src.write_text(text)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    return str(exe)


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_cube_launch_shapes(tmp_path):
    exe = build(tmp_path, "grid", CHECKER)
    cases = {(100000, 256, 0, 0, 8): (512, 2048), (100000, 256, -1, 1, 8): (256, 2048), (100000, 256, 16, 0, 8): (512, 4096),
             (100000, 256, 16, 1, 8): (256, 4096), (100000, 256, 24, 0, 8): (768, 6144), (100000, 256, 4, 0, 8): (256, 1024),
             (1000, 256, 0, 0, 8): (512, 1000), (7, 256, 0, 0, 8): (7, 7), (0, 256, 0, 0, 8): (1, 1),
             (5000, 1, 1, 0, 8): (1, 1), (100000, 256, 0, 0, 2): (2048, 2048), (100000, 256, 0, 1, 2): (1024, 2048),
             (100000, 256, 4, 0, 2): (512, 1024)}
    out = subprocess.run([exe], input="".join("%d %d %d %d %d\n" % c for c in cases), check=True,
                         capture_output=True, text=True).stdout.split()
    assert list(zip(map(int, out[0::2]), map(int, out[1::2]))) == list(cases.values())


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_cube_workgroup_size(tmp_path):
    tot, bad = map(int, subprocess.run([build(tmp_path, "steps", STEPS)], check=True, capture_output=True,
                                       text=True).stdout.split())
    assert tot > 10000 and bad == 0
    exe = build(tmp_path, "grid", CHECKER)
    # few triples, or one long one among many: eight waves; many small ones: two
    cases = [([(1, 300, 300)], 8), ([(512, 30, 30)], 8), ([(1024, 300, 300)], 8), ([(20000, 6, 6)], 2), ([(4096, 20, 20)], 2),
             ([(2048, 100, 100)], 2), ([(1024, 100, 100)], 8), ([(4096, 40, 40), (1, 500, 500)], 8), ([(5, 1, 1)], 8), ([], 8)]
    text = "".join("0 256 0 0 0 %d %s\n" % (len(k), " ".join("%d %d %d" % x for x in k)) for k, _ in cases)
    out = subprocess.run([exe], input=text, check=True, capture_output=True, text=True).stdout.split()
    assert list(map(int, out)) == [w for _, w in cases]
