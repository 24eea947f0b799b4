"""Launch shapes of the three-way plans (poyd_amd/csrc/poyg_cube.h): the block
kernels count workgroups of eight waves, the chunked kernel, whose workgroup is
one wave, waves.  The header is plain C++; the test compiles a small checker
with g++."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "poyd_amd", "csrc")

CHECKER = r'''
#include <cstdio>
#include "poyg_cube.h"
int main() {
  int n, cus, waves, one;
  while (scanf("%d %d %d %d", &n, &cus, &waves, &one) == 4) {
    const poyg::CubeGrid g = poyg::cube_grid(n, cus, waves, one != 0);
    printf("%d %d\n", g.rows, g.fill);
  }
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_cube_launch_shapes(tmp_path):
    src, exe = tmp_path / "grid.cpp", tmp_path / "grid"
    src.write_text(CHECKER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    cases = {(100000, 256, 0, 0): (512, 2048), (100000, 256, -1, 1): (256, 2048), (100000, 256, 16, 0): (512, 4096),
             (100000, 256, 16, 1): (256, 4096), (100000, 256, 24, 0): (768, 6144), (100000, 256, 4, 0): (256, 1024),
             (1000, 256, 0, 0): (512, 1000), (7, 256, 0, 0): (7, 7), (0, 256, 0, 0): (1, 1), (5000, 1, 1, 0): (1, 1)}
    out = subprocess.run([str(exe)], input="".join("%d %d %d %d\n" % c for c in cases), check=True,
                         capture_output=True, text=True).stdout.split()
    assert list(zip(map(int, out[0::2]), map(int, out[1::2]))) == list(cases.values())
