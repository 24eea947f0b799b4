"""Host geometry of the diagonal linear fill (poyd_amd/csrc/poyg_lindiag.h):
the diagonals it is given are exactly the cells of lin_row_host's rows
(src/algn.c:872-968) in all three band cases, whatever the band parameter, and
a plain walk over its pairs, times and shared halves reaches each of them.
The header is plain C++; the test compiles a small checker with g++."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "poyd_amd", "csrc")

CHECKER = r'''
#include <cstdio>
#include "poyg_lindiag.h"
using namespace poyg;
int main() {
  long bad = 0, tot = 0, cases[3] = {0, 0, 0}, refused = 0;
  for (int n = 2; n <= 260; n += (n < 12 ? 1 : 7))
    for (int m = n; m <= n + 500; m += (m < n + 20 ? 1 : 23))
      for (int dw = -60; dw <= 150; dw += 7) {
        const LinGeom g = lin_geom(m, n, dw);
        ++tot;
        if (!lin_diag_fits(m, n, g)) { ++refused; continue; }
        ++cases[g.cs];
        int dlo, dhi;
        lin_diag_range(m, n, g, dlo, dhi);
        if (dlo > 0 || dhi < 0 || n - m < dlo || n - m > dhi) ++bad;
        for (int i = 0; i < m; ++i) {
          int lo, hi;
          lin_row_host(i, m, n, g, lo, hi);
          if (lo != std::max(0, i + dlo) || hi != std::min(n - 1, i + dhi)) { ++bad; break; }
        }
        // pair and time of both corners; the last time step's group is stored
        const int L0 = (-dlo) >> 1, rel = n - m - dlo, Lend = rel >> 1, T = m - 1 - L0 + Lend;
        if (T < 1 || T - Lend + L0 != m - 1 || T + Lend + L0 + dlo + (rel & 1) != n - 1) ++bad;
        const int pairs = (dhi - dlo) / 2 + 1;
        const int w = lin_diag_waves(dlo, dhi), r = lin_diag_regs(dlo, dhi);
        if (w && (kLinDiagStep * (w - 1) + 128 < pairs || (w > 1 && kLinDiagStep * (w - 2) + 128 >= pairs))) ++bad;
        if (r && 128 * r < pairs) ++bad;
        if (w && 2 * lin_diag_cols(true, w) < pairs) ++bad;
        if (r && lin_diag_bytes(m, n, dlo, lin_diag_cols(false, r)) < (int64_t)((T + 7) / 8) * 64 * r * 8) ++bad;
      }
  printf("%ld %ld %ld %ld %ld %ld\n", tot, bad, refused, cases[0], cases[1], cases[2]);
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_diagonals_equal_row_walk(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECKER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    tot, bad, refused, full, case2, case3 = map(int, subprocess.run([str(exe)], check=True, capture_output=True,
                                                                     text=True).stdout.split())
    assert bad == 0 and tot > 10000
    assert full > 0 and case2 > 0 and case3 > 0
