"""Host geometry of the diagonal linear fill (poyd_amd/csrc/poyg_lindiag.h):
the diagonals it is given are exactly the cells of lin_row_host's rows
(src/algn.c:872-968) in all three band cases, whatever the band parameter, and
the schedule of its workgroup form (the waves' pairs, the origin above a wave
at time 0, the halo exchange) gives every owned cell the plain recurrence's
value.  The header is plain C++; the tests compile small checkers with g++."""
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


# Every wave's pairs, step by step as diag_fill_group takes them: at time T the
# even cells of pair L read their own odd value (above them), the pair below's
# odd value (left) and their own last even one, the odd cells the pair above's
# even value, their own even one and their own last odd one; what lies outside a
# wave is "no cell".  Costs differ from cell to cell, so that any cell that reads
# a wrong or missing neighbour has another value than the plain recurrence.
SCHEDULE = r'''
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "poyg_lindiag.h"
using namespace poyg;
static const int INF = 1 << 29;
static unsigned mix(unsigned a, unsigned b) {
  unsigned x = a * 2654435761u ^ (b + 0x9e3779b9u) * 2246822519u;
  x ^= x >> 15;
  x *= 2654435761u;
  return x >> 13;
}
static int del(int i) { return 1 + mix(i, 77777) % 1000; }
static int ins(int j) { return 1 + mix(99999, j) % 1000; }
static int sub(int i, int j) { return mix(i, j) % 2000; }
int main(int argc, char **argv) {
  // lines: rows, columns, first and last diagonal, time steps to walk (0: all)
  int M, N, dlo, dhi, steps;
  while (scanf("%d %d %d %d %d", &M, &N, &dlo, &dhi, &steps) == 5) {
    const int waves = lin_diag_waves(dlo, dhi), L0 = (-dlo) >> 1, top = (dhi - dlo) >> 1;
    const bool odd_top = (dhi - dlo) & 1;
    const int t_end = M - 1 - L0 + ((N - M - dlo) >> 1);
    const int t_last = steps ? std::min(steps, t_end) : t_end, groups = (t_end + 7) / 8;
    // the plain recurrence over the band, of the rows and columns within reach
    const int rows = std::min(M, 2 * t_last + 4), width = dhi - dlo + 1;
    std::vector<int> ref((size_t)rows * width, INF);
    auto at = [&](int i, int j) -> int & { return ref[(size_t)i * width + (j - i - dlo)]; };
    auto get = [&](int i, int j) { return i < 0 || j < 0 || j - i < dlo || j - i > dhi ? INF : at(i, j); };
    for (int i = 0; i < rows; ++i)
      for (int j = std::max(0, i + dlo); j <= std::min(N - 1, i + dhi); ++j) {
        int v = i == 0 && j == 0 ? 0 : INF;
        v = std::min(v, get(i - 1, j) + del(i));
        v = std::min(v, get(i, j - 1) + ins(j));
        v = std::min(v, get(i - 1, j - 1) + sub(i, j));
        at(i, j) = std::min(v, INF);
      }
    const int P = 128;   // pairs of a wave
    struct Wave { int E[128], O[128]; };
    std::vector<Wave> W(waves);
    long bad = 0, cells = 0, first_i = -1, first_j = -1;
    auto odd_half = [&](int w, int T, int above) {
      Wave &x = W[w];
      const int Lw = kLinDiagStep * w;
      for (int l = 0; l < P; ++l) {
        const int L = Lw + l, i = T - L + L0, j = T + L + L0 + dlo + 1;
        const int up = l + 1 < P ? x.E[l + 1] : above;
        int v = std::min(up + del(i), std::min(x.E[l] + ins(j), x.O[l] + sub(i, j)));
        if (L > top || (L == top && !odd_top)) v = INF;
        x.O[l] = std::min(v, INF);
      }
    };
    auto even_half = [&](int w, int T) {
      Wave &x = W[w];
      const int Lw = kLinDiagStep * w;
      for (int l = P - 1; l >= 0; --l) {
        const int L = Lw + l, i = T - L + L0, j = T + L + L0 + dlo;
        const int left = l ? x.O[l - 1] : INF;
        int v = std::min(x.O[l] + del(i), x.E[l] + sub(i, j));
        if (L <= top) v = std::min(v, left + ins(j));
        x.E[l] = std::min(v, INF);
      }
    };
    auto check = [&](int T) {
      for (int w = 0; w < waves; ++w)
        for (int l = w ? kLinDiagHalo : 0; l < (w < waves - 1 ? P - kLinDiagHalo : P); ++l) {
          const int L = kLinDiagStep * w + l;
          for (int o = 0; o < 2; ++o) {
            const int i = T - L + L0, j = T + L + L0 + dlo + o;
            if (2 * L + o > dhi - dlo || i < 0 || j < 0 || i >= rows || j >= N) continue;
            ++cells;
            if ((o ? W[w].O[l] : W[w].E[l]) != at(i, j)) {
              if (!bad) first_i = i, first_j = j;
              ++bad;
            }
          }
        }
    };
    for (int w = 0; w < waves; ++w) {
      const int Lw = kLinDiagStep * w;
      for (int l = 0; l < P; ++l) {
        W[w].E[l] = !(dlo & 1) && Lw + l == L0 ? 0 : INF;
        W[w].O[l] = INF;
      }
      odd_half(w, 0, lin_diag_origin_above(dlo, Lw + P) ? 0 : INF);
      if (dlo & 1)
        for (int l = 0; l < P; ++l)
          if (Lw + l == L0) W[w].O[l] = 0;
    }
    check(0);
    for (int T = 1; T <= t_last; ++T) {
      for (int w = 0; w < waves; ++w) {
        even_half(w, T);
        odd_half(w, T, INF);
      }
      check(T);
      const int k = (T - 1) / 8;
      if (T % 8 == 0 && k < groups - 1 && lin_diag_exchange(k)) {
        const std::vector<Wave> old = W;
        for (int w = 0; w < waves; ++w)
          for (int q = 0; q < kLinDiagHalo; ++q) {
            if (w > 0) {
              W[w].E[q] = old[w - 1].E[P - 2 * kLinDiagHalo + q];
              W[w].O[q] = old[w - 1].O[P - 2 * kLinDiagHalo + q];
            }
            if (w < waves - 1) {
              W[w].E[P - kLinDiagHalo + q] = old[w + 1].E[kLinDiagHalo + q];
              W[w].O[P - kLinDiagHalo + q] = old[w + 1].O[kLinDiagHalo + q];
            }
          }
      }
    }
    printf("%d %d %d %d %d %ld %ld %ld %ld\n", M, N, dlo, dhi, waves, cells, bad, first_i, first_j);
  }
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_group_schedule_equals_recurrence(tmp_path):
    """Every first diagonal of two to eight waves over 50 time steps (three
    exchanges), with the last diagonals that give each its fewest and its most
    waves; full bands and whole runs where the origin lies at a wave's ends and
    beside them."""
    src, exe = tmp_path / "schedule.cpp", tmp_path / "schedule"
    src.write_text(SCHEDULE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    lines = []
    for lo in range(0, 1598):
        for hi in {max(260 - lo, 0), max(260 - lo, 0) + 1, 1598 - lo, 1599 - lo}:
            if hi >= 0:
                lines.append((lo + 40, hi + 40, -lo, hi, 50))
    for lo in (200, 223, 224, 255, 256, 257, 416, 447, 448, 449, 639, 640, 641):
        lines += [(lo + 1, n, -lo, n - 1, 0) for n in (lo + 1, lo // 2)]   # full bands
        lines += [(lo + 300, lo + 280, -lo, hi, 0) for hi in (30, 31, 300)]
    out = subprocess.run([str(exe)], input="".join("%d %d %d %d %d\n" % x for x in lines), check=True,
                         capture_output=True, text=True).stdout.splitlines()
    rows = [tuple(map(int, x.split())) for x in out]
    assert len(rows) == len(lines)
    assert {r[4] for r in rows} >= set(range(2, 9))
    assert all(r[5] > 0 for r in rows)
    wrong = [r for r in rows if r[6]]
    assert not wrong, (len(wrong), wrong[:5])


CHOICE = r'''
#include <cstdio>
#include "poyg_lindiag.h"
using namespace poyg;
// lines: align fast cus kinds, then per kind: count rows columns band-parameter fill strips
int main() {
  int align, fast, cus, kinds;
  while (scanf("%d %d %d %d", &align, &fast, &cus, &kinds) == 4) {
    std::vector<LinDiagPair> p;
    std::vector<int> kind;
    for (int q = 0; q < kinds; ++q) {
      int count, m, n, dw, fill, strips;
      scanf("%d %d %d %d %d %d", &count, &m, &n, &dw, &fill, &strips);
      const LinGeom g = lin_geom(m, n, dw);
      LinDiagPair x{1, 0, n, strips != 0};
      if (fill && lin_diag_fits(m, n, g)) lin_diag_range(m, n, g, x.dlo, x.dhi);
      p.insert(p.end(), count, x);
      kind.insert(kind.end(), count, q);
    }
    const LinDiagChoice c = lin_diag_choose(p, align != 0, fast != 0, cus);
    printf("%d", c.group ? 1 : 0);
    for (int q = 0; q < kinds; ++q)
      for (size_t k = 0; k < p.size(); ++k)
        if (kind[k] == q) {
          printf(" %d", c.form[k]);
          break;
        }
    printf("\n");
  }
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_choice_of_fill(tmp_path):
    """Which batches go to the diagonal fill, with several waves per pair or
    one, and which to the strips, on both sides of every rule."""
    src, exe = tmp_path / "choice.cpp", tmp_path / "choice"
    src.write_text(CHOICE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    cost, align, fast, table = 0, 1, 1, 0
    near, plane, wide, skinny = (1000, 995, 10), (600, 300, 10), (1500, 900, 10), (950, 40, 10)
    two, long = (300, 150, 10), (3000, 2990, 60)
    cases = [
        # one pair each, and batches that several waves per pair fill
        (cost, fast, [(1, *near, 1, 1)], (0, 1)), (cost, fast, [(1, *plane, 1, 1)], (1, 5)),
        (cost, fast, [(409, *plane, 1, 1)], (1, 5)), (cost, fast, [(410, *plane, 1, 1)], (0, 4)),
        (align, fast, [(204, *plane, 1, 1)], (1, 5)), (align, fast, [(205, *plane, 1, 1)], (0, 4)),
        # tables
        (cost, table, [(1, *plane, 1, 1)], (1, 0)), (cost, table, [(2000, *plane, 1, 1)], (0, 0)),
        (cost, table, [(16, *near, 1, 1)], (0, 1)), (cost, table, [(2000, *two, 1, 1)], (0, 2)),
        (cost, table, [(2000, *near, 1, 1), (2000, *plane, 1, 1)], (0, 1, 4)),
        (cost, table, [(1999, *near, 1, 1), (2000, *plane, 1, 1)], (0, 0, 0)),
        (cost, table, [(512, 500, 50, 10, 1, 1)], (1, 3)), (cost, table, [(513, 500, 50, 10, 1, 1)], (1, 0)),
        (cost, table, [(1024, 200, 100, 10, 1, 1)], (1, 2)),
        (cost, fast, [(513, 500, 50, 10, 1, 1)], (1, 3)),
        (cost, table, [(100, *near, 1, 1), (1, *plane, 1, 1)], (1, 0, 0)),
        (align, table, [(204, *plane, 1, 1)], (1, 5)), (align, table, [(256, *plane, 1, 1)], (0, 0)),
        (align, table, [(257, *plane, 1, 1)], (0, 4)),
        # few columns
        (cost, fast, [(204, *skinny, 1, 1)], (1, 5)), (cost, fast, [(205, *skinny, 1, 1)], (1, 0)), (cost, fast, [(2000, *skinny, 1, 1)], (0, 0)),
        (cost, fast, [(2000, 900, 65, 10, 1, 1)], (0, 4)),
        (cost, fast, [(2000, 900, 64, 10, 1, 1), (2001, 900, 65, 10, 1, 1)], (0, 4, 4)),
        (align, fast, [(2000, *skinny, 1, 1)], (0, 4)),
        # pairs of more diagonals than the fill holds among others
        (cost, fast, [(7, *near, 1, 1), (1, *wide, 1, 1)], (0, 0, 0)),
        (cost, fast, [(511, *near, 1, 1), (1, *wide, 1, 1)], (0, 0, 0)),
        (cost, fast, [(512, *near, 1, 1), (1, *wide, 1, 1)], (0, 1, 0)),
        (align, fast, [(900, *near, 1, 1), (300, *wide, 1, 1)], (0, 1, 0)),
        (align, fast, [(900, *near, 1, 1), (301, *wide, 1, 1)], (0, 0, 0)),
        (align, fast, [(1024, *near, 1, 1), (1024, *wide, 1, 1)], (0, 1, 0)),
        # what the strips cannot take stays with the fill
        (cost, fast, [(7, *long, 1, 0), (1, *wide, 1, 1)], (0, 1, 0)),
        (cost, table, [(1, *plane, 1, 0)], (1, 5)), (align, fast, [(7, *near, 0, 1), (2, *near, 1, 1)], (0, 0, 0)),
        (cost, fast, [(7, *near, 0, 0), (2, *near, 1, 1)], (0, 0, 1)),
    ]
    text = "".join(f"{mode} {kind} 256 {len(ks)} " + " ".join(" ".join(map(str, k)) for k in ks) + "\n"
                   for mode, kind, ks, _ in cases)
    out = subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout.splitlines()
    got = [tuple(map(int, x.split())) for x in out]
    assert len(got) == len(cases)
    for c, g in zip(cases, got):
        assert g == c[3], (c, g)
