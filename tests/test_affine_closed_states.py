"""Which affine pairs the three-cost groups of the one-pair-per-wave fill may
take (aff_below_high, poyd_amd/csrc/poyg_internal.h).  They close the states
beyond the band's edges with any value from HIGH_NUM (src/algn.c:38) on, where
the reference holds HIGH_NUM itself: for the pairs the rule accepts, a band whose
closed states are unreachable costs what the oracle's costs, and for costs that
reach HIGH_NUM it does not.  The header is plain C++; the test compiles a small
checker with g++."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import pyoracle as po

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "poyd_amd", "csrc")

CHECKER = r'''
#include <algorithm>
#include <cstdio>
#include <vector>
#include "poyg_internal.h"
using namespace poyg;
typedef long long ll;
// lines: sub indel opening la lb, then both sequences' symbols
int main() {
  const ll INF = 1ll << 50;
  int sub, gap, go, la, lb;
  while (scanf("%d %d %d %d %d", &sub, &gap, &go, &la, &lb) == 5) {
    std::vector<int> A(la + 1), B(lb + 1);
    for (int i = 1; i <= la; ++i) scanf("%d", &A[i]);
    for (int j = 1; j <= lb; ++j) scanf("%d", &B[j]);
    std::vector<ll> eh(lb + 1, INF), ev(lb + 1, INF), cb(lb + 1, INF), peh, pev, pcb;
    for (int j = 0; j <= lb; ++j) eh[j] = cb[j] = go + (ll)j * gap;
    cb[0] = 0;
    ev[0] = go;
    int end = std::min(lb, std::max(40, lb - la + 8)), start = 1;
    for (int i = 1; i <= la; ++i) {
      peh = eh, pev = ev, pcb = cb;
      std::fill(eh.begin(), eh.end(), INF);
      std::fill(ev.begin(), ev.end(), INF);
      std::fill(cb.begin(), cb.end(), INF);
      if (i > 40) ++start;
      ev[start - 1] = pev[start - 1] + gap;
      for (int j = start; j <= end; ++j) {
        eh[j] = std::min(eh[j - 1], cb[j - 1] + go) + gap;
        ev[j] = std::min(pev[j], pcb[j] + go) + gap;
        cb[j] = std::min(std::min(pcb[j - 1], pev[j - 1]), peh[j - 1]) + ((A[i] & B[j]) ? 0 : sub);
      }
      if (end < lb) ++end;
    }
    const AffUniform u{1, sub, gap, gap};
    printf("%d %lld\n", aff_below_high(u, go, la + lb) ? 1 : 0, std::min(std::min(eh[lb], ev[lb]), cb[lb]));
  }
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_three_cost_pairs_never_reach_closed_states(tmp_path):
    src, exe = tmp_path / "closed.cpp", tmp_path / "closed"
    src.write_text(CHECKER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    rng = np.random.default_rng(90)
    lines, want = [], []
    for la, lb in [(4, 4), (30, 30), (60, 75), (80, 110), (60, 505), (200, 380), (300, 300), (41, 90)]:
        for sub in (0, 1, 63):
            for gap, go in [(1, 3), (2, 0), (1, 400), (1000, 5), (1600, 3), (2500, 3), (20000, 1), (1, 299000),
                            (1, 333200), (1, 600000), (1, 999980), (1, 1000100), (1, 1200000), (0, 1000001)]:
                a = 1 << rng.integers(0, 4, la)
                b = 1 << rng.integers(0, 4, lb)
                b[:la] = np.where(rng.random(la) < 0.7, a, b[:la])
                lines.append(" ".join(map(str, [sub, gap, go, la, lb, *a, *b])))
                ref = po.CM2.sub_indel(sub, gap, go)
                want.append(po.cost_affine_3(np.concatenate([[16], a]).astype(np.uint8),
                                             np.concatenate([[16], b]).astype(np.uint8), ref))
    out = subprocess.run([str(exe)], input="\n".join(lines) + "\n", check=True, capture_output=True,
                         text=True).stdout.split()
    taken, cost = np.array(out[0::2], int), np.array(out[1::2], np.int64)
    want = np.array(want)
    assert len(taken) == len(want)
    differ = cost != want
    assert not (differ & (taken == 1)).any(), [lines[k][:40] for k in np.flatnonzero(differ & (taken == 1))[:5]]
    assert differ.sum() > 20 and taken.sum() > 100   # costs beyond the closed states' do differ, ordinary ones are taken
