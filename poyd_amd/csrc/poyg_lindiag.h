// Which linear pairs the diagonal fill (poyg_lindiag.hip) takes, and how.
// Plain C++ (no HIP), so that a CPU test can check it.
#pragma once

#include <stdint.h>

#include <algorithm>

#include "poyg_band.h"
#include "poyg_internal.h"

namespace poyg {

constexpr int kLinDiagWaves = 8;     // most waves of a workgroup on one pair
constexpr int kLinDiagStep = 96;     // diagonal pairs a further wave adds (128, 32 of them shared)
constexpr int kLinDiagRegs = 4;      // most registers per lane of the one-wave form
constexpr int kLinDiagPairsReg = 128;   // diagonal pairs per register of a wave

// Costs as the kernels take them.  fast: 2 where symbols without a common bit
// cost K and symbols without the gap bit cost G against the gap, whatever
// their other bits; 1 where that holds for symbols without the gap bit; 0
// otherwise (tables).
struct LinDiagCosts {
  int K, G, fast;
};

// Diagonals of the band of algn_fill_plane_2 (lin_row_host): row i holds the
// columns max(0, i + dlo) .. min(n - 1, i + dhi).
inline void lin_diag_range(int m, int n, const LinGeom &g, int &dlo, int &dhi) {
  dlo = g.cs == kBandFull ? -(m - 1) : (g.cs == kBandCase2 ? -(g.h - 1) : -g.h);
  dhi = g.cs == kBandFull ? n - 1 : g.w - 1;
}

// Whether the band is such a set of diagonals that holds both corners (a
// caller's band parameter may be anything).
inline bool lin_diag_fits(int m, int n, const LinGeom &g) {
  if (m < 2 || n < 2) return false;
  if (g.cs == kBandFull) return true;
  return g.w >= 1 && g.w <= n && g.h == m - n + g.w;
}

// Waves (workgroup form) or registers per lane (one-wave form) that hold the
// pairs of diagonals dlo .. dhi; 0 where they do not fit.
inline int lin_diag_waves(int dlo, int dhi) {
  const int pairs = (dhi - dlo) / 2 + 1;
  const int w = pairs <= kLinDiagPairsReg ? 1 : 1 + (pairs - kLinDiagPairsReg + kLinDiagStep - 1) / kLinDiagStep;
  return w <= kLinDiagWaves ? w : 0;
}
inline int lin_diag_regs(int dlo, int dhi) {
  const int pairs = (dhi - dlo) / 2 + 1;
  for (int r = 1; r <= kLinDiagRegs; r *= 2)
    if (pairs <= r * kLinDiagPairsReg) return r;
  return 0;
}
// The workgroup form's schedule.  A wave holds the pairs Lw .. Lw + 127 and
// nothing outside them ("no cell"), so its outermost pairs go wrong, one on
// each side a time step: an even cell takes a value of the pair below, an odd
// one of the pair above.  After every sixteenth time step, before an owned pair
// is wrong, its outer kLinDiagHalo pairs are replaced by the neighbours' own.
// Time 0 must not cost a pair of them: its odd half step is the first to read
// the pair above, of which only the origin's holds a cell then
// (lin_diag_origin_above).
constexpr int kLinDiagHalo = 16;
constexpr bool lin_diag_exchange(int group) { return group & 1; }   // behind this group of eight time steps
// Whether cell (0, 0) is the even cell of pair `above`, the pair above a wave's last.
constexpr bool lin_diag_origin_above(int dlo, int above) { return !(dlo & 1) && ((-dlo) >> 1) == above; }

// Columns of codes per group of eight time steps, and the bytes of all groups.
inline int lin_diag_cols(bool group, int k) {
  return group ? kWave + kLinDiagStep / 2 * (k - 1) : kWave * k;
}
inline int64_t lin_diag_bytes(int m, int n, int dlo, int cols) {
  const int t_end = m - 1 - ((-dlo) >> 1) + ((n - m - dlo) >> 1);
  return (int64_t)((t_end + 7) / 8) * cols * 8;
}

// K, G and fast of a matrix.
inline LinDiagCosts lin_diag_costs(const DevTcm &t, int scale) {
  LinDiagCosts c{t.cost[1 * 32 + 2], t.cost[1 * 32 + kGap], 2};
  // the bit-wise form compares K with a symbol bit of 2^11 and holds G and a rank in 16 bits
  if (scale * c.K >= 2048 || scale * c.G >= 16384) return LinDiagCosts{0, 0, 0};
  for (int a = 1; a < 32; ++a)
    for (int b = 1; b < 32; ++b) {
      if (a == kGap && b == kGap) continue;
      const int want = (a == kGap || b == kGap) ? ((a & b & kGap) ? 0 : c.G) : ((a & b) ? 0 : c.K);
      if (t.cost[a * 32 + b] == want) continue;
      const bool plain = (a == kGap || !(a & kGap)) && (b == kGap || !(b & kGap));
      if (plain) return LinDiagCosts{0, 0, 0};
      c.fast = 1;
    }
  return c;
}

}  // namespace poyg
