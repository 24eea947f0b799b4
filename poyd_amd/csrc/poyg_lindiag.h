// Which linear pairs the diagonal fill (poyg_lindiag.hip) takes, and how.
// Plain C++ (no HIP), so that a CPU test can check it.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <vector>

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
// A pair of a batch as the choice below sees it: its diagonals (dlo > dhi where
// the fill cannot take it), its columns, and whether the strips can take it.
struct LinDiagPair {
  int dlo, dhi, cols;
  bool strips;
};

// Which pairs of a batch the diagonal fill takes (form: waves or registers per
// pair, 0 for the strips), and whether with several waves on a pair.
//
// Several waves: where pairs need more than one register per lane and the batch
// leaves SIMDs idle (a wave's step is shortest with one register; past that the
// wave per pair wins, which computes no shared diagonals).  Pairs of 1,500-2,000
// (2.4 waves each), several waves against one: costs of 256 / 768 / 1,024 pairs
// 186 / 364 / 442 us against 374 / 382 / 385; alignments of 256 / 512 / 1,024
// pairs 283 / 370 / 398 against 353 / 356 / 361.
//
// The strips for a batch of whole planes of many diagonals and few cells, times
// in us, the fill's against theirs:
// * Costs from tables (fast false) with four registers: 1,024 of 600 x 100 150 against 95,
//   2,048 of 500 x 50 199 / 122, 2,048 of 600 x 300 298 / 288 (two registers: 113
//   / 128 for 2,048 of 300 x 150); with five waves or more, three
//   where a SIMD holds more than 1.5 waves: 16 of 600 x 300 84 / 74, of 1,000 x 20
//   93 / 77 (four waves: 50 / 56 for 400 x 250), 640 of 500 x 50 75 / 62 (two
//   waves: 49 / 52 for 1,024 of 200 x 100).
// * Costs without tables of up to 64 columns, four registers: 1,024 of 500 x 50 75
//   / 70, 2,048 of 1,000 x 20 212 / 179 (900 x 80: 206 / 221); five waves or more
//   where the batch has more waves than SIMDs: 300 of 1,000 x 20 112 / 95 (200 of
//   them 75 / 78).
// * Alignments with tables and four registers where the strips have four waves
//   per pair and compute unit: 256 of 600 x 300 328 / 309 (300 of them 328 / 352).
//
// And for all pairs of a batch where some have to take them: both kernels then
// run one after the other, and in a small batch each lasts as long as its longest
// pair.  8 costs of 1,000 x 1,000 with one of 1,500 x 900 328 us against 256 in
// strips alone, 512 of 400-800 with 28% such 207 / 156 (768 of them 209 / 254);
// alignments of 8 with one 819 / 724, 1,024 of 400-800 with 28% 727 / 630 (3,000
// of them 1,117 / 1,378, 1,024 of 1,000 x 1,000 with one 863 / 1,384).  For the
// same reason a batch is not split by the rules above: its majority decides, in
// a small one any pair.
struct LinDiagChoice {
  bool group = false;
  std::vector<int> form;
};

inline LinDiagChoice lin_diag_choose(const std::vector<LinDiagPair> &pairs, bool align, bool fast, int cus) {
  const int64_t n = (int64_t)pairs.size();
  LinDiagChoice c;
  c.form.assign(pairs.size(), 0);
  int64_t waves = 0;
  bool multi = false;
  for (const LinDiagPair &p : pairs) {
    if (p.dlo > p.dhi) continue;
    const int w = lin_diag_waves(p.dlo, p.dhi);
    waves += w ? w : 1 << 20;
    multi = multi || w > 1;
  }
  c.group = multi && waves <= (align ? 4 : 8) * (int64_t)cus;
  auto slow = [&](const LinDiagPair &p, int f) {
    if (!f || !p.strips) return false;
    if (c.group) {
      if (align) return false;
      return fast ? f >= 5 && p.cols <= 64 && waves > 4 * (int64_t)cus : f >= (waves > 6 * (int64_t)cus ? 3 : 5);
    }
    if (f < 4) return false;
    if (align) return !fast && n <= cus;
    return !fast || p.cols <= 64;
  };
  int64_t strips = 0, slower = 0;
  bool every = true;   // the strips can take all pairs of the fill
  for (size_t k = 0; k < pairs.size(); ++k) {
    const LinDiagPair &p = pairs[k];
    const int f = p.dlo > p.dhi ? 0 : c.group ? lin_diag_waves(p.dlo, p.dhi) : lin_diag_regs(p.dlo, p.dhi);
    c.form[k] = f;
    strips += !f && p.strips;
    slower += slow(p, f);
    every = every && (!f || p.strips);
  }
  const bool small = n <= 2 * (int64_t)cus;
  const bool apart = strips && (small || (align && 4 * strips > n && n < 8 * (int64_t)cus));
  if (every && (apart || (small ? slower > 0 : 2 * slower > n))) c.form.assign(pairs.size(), 0);
  return c;
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
