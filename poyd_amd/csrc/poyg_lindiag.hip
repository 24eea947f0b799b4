// The linear band as an anti-diagonal wavefront over its diagonals: fill and
// backtrace (algn_fill_plane_2, src/algn.c:872-968; backtrack_2d, :3551-3666;
// median_2, :4042-4055).
//
// A cell (i, j) lies on diagonal d = j - i of the band dlo .. dhi.  Diagonals
// go in pairs: pair L holds dlo + 2L ("even") and dlo + 2L + 1 ("odd").  At
// time T the even diagonals' cells (T - L + L0, T + L + L0 + dlo) are computed,
// then the odd ones' one column further, with L0 = -dlo / 2 rounded down.  Of
// a cell's neighbours, the diagonal one is the pair's own value of time T - 1,
// and of the upper and the left one, one is the pair's other diagonal and the
// other the next pair's: every step moves one value by one pair.  A register
// holds two neighbouring pairs in its 16-bit halves, a lane R registers
// (pairs 2 R q .. 2 R q + 2 R - 1), so a wave covers 256 R diagonals, and such
// a move is one DPP and one v_alignbit for all of them.  Row and column
// symbols ride along the same way, half as often.  No LDS, no band edge other
// than the first and the last pair, and no work outside the band but its two
// corners, where the strip kernels (lin_cost16_kernel) spend half of their
// steps on the skew of 128-row strips and hold rows and columns in LDS, one
// wave per SIMD for sequences of 2,000.
//
// Values are held as 0xffff - v (v the cost, times 4 with direction codes), so
// that a DPP's zero fill is the "no cell" value: candidates are saturating
// differences, the minimum a maximum, and 0 stays 0.  Cells outside the matrix
// need no test: those before its first row or column are unreachable, those
// past its last ones feed no cell inside.  With direction codes a candidate's
// low two bits are 3 - rank (ALIGN rank 0, then INSERT and DELETE in the order
// backtrack_2d prefers for the pair), so the maximum also names the direction
// the backtrace takes.
//
// Costs: where the matrix prices every two symbols without a common bit alike
// (K) and every symbol without the gap bit alike against the gap (G) -- DNA
// under a substitution / indel model -- the costs come from the symbols' bits
// in two packed operations and no table ("fast"); other pairs read LDS tables.
//
// Bound by VALU issue.  Instructions per time step (four cells a register),
// from the compiled loops: 29 fast and cost-only, 35 with codes (R = 1), 26 and
// 32 a register at R = 2, no other instruction but 2-4 wait states.  Measured
// against the strips with their prefix-sum and backtrace kernels (one MI355X), a
// pass: 16,384 distances of 500-2,000 positions 6.0 to 1.95 ms; 1,000 alignments
// of 200-400 186 to 69 us; a call, its kernels in brackets: a tree level of 6
// medians of 300-1,500 509 to 255 us (448 to 183), one distance of 300 positions
// 74 to 51 us (50 to 27).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "poyg_internal.h"
#include "poyg_lindiag.h"
#include "poyg_wave.h"

namespace poyg {

namespace {

constexpr int kDropOff = 0x7ffffff0;   // buffer offset past any pair's codes
constexpr int kTileT = 32;             // time steps of a backtrace tile

__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b) {
  return c16u(__builtin_elementwise_max(c16v(a), c16v(b)));
}
// per half: max(k - x, 0); written out, since the compiler turns a saturated
// difference from a constant into a compare and a select per half
__device__ __forceinline__ uint32_t pk_rsub(uint32_t k, uint32_t x) {
  uint32_t r;
  asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(r) : "s"(k), "v"(x));
  return r;
}
// per half: c2 - (x >> 15) * c1
__device__ __forceinline__ uint32_t pk_gap(uint32_t x, uint32_t c1, uint32_t c2) {
  uint32_t g, r;
  asm("v_pk_lshrrev_b16 %0, 15, %1 op_sel_hi:[0,1]" : "=v"(g) : "v"(x));
  asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(r) : "v"(g), "v"(c1), "v"(c2));
  return r;
}
__device__ __forceinline__ uint32_t lane_below(uint32_t v) {   // lane q <- q - 1, lane 0 <- 0
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xf, 0xf, true);
}
__device__ __forceinline__ uint32_t lane_above(uint32_t v) {   // lane q <- q + 1, lane 63 <- 0
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xf, 0xf, true);
}
__device__ __forceinline__ uint32_t lane_above(uint32_t v, uint32_t last) {   // lane 63 <- last
  return (uint32_t)__builtin_amdgcn_update_dpp((int)last, (int)v, 0x130, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t both(uint32_t v) { return v * 0x00010001u; }
__device__ __forceinline__ uint32_t table_pair(const uint16_t *t, uint32_t a) {
  const uint32_t lo = *(const uint16_t *)((const char *)t + (a & 0xffffu));
  const uint32_t hi = *(const uint16_t *)((const char *)t + (a >> 16));
  return lo | (hi << 16);
}

// A pair's geometry (wave-uniform).
struct DiagGeom {
  const uint8_t *s1, *s2;   // rows (the longer sequence), columns
  int M, N, dlo, dhi, L0, T_end, L_end, odd_end, groups, cols;
  __device__ __forceinline__ DiagGeom(const PairMeta &m, const uint8_t *seq) {
    s1 = seq + m.off_r;
    s2 = seq + m.off_c;
    M = m.lr;
    N = m.lc;
    dlo = m.p0;
    dhi = m.p1;
    L0 = (-dlo) >> 1;
    const int rel = N - M - dlo;
    L_end = rel >> 1;
    odd_end = rel & 1;
    T_end = M - 1 - L0 + L_end;
    groups = (T_end + 7) >> 3;
    cols = m.stride;
  }
};

// The state of one wave's diagonals, pairs Lw .. Lw + 128 R - 1.
template <bool kDm, bool kFast, int R>
struct DiagFill {
  uint32_t E[R], O[R];           // latest even / odd values
  uint32_t rc[R], cc[R];         // row and column symbols
  uint32_t cd[R], gj[R];         // deletion cost of the row, insertion cost of the column
  uint32_t k1[R], k2[R], om[R];  // gap cost constants (blocked past the last pair), odd-diagonal mask
  uint32_t aE[R], aO[R];         // codes of the group
  uint32_t rwin, cwin;           // entering symbols: rows at lane 0, columns at lane 63
  uint32_t rnext, cnext;         // the next 64 time steps' windows
  uint32_t K, del1, del2;
  int A, B, Lw;
  const uint16_t *tab;

  __device__ __forceinline__ uint32_t row_code(const DiagGeom &g, int i) const {
    const int x = i == 0 ? kGap : (i > 0 && i < g.M ? g.s1[i] & 31 : 0);
    return (uint32_t)x << (kFast ? 11 : 6);
  }
  __device__ __forceinline__ uint32_t col_code(const DiagGeom &g, int j) const {
    const int x = j == 0 ? kGap : (j > 0 && j < g.N ? g.s2[j] & 31 : 0);
    return (uint32_t)x << (kFast ? 11 : 1);
  }
  // windows of the time steps Tb .. Tb + 63
  __device__ __forceinline__ void load_windows(const DiagGeom &g, int Tb) {
    const int lane = lane_id();
    rnext = row_code(g, Tb + lane + A - Lw) << 16;
    cnext = col_code(g, Tb + (kWave - 1 - lane) + Lw + 2 * kWave * R + B);
  }
  __device__ __forceinline__ void swap_windows(const DiagGeom &g, int Tb) {
    rwin = rnext;
    cwin = cnext;
    load_windows(g, Tb + 64);
  }

  __device__ __forceinline__ void row_costs() {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (kFast) cd[r] = pk_gap(rc[r], del1, del2);
      else cd[r] = c16_add(table_pair(tab, rc[r] + both(2 * kGap)), del2);
    }
  }
  __device__ __forceinline__ void col_costs() {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (kFast) gj[r] = pk_gap(cc[r], k1[r], k2[r]);
      else gj[r] = c16_add(table_pair(tab, cc[r] + both(64 * kGap)), k1[r]) | k2[r];
    }
  }
  __device__ __forceinline__ uint32_t sub_cost(int r) const {
    if (kFast) return pk_rsub(K, rc[r] & cc[r]);   // a common bit is at least 2^11 > K
    return table_pair(tab, rc[r] + cc[r]);
  }
  // the code of a maximum joins the group's codes
  __device__ __forceinline__ static uint32_t push(uint32_t acc, uint32_t best, bool first) {
    const uint32_t f = best & 0x00030003u;
    return first ? f : (acc << 2) | f;
  }
  __device__ __forceinline__ void even(bool first) {
    const uint32_t below = lane_below(O[R - 1]);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t left = __builtin_amdgcn_alignbit(O[r], r ? O[r > 0 ? r - 1 : 0] : below, 16);
      const uint32_t t1 = c16_sub_sat(O[r], cd[r]), t2 = c16_sub_sat(left, gj[r]);
      const uint32_t t3 = c16_sub_sat(E[r], sub_cost(r));
      const uint32_t best = pk_max(pk_max(t1, t2), t3);
      if (kDm) aE[r] = push(aE[r], best, first);
      E[r] = kDm ? best | 0x00030003u : best;
    }
  }
  __device__ __forceinline__ void odd(bool first) { odd(first, lane_above(E[0])); }
  __device__ __forceinline__ void odd(bool first, uint32_t above) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t up = __builtin_amdgcn_alignbit(r < R - 1 ? E[r < R - 1 ? r + 1 : 0] : above, E[r], 16);
      const uint32_t t1 = c16_sub_sat(up, cd[r]), t2 = c16_sub_sat(E[r], gj[r]);
      const uint32_t t3 = c16_sub_sat(O[r], sub_cost(r));
      const uint32_t best = pk_max(pk_max(t1, t2), t3) & om[r];
      if (kDm) aO[r] = push(aO[r], best, first);
      O[r] = kDm ? best | 0x00030003u : best;
    }
  }
  __device__ __forceinline__ void step(bool first) {
    {   // rows move up one pair
      const uint32_t next = lane_above(rwin);
      const uint32_t in = (uint32_t)__builtin_amdgcn_update_dpp((int)rwin, (int)rc[R - 1], 0x138, 0xf, 0xf, false);
      rwin = next;
#pragma unroll
      for (int r = R - 1; r >= 0; --r) rc[r] = __builtin_amdgcn_alignbit(rc[r], r ? rc[r > 0 ? r - 1 : 0] : in, 16);
      row_costs();
    }
    even(first);
    {   // columns move down one pair
      const uint32_t next = lane_below(cwin);
      const uint32_t in = (uint32_t)__builtin_amdgcn_update_dpp((int)cwin, (int)cc[0], 0x130, 0xf, 0xf, false);
      cwin = next;
#pragma unroll
      for (int r = 0; r < R; ++r) cc[r] = __builtin_amdgcn_alignbit(r < R - 1 ? cc[r < R - 1 ? r + 1 : 0] : in, cc[r], 16);
      col_costs();
    }
    odd(first);
  }

  // time 0: row 0's and column 0's first cells; above: the even value of the
  // pair above the wave's last (kGroup: the one-wave form has none)
  template <bool kGroup>
  __device__ __forceinline__ void begin(const DiagGeom &g, int Lw_, const LinDiagCosts &c, bool ins_first,
                                        const uint16_t *t, uint32_t above = 0u) {
    const int lane = lane_id();
    tab = t;
    Lw = Lw_;
    A = g.L0;
    B = g.L0 + g.dlo;
    // with codes: costs times 4 and the rank of a candidate
    const uint32_t sc = kDm ? 4 : 1, ins = kDm ? (ins_first ? 1 : 2) : 0, del = kDm ? 3 - ins : 0;
    K = both(sc * c.K);
    del1 = both((0u - sc * c.G) & 0xffffu);
    del2 = kFast ? both(sc * c.G + del) : both(del);
    const int top = (g.dhi - g.dlo) >> 1;
    const bool odd_top = (g.dhi - g.dlo) & 1;   // the last pair has both diagonals
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int L = Lw + 2 * (lane * R + r);
      auto half = [&](auto f) { return (uint32_t)f(L) | ((uint32_t)f(L + 1) << 16); };
      rc[r] = half([&](int l) { return row_code(g, A - l); });
      cc[r] = half([&](int l) { return col_code(g, l + B + 1); });
      const uint32_t blocked = half([&](int l) { return l > top ? 0xffffu : 0u; });
      if (kFast) {
        k1[r] = both((0u - sc * c.G) & 0xffffu) & ~blocked;
        k2[r] = both(sc * c.G + ins) | blocked;
      } else {
        k1[r] = both(ins);
        k2[r] = blocked;
      }
      om[r] = half([&](int l) { return l > top || (l == top && !odd_top) ? 0u : 0xffffu; });
      const uint32_t origin = half([&](int l) { return l == g.L0 ? 0xffffu : 0u; });
      E[r] = (g.dlo & 1) ? 0u : origin;
      O[r] = 0u;
      aE[r] = aO[r] = 0u;
    }
    row_costs();
    col_costs();
    dpp_exec_guard();
    odd(true, kGroup ? lane_above(E[0], above) : lane_above(E[0]));
    if (g.dlo & 1)
#pragma unroll
      for (int r = 0; r < R; ++r)
        O[r] |= (Lw + 2 * (lane * R + r) == g.L0 ? 0xffffu : 0u) | (Lw + 2 * (lane * R + r) + 1 == g.L0 ? 0xffff0000u : 0u);
    load_windows(g, 1);
  }

  __device__ __forceinline__ void store(const DiagGeom &g, __amdgpu_buffer_rsrc_t rsrc, int group, int col, bool own) {
    if (!kDm) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      uint32_t e = aE[r], o = aO[r];
      asm volatile("" : "+v"(e), "+v"(o));   // (a vector load of both would keep the arrays out of registers)
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{e, o}, rsrc, own ? 8 * (group * g.cols + col + r) : kDropOff, 0,
                                            0);
    }
  }
  // a group of eight time steps
  __device__ __forceinline__ void run8() {
#pragma unroll
    for (int u = 0; u < 8; ++u) step(u == 0);
  }
  // the last group: the value of the end cell, which later steps overwrite
  __device__ __forceinline__ int run_last(const DiagGeom &g, int group) {
    const int at = g.L_end - Lw;
    const int lane = at / (2 * R), reg = (at >> 1) % R;
    int end = 0;
#pragma unroll 1
    for (int u = 0; u < 8; ++u) {
      step(u == 0);
      if (1 + 8 * group + u == g.T_end) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (r == reg) end = __builtin_amdgcn_readlane((int)(g.odd_end ? O[r] : E[r]), lane);
      }
    }
    return (0xffff - ((at & 1) ? (int)((uint32_t)end >> 16) : end & 0xffff)) / (kDm ? 4 : 1);
  }
};

// Whether every symbol past the leading gaps suits the bit-wise costs.
__device__ __forceinline__ bool diag_symbols_fast(const DiagGeom &g, int fast) {
  bool ok = true;
  auto scan = [&](const uint8_t *s, int n) {
    for (int k = 1 + lane_id(); k < n; k += kWave) {
      const int x = s[k] & 31;
      ok = ok && x != 0 && x != kGap && (fast == 2 || !(x & kGap));
    }
  };
  scan(g.s1, g.M);
  scan(g.s2, g.N);
  return __all(ok);
}

__device__ __forceinline__ void load_cost_table(const DevTcm *tcm, uint16_t *tab, int scale) {
  // every wave that needs the table writes the same entries
  for (int k = lane_id(); k < 32 * 32; k += kWave) tab[k] = (uint16_t)min(scale * tcm->cost[k], 0xffff);
  wave_sync_mem();
}

// One pair on one wave: cost and, with codes, the direction codes.
template <bool kDm, bool kFast, int R>
__device__ __forceinline__ int diag_fill_one(const DiagGeom &g, const LinDiagCosts &c, bool ins_first,
                                             const uint16_t *tab, uint8_t *dm) {
  DiagFill<kDm, kFast, R> f;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(dm, 0, kDm ? 8 * g.groups * g.cols : 0, 0x00020000);
  f.template begin<false>(g, 0, c, ins_first, tab);
  const int col = lane_id() * R;
  int k = 0;
  for (; k < g.groups - 1; ++k) {
    if ((k & 7) == 0) {
      f.swap_windows(g, 1 + 8 * k);
      dpp_exec_guard();
    }
    f.run8();
    f.store(g, rsrc, k, col, true);
  }
  if ((k & 7) == 0) f.swap_windows(g, 1 + 8 * k);
  dpp_exec_guard();
  const int cost = f.run_last(g, k);
  f.store(g, rsrc, k, col, true);
  return cost;
}

// One pair on the workgroup's first `waves` waves: wave w holds pairs
// 96 w .. 96 w + 127, so that neighbours share 32 pairs, and takes its outer 16
// pairs from them every 16 time steps (lin_diag_exchange).  Every wave of the
// workgroup takes the barriers.
constexpr int kHaloLanes = kLinDiagHalo / 2;   // two pairs a lane
template <bool kDm, bool kFast>
__device__ __forceinline__ int diag_fill_group(const DiagGeom &g, const LinDiagCosts &c, bool ins_first,
                                               const uint16_t *tab, uint8_t *dm, int waves,
                                               uint2 (*halo)[kLinDiagWaves][2][kHaloLanes]) {
  const int lane = lane_id(), wv = wave_in_group();
  DiagFill<kDm, kFast, 1> f;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(dm, 0, kDm ? 8 * g.groups * g.cols : 0, 0x00020000);
  const bool on = wv < waves;
  const int first = kLinDiagStep * wv;
  if (on)
    f.template begin<true>(g, first, c, ins_first, tab,
                           lin_diag_origin_above(g.dlo, first + kLinDiagPairsReg) ? 0xffffu : 0u);
  const bool own = (lane >= kHaloLanes || wv == 0) && (lane < kWave - kHaloLanes || wv == waves - 1);
  const int col = kLinDiagStep / 2 * wv + lane;
  int k = 0, cost = -1;
  for (; k < g.groups - 1; ++k) {
    if (on) {
      if ((k & 7) == 0) f.swap_windows(g, 1 + 8 * k);
      dpp_exec_guard();
      f.run8();
      f.store(g, rsrc, k, col, own);
    }
    if (lin_diag_exchange(k) && waves > 1) {
      uint2 (*h)[2][kHaloLanes] = halo[(k >> 1) & 1];
      if (on) {
        if (lane >= kHaloLanes && lane < 2 * kHaloLanes) h[wv][0][lane - kHaloLanes] = make_uint2(f.E[0], f.O[0]);
        if (lane >= kWave - 2 * kHaloLanes && lane < kWave - kHaloLanes)
          h[wv][1][lane - (kWave - 2 * kHaloLanes)] = make_uint2(f.E[0], f.O[0]);
      }
      __syncthreads();
      if (on) {
        if (lane < kHaloLanes && wv > 0) {
          const uint2 v = h[wv - 1][1][lane];
          f.E[0] = v.x;
          f.O[0] = v.y;
        }
        if (lane >= kWave - kHaloLanes && wv < waves - 1) {
          const uint2 v = h[wv + 1][0][lane - (kWave - kHaloLanes)];
          f.E[0] = v.x;
          f.O[0] = v.y;
        }
      }
    }
  }
  if (on) {
    if ((k & 7) == 0) f.swap_windows(g, 1 + 8 * k);
    dpp_exec_guard();
    // the end cell belongs to the wave that owns its pair
    const int owner = min(max((g.L_end - 2 * kHaloLanes) / kLinDiagStep, 0), waves - 1);
    if (wv == owner) cost = f.run_last(g, k);
    else f.run8();
    f.store(g, rsrc, k, col, own);
  }
  return cost;
}

// ---------------------------------------------------------------------------
// Backtrace of a pair by the calling wave, fused behind its fill.  A lane
// holds one column of codes (two pairs, four diagonals) over 32 time steps:
// per diagonal 64 bits, the latest time step lowest, two bits a cell, 0 for
// ALIGN.  A run of ALIGN from a cell is then the trailing zeros of two
// readlanes shifted to the cell, and the bits that end it name the next move.
// The moves go to a log of two bits per alignment column (16 a lane), which
// the lanes expand together every 1,024 columns: positions by prefix sums, 16
// bytes of both aligned sequences a lane, the medians compacted by rank.
// ---------------------------------------------------------------------------
constexpr int kLogSteps = 16;
constexpr int kLogBatch = kLogSteps * kWave;

__device__ __forceinline__ void diag_trace(const PairMeta &m, const DiagGeom &g, int p, const uint8_t *dm,
                                           const uint8_t *s_med, uint8_t *out, int32_t *out_len, int32_t *status) {
  const int lane = lane_id();
  const bool ins_first = m.swap == 0;   // backtrack_2d's swaped
  const int cap = m.cap;
  uint8_t *o = out + m.out_off;
  uint8_t *o1 = o + (ins_first ? 0 : cap), *o2 = o + (ins_first ? cap : 0), *om = o + 2 * cap;
  uint32_t oplog = 0, acc = 0;   // lane l: columns 16 l .. of the batch (0 ALIGN, 2 DELETE, 3 INSERT); the word being filled
  int s = 0, S0 = 0, ib = g.M - 1, jb = g.N - 1, medpos = cap;

  auto expand = [&](int nst) {
    const uint32_t c = oplog;
    const int v = min(max(nst - kLogSteps * lane, 0), kLogSteps);
    const uint32_t vm = v >= kLogSteps ? 0xffffffffu : ((1u << (2 * v)) - 1u);
    const uint32_t lo = c & 0x55555555u & vm, hi = (c >> 1) & 0x55555555u & vm;
    const int nI = v - __popc(lo & hi), nJ = v - __popc(hi & ~lo);
    const int cI = wave_prefix_sum(nI), cJ = wave_prefix_sum(nJ);
    uint32_t wa[4] = {0u, 0u, 0u, 0u}, wb[4] = {0u, 0u, 0u, 0u}, wm[4] = {0u, 0u, 0u, 0u};
    uint32_t em = 0u;
    int ii = ib - (cI - nI), jj = jb - (cJ - nJ);
#pragma unroll
    for (int h = 0; h < kLogSteps; h += 8) {
      int av[8], bv[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const uint32_t code = (c >> (2 * (h + q))) & 3u;
        av[q] = code == 3u ? kGap : g.s1[min(max(ii, 0), g.M - 1)];
        bv[q] = code == 2u ? kGap : g.s2[min(max(jj, 0), g.N - 1)];
        ii -= code != 3u;
        jj -= code != 2u;
      }
#pragma unroll
      for (int q0 = 0; q0 < 8; ++q0) {
        const int q = h + q0;
        const bool live = q < v;
        const int a = live ? av[q0] : 0, b = live ? bv[q0] : 0;
        const int md = ins_first ? s_med[(a & 31) * 32 + (b & 31)] : s_med[(b & 31) * 32 + (a & 31)];
        const int byte = kLogSteps - 1 - q;   // columns are written right to left
        wa[byte >> 2] |= (uint32_t)a << (8 * (byte & 3));
        wb[byte >> 2] |= (uint32_t)b << (8 * (byte & 3));
        wm[byte >> 2] |= (uint32_t)md << (8 * (byte & 3));
        em |= (uint32_t)(live && md != kGap) << q;
      }
    }
    const int P = cap - kLogSteps - (S0 + kLogSteps * lane);   // 16-byte aligned: cap and S0 are multiples of 16
    if (v > 0 && P >= 0) {
      *(uint4 *)(o1 + P) = make_uint4(wa[0], wa[1], wa[2], wa[3]);
      *(uint4 *)(o2 + P) = make_uint4(wb[0], wb[1], wb[2], wb[3]);
    }
    const int ne = __popc(em), cE = wave_prefix_sum(ne);
    int at = medpos - 1 - (cE - ne);
#pragma unroll
    for (int q = 0; q < kLogSteps; ++q) {
      const int byte = kLogSteps - 1 - q;
      if ((em >> q) & 1u) om[at] = (uint8_t)(wm[byte >> 2] >> (8 * (byte & 3)));
      at -= (em >> q) & 1u;
    }
    medpos -= lane63(cE);
    ib -= lane63(cI);
    jb -= lane63(cJ);
    S0 += nst;
    oplog = 0u;
  };
  // appends r columns of one operation
  auto append = [&](uint32_t code, int r) {
    while (r > 0) {
      const int q = s & 15, n = code ? min(r, 16 - q) : min(r, kLogBatch - s);
      if (code) acc |= ((code * 0x55555555u) & (n >= 16 ? 0xffffffffu : ((1u << (2 * n)) - 1u))) << (2 * q);
      if (((s + n) >> 4) != (s >> 4)) {   // the word is full (a longer run's others hold zeros)
        oplog = lane == (s >> 4) ? acc : oplog;
        acc = 0u;
      }
      s += n;
      r -= n;
      if (s == kLogBatch) {
        expand(s);
        s = 0;
      }
    }
  };

  int i = g.M - 1, j = g.N - 1, L = g.L_end, odd = g.odd_end, T = g.T_end, bad = 0;
  int tile = 0, base = 0, pbase = 0;
  uint2 pre[4];
  // 64 bits (0 low, 1 high) per diagonal: e / o even / odd, a / b the pair's half
  uint32_t ea0 = 0, ea1 = 0, eb0 = 0, eb1 = 0, oa0 = 0, oa1 = 0, ob0 = 0, ob1 = 0;
  auto base_of = [&](int l) { return min(max((l >> 1) - kWave / 2, 0), max(0, g.cols - kWave)); };
  auto fetch = [&](int t, int b) {
    const uint2 *src = (const uint2 *)dm + min(b + lane, g.cols - 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) pre[q] = src[(int64_t)min(4 * t + q, g.groups - 1) * g.cols];
  };
  auto commit = [&]() {
    ea0 = ~__builtin_amdgcn_perm(pre[2].x, pre[3].x, 0x05040100u);
    ea1 = ~__builtin_amdgcn_perm(pre[0].x, pre[1].x, 0x05040100u);
    eb0 = ~__builtin_amdgcn_perm(pre[2].x, pre[3].x, 0x07060302u);
    eb1 = ~__builtin_amdgcn_perm(pre[0].x, pre[1].x, 0x07060302u);
    oa0 = ~__builtin_amdgcn_perm(pre[2].y, pre[3].y, 0x05040100u);
    oa1 = ~__builtin_amdgcn_perm(pre[0].y, pre[1].y, 0x05040100u);
    ob0 = ~__builtin_amdgcn_perm(pre[2].y, pre[3].y, 0x07060302u);
    ob1 = ~__builtin_amdgcn_perm(pre[0].y, pre[1].y, 0x07060302u);
  };
  if (i > 0 && j > 0) {
    tile = (T - 1) >> 5;
    base = base_of(L);
    fetch(tile, base);
    commit();
    pbase = base_of(L);
    if (tile > 0) fetch(tile - 1, pbase);
  }
  while (i > 0 && j > 0) {
    if (T < 1 || L < 0 || (L >> 1) >= g.cols) {   // left the band
      bad = 1;
      break;
    }
    if (((T - 1) >> 5) < tile) {
      tile -= 1;
      base = pbase;
      // a tile's 32 time steps move the walk by at most 16 columns
      if (((L >> 1) - base < 17 || (L >> 1) - base > kWave - 18) && base_of(L) != base) {
        base = base_of(L);
        fetch(tile, base);
      }
      commit();
      pbase = base_of(L);
      if (tile > 0) fetch(tile - 1, pbase);
    }
    const int k = 31 - ((T - 1) & 31), c = (L >> 1) - base;
    const bool h = L & 1;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(odd ? (h ? ob0 : oa0) : (h ? eb0 : ea0)), c);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(odd ? (h ? ob1 : oa1) : (h ? eb1 : ea1)), c);
    const uint64_t x = (((uint64_t)hi << 32) | lo) >> (2 * k);
    const int zeros = x ? (int)(__builtin_ctzll(x) >> 1) : kTileT - k;
    const int run = min(min(zeros, kTileT - k), min(i, j));
    if (run > 0) append(0u, run);
    i -= run;
    j -= run;
    T -= run;
    if (run == zeros && k + run < kTileT && i > 0 && j > 0) {   // the move that ends the run
      const uint32_t rank = (uint32_t)(x >> (2 * run)) & 3u;
      if (rank == 3u) {
        bad = 1;
        break;
      }
      const bool ins = (rank == 1u) == ins_first;
      append(ins ? 3u : 2u, 1);
      i -= !ins;
      j -= ins;
      T -= !odd;
      L += odd ? !ins : -(int)ins;
      odd = !odd;
    }
  }
  if (!bad) {   // column 0, row 0, and the column of the two leading symbols
    append(2u, i);
    append(3u, j);
    append(0u, 1);
  }
  if (s & 15) oplog = lane == (s >> 4) ? acc : oplog;
  if (s) expand(s);
  if (lane == 0 && !bad) om[medpos - 1] = kGap;   // the leading gap of median_2
  out_len[3 * p + 0] = S0;
  out_len[3 * p + 1] = S0;
  out_len[3 * p + 2] = cap - (medpos - 1);
  if (bad) {
    const int old = atomicOr(&status[kStatusFlags + p], 1);
    atomicAdd(&status[0], old == 0 ? 1 : 0);
  }
}

__device__ __forceinline__ void load_medians(const DevTcm *tcm, uint8_t *s_med) {
  ((uint4 *)s_med)[lane_id()] = ((const uint4 *)tcm->median)[lane_id()];
  wave_sync_mem();
}

}  // namespace

// One pair per wave, four waves a workgroup; PairMeta::p2 registers per lane.
template <bool kDm>
__global__ __launch_bounds__(kWave * 4) void lin_diag_kernel(const PairMeta *__restrict__ meta,
                                                             const int32_t *__restrict__ order, int n, int *counter,
                                                             const uint8_t *__restrict__ seq,
                                                             const DevTcm *__restrict__ tcm, LinDiagCosts costs,
                                                             uint8_t *dm_base, int32_t *__restrict__ cost_out,
                                                             uint8_t *out, int32_t *out_len, int32_t *status) {
  __shared__ uint16_t tab[32 * 32];
  __shared__ __attribute__((aligned(16))) uint8_t s_med[32 * 32];
  if (kDm) load_medians(tcm, s_med);
  bool have_tab = false;
  for (;;) {
    const int item = next_item(counter);
    if (item >= n) break;
    const int p = uniform32(order[item]);
    const PairMeta m = uniform_meta(meta, p);
    const DiagGeom g(m, seq);
    uint8_t *dm = dm_base + m.dm_off;
    const bool ins_first = m.swap == 0;
    const bool fast = costs.fast && diag_symbols_fast(g, costs.fast);
    if (!fast && !have_tab) {
      load_cost_table(tcm, tab, kDm ? 4 : 1);
      have_tab = true;
    }
    int cost;
    if (m.p2 == 1) {
      cost = fast ? diag_fill_one<kDm, true, 1>(g, costs, ins_first, tab, dm)
                  : diag_fill_one<kDm, false, 1>(g, costs, ins_first, tab, dm);
    } else if (m.p2 == 2) {
      cost = fast ? diag_fill_one<kDm, true, 2>(g, costs, ins_first, tab, dm)
                  : diag_fill_one<kDm, false, 2>(g, costs, ins_first, tab, dm);
    } else {
      cost = fast ? diag_fill_one<kDm, true, 4>(g, costs, ins_first, tab, dm)
                  : diag_fill_one<kDm, false, 4>(g, costs, ins_first, tab, dm);
    }
    cost_out[p] = cost;   // every lane stores the same value
    if (kDm) diag_trace(m, g, p, dm, s_med, out, out_len, status);
  }
}

// One pair per workgroup; PairMeta::p2 of its waves fill, the first one traces.
template <bool kDm>
__global__ __launch_bounds__(kWave * kLinDiagWaves) void lin_diag_group_kernel(
    const PairMeta *__restrict__ meta, const int32_t *__restrict__ order, int n, int *counter,
    const uint8_t *__restrict__ seq, const DevTcm *__restrict__ tcm, LinDiagCosts costs, uint8_t *dm_base,
    int32_t *__restrict__ cost_out, uint8_t *out, int32_t *out_len, int32_t *status) {
  __shared__ uint16_t tab[32 * 32];
  __shared__ __attribute__((aligned(16))) uint8_t s_med[32 * 32];
  __shared__ uint2 halo[2][kLinDiagWaves][2][kHaloLanes];
  __shared__ int s_item;
  if (kDm) load_medians(tcm, s_med);
  bool have_tab = false;
  for (;;) {
    __syncthreads();   // the previous pair is done in every wave
    if (threadIdx.x == 0) s_item = atomicAdd(counter, 1);
    __syncthreads();
    const int item = uniform32(s_item);
    if (item >= n) break;
    const int p = uniform32(order[item]);
    const PairMeta m = uniform_meta(meta, p);
    const DiagGeom g(m, seq);
    uint8_t *dm = dm_base + m.dm_off;
    const bool ins_first = m.swap == 0;
    const bool fast = costs.fast && diag_symbols_fast(g, costs.fast);
    if (!fast && !have_tab) {
      load_cost_table(tcm, tab, kDm ? 4 : 1);
      have_tab = true;
    }
    const int cost = fast ? diag_fill_group<kDm, true>(g, costs, ins_first, tab, dm, m.p2, halo)
                          : diag_fill_group<kDm, false>(g, costs, ins_first, tab, dm, m.p2, halo);
    if (cost >= 0) cost_out[p] = cost;
    if (kDm) {
      __syncthreads();   // every wave's codes are stored
      if (wave_in_group() == 0) diag_trace(m, g, p, dm, s_med, out, out_len, status);
    }
  }
}

template <bool kDm>
static int diag_occupancy() {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, lin_diag_kernel<kDm>, kWave * 4, 0) != hipSuccess || nb < 1) nb = 1;
  return nb;
}

int lin_diag_blocks_per_cu(bool with_dm) {
  static const int with = diag_occupancy<true>(), without = diag_occupancy<false>();
  return with_dm ? with : without;
}

hipError_t launch_lin_diag(bool with_dm, int waves, int grid, const PairMeta *meta, const int32_t *order, int n,
                           int *counter, const uint8_t *seq, const DevTcm *tcm, const LinDiagCosts &costs, uint8_t *dm,
                           int32_t *cost, uint8_t *out, int32_t *out_len, int32_t *status, hipStream_t s) {
  if (waves) {
    auto k = with_dm ? lin_diag_group_kernel<true> : lin_diag_group_kernel<false>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kWave * waves), 0, s, meta, order, n, counter, seq, tcm, costs, dm, cost, out,
                       out_len, status);
  } else {
    auto k = with_dm ? lin_diag_kernel<true> : lin_diag_kernel<false>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kWave * 4), 0, s, meta, order, n, counter, seq, tcm, costs, dm, cost, out,
                       out_len, status);
  }
  return hipGetLastError();
}

}  // namespace poyg
