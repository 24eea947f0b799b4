// Three-sequence alignment on gfx950: algn_fill_cube (src/algn.c:2885-3055)
// and backtrack_3d (:3829-3905).
//
// A cube is filled row by row (a row = the n3 cells of one (plane, line)),
// lanes across the s3 axis and the self-gap chain along s3 evaluated as a
// prefix minimum: a workgroup of eight waves per triple takes the rows whose
// inputs are final (the block kernel and its packed form), one wave the
// triples with rows above 1,024 cells or negative costs.  The reference walks three row pointers
// that advance n2-1 rows per plane while the output advances n2 rows, so
// plane p >= 1, line r >= 1 reads its "diagonal", "upper" and "previous"
// rows at flat row indices out-n2-p, out-n2-p+1 and out-p-1 (and the first
// line of plane p reads out-n2-p+1).  Those rows are kept in a ring in
// global memory.  The direction cube (4 bits per cell; a byte in the one-wave
// kernel) is walked afterwards by one thread per triple.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <numeric>
#include <type_traits>
#include <vector>

#include "poyg_cube.h"
#include "poyg_internal.h"

namespace poyg {

struct TripleMeta {
  int64_t off1, off2, off3, out_off, dm_off;
  int32_t l1, l2, l3, cap;
  int32_t dstride;   // bytes per row of the direction cube
  int32_t flags;     // bit 0: two 4-bit codes per byte (else one per byte); bits 1-2: wave priority
};

// Direction codes, one byte per cell: the index of the winning move in the
// reference's evaluation order (fill_parallel P3, P1, P2, then fill_moved S3,
// S1, S2, then the self pass SS; src/algn.c:2812-2858, 3041-3048).  With
// strict-< first-wins updates the winner is the first minimum in this order.
constexpr int kP3 = 0, kP1 = 1, kP2 = 2, kS3 = 3, kS1 = 4, kS2 = 5, kSS = 6;

__device__ __forceinline__ int c_lane() { return (int)__lane_id(); }

__device__ __forceinline__ int64_t c_uniform64(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// LDS ordering across lanes of one wave (see wave_sync_mem in poyg_kernels.hip).
__device__ __forceinline__ void c_lds_sync() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_wave_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Ordering of one wave's own global stores before its later loads of the
// same rows (a triple's rows are written and read by one workgroup, so workgroup
// scope suffices: no L2 write-back or invalidate is needed).
__device__ __forceinline__ void c_wave_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup"); }

// DPP-only cross-lane helpers (see poyg_kernels.hip).
// Eight wait states and a scheduling barrier between any EXEC change and the
// DPP moves that follow (a DPP issued shortly after an EXEC restore has been
// seen to treat enabled source lanes as disabled).
__device__ __forceinline__ void c_dpp_guard() {
  asm volatile("s_nop 7");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ int c_prefix_min(int v) {
  c_dpp_guard();
  constexpr int I = 0x7fffffff;
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x111, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x112, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x114, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x118, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x142, 0xa, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x143, 0xc, 0xf, false));
  return v;
}
__device__ __forceinline__ int c_prefix_sum(int v) {
  c_dpp_guard();
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

// Self-gap chain along s3 with the reference's strict-< rule: the value of
// a cell becomes mm[k-1] + ggs3[k] only when that is strictly smaller.
// v: value after the six plane/line moves; G3: prefix sums of ggs3.
struct ChainOut {
  int mm;
  bool ss;
};
__device__ __forceinline__ ChainOut c_chain(int v, bool act, int G3k, int g, int &carry_mm, int &carry_g3,
                                           bool k0) {
  const int big = 0x3fffffff;
  int pm = c_prefix_min(act ? v - G3k : big);
  pm = min(pm, carry_mm - carry_g3);
  const int mm = G3k + pm;
  c_dpp_guard();
  const int left = __builtin_amdgcn_update_dpp(carry_mm, mm, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
  ChainOut o;
  o.ss = act && !k0 && (left + g < v);
  o.mm = o.ss ? left + g : v;
  carry_mm = __builtin_amdgcn_readlane(mm, 63);
  carry_g3 = __builtin_amdgcn_readlane(G3k, 63);
  return o;
}

__global__ __launch_bounds__(64) void cube_fill_kernel(const TripleMeta *__restrict__ meta,
                                                       const int32_t *__restrict__ order, int n, int *counter,
                                                       const uint8_t *__restrict__ seq,
                                                       const DevTcm3 *__restrict__ tcm, uint8_t *dm_base,
                                                       int *scratch, int64_t scratch_per_wave, int32_t *cost_out) {
  __shared__ int s_r[4][32];   // ggs3, s1gs3, gs2s3, s1s2s3 rows indexed by the s3 symbol
  const int lane = c_lane();
  int *ring = scratch + (size_t)blockIdx.x * scratch_per_wave;
  const int gap = tcm->gap;
  if (lane < 32) s_r[0][lane] = tcm->cost[(gap * 32 + gap) * 32 + lane];
  c_lds_sync();
  for (;;) {
    int kk = 0;
    if (lane == 0) kk = atomicAdd(counter, 1);
    kk = __builtin_amdgcn_readfirstlane(kk);
    if (kk >= n) break;
    // the descriptor is wave-uniform: keep it in scalar registers so that the
    // loops over it compile to scalar branches
    const int t = __builtin_amdgcn_readfirstlane(order[kk]);
    TripleMeta m = meta[t];
    m.off1 = c_uniform64(m.off1);
    m.off2 = c_uniform64(m.off2);
    m.off3 = c_uniform64(m.off3);
    m.out_off = c_uniform64(m.out_off);
    m.dm_off = c_uniform64(m.dm_off);
    m.l1 = __builtin_amdgcn_readfirstlane(m.l1);
    m.l2 = __builtin_amdgcn_readfirstlane(m.l2);
    m.l3 = __builtin_amdgcn_readfirstlane(m.l3);
    m.cap = __builtin_amdgcn_readfirstlane(m.cap);
    const uint8_t *s1 = seq + m.off1, *s2 = seq + m.off2, *s3 = seq + m.off3;
    const int n1 = m.l1, n2 = m.l2, n3 = m.l3, W = n1 + n2;
    int *G3 = ring + (size_t)W * n3;
    uint8_t *dm = dm_base + m.dm_off;
    const int s30 = s3[0] & 31;
    // prefix sums of the (gap, gap, s3[k]) row
    {
      int carry = 0;
      for (int k0 = 0; k0 < n3; k0 += 64) {
        const int k = k0 + lane;
        const int g = (k >= 1 && k < n3) ? s_r[0][s3[k] & 31] : 0;
        const int ps = c_prefix_sum(g) + carry;
        if (k < n3) G3[k] = ps;
        carry = __builtin_amdgcn_readlane(ps, 63);
      }
    }
    c_wave_fence();
#define ROW(R) (ring + (size_t)((R) % W) * n3)
    // plane 0, line 0: 0, then the self-gap chain
    for (int k0 = 0; k0 < n3; k0 += 64) {
      const int k = k0 + lane;
      if (k < n3) {
        ROW(0)[k] = G3[k];
        dm[k] = k == 0 ? kS2 : kSS;
      }
    }
    c_wave_fence();
    int fenced = 0;   // rows [0, fenced] are visible to loads
    // plane 0, lines r >= 1
    for (int r = 1; r < n2; ++r) {
      const int x = s2[r] & 31;
      c_lds_sync();   // previous row's reads of the tables are done
      if (lane < 32) s_r[2][lane] = tcm->cost[(gap * 32 + x) * 32 + lane];
      c_lds_sync();
      const int *pv = ROW(r - 1);
      int *cur = ROW(r);
      uint8_t *dc = dm + (size_t)r * n3;
      const int gs2g = s_r[2][s30];
      int carry_mm = 0x3fffffff, carry_g3 = 0;
      for (int k0 = 0; k0 < n3; k0 += 64) {
        const int k = k0 + lane;
        const bool act = k < n3;
        int v = 0, code = kP1, G3k = 0, g = 0;
        if (act) {
          const int y = s3[k];
          G3k = G3[k];
          g = s_r[0][y];
          v = pv[k] + gs2g;
          if (k > 0) {
            const int tt = pv[k - 1] + s_r[2][y];
            if (tt < v) { v = tt; code = kS1; }
          }
        }
        const ChainOut o = c_chain(v, act, G3k, g, carry_mm, carry_g3, k == 0);
        if (act) {
          cur[k] = o.mm;
          dc[k] = (uint8_t)(o.ss ? kSS : code);
        }
      }
      c_wave_fence();
      fenced = r;
    }
    // planes p >= 1
    for (int p = 1; p < n1; ++p) {
      const int a = s1[p] & 31;
      c_lds_sync();
      if (lane < 32) s_r[1][lane] = tcm->cost[(a * 32 + gap) * 32 + lane];
      c_lds_sync();
      const int s1gg = s_r[1][s30];
      // line 0: reads the row the "diagonal" pointer holds, out-(n2+p-1)
      {
        const int out = p * n2;
        if (out - (n2 + p - 1) > fenced) { c_wave_fence(); fenced = out - 1; }
        const int *dg = ROW(out - (n2 + p - 1));
        int *cur = ROW(out);
        uint8_t *dc = dm + (size_t)out * n3;
        int carry_mm = 0x3fffffff, carry_g3 = 0;
        for (int k0 = 0; k0 < n3; k0 += 64) {
          const int k = k0 + lane;
          const bool act = k < n3;
          int v = 0, code = kP3, G3k = 0, g = 0;
          if (act) {
            const int y = s3[k] & 31;
            G3k = G3[k];
            g = s_r[0][y];
            v = dg[k] + s1gg;
            if (k > 0) {
              const int tt = dg[k - 1] + s_r[1][y];
              if (tt < v) { v = tt; code = kS3; }
            }
          }
          const ChainOut o = c_chain(v, act, G3k, g, carry_mm, carry_g3, k == 0);
          if (act) {
            cur[k] = o.mm;
            dc[k] = (uint8_t)(o.ss ? kSS : code);
          }
        }
      }
      for (int r = 1; r < n2; ++r) {
        const int out = p * n2 + r;
        const int b = s2[r] & 31;
        c_lds_sync();
        if (lane < 32) {
          s_r[2][lane] = tcm->cost[(gap * 32 + b) * 32 + lane];
          s_r[3][lane] = tcm->cost[(a * 32 + b) * 32 + lane];
        }
        c_lds_sync();
        if (out - p - 1 > fenced) { c_wave_fence(); fenced = out - 1; }
        const int *dg = ROW(out - n2 - p), *up = ROW(out - n2 - p + 1), *pv = ROW(out - p - 1);
        int *cur = ROW(out);
        uint8_t *dc = dm + (size_t)out * n3;
        const int gs2g = s_r[2][s30], s1s2g = s_r[3][s30];
        int carry_mm = 0x3fffffff, carry_g3 = 0;
        for (int k0 = 0; k0 < n3; k0 += 64) {
          const int k = k0 + lane;
          const bool act = k < n3;
          int v = 0, code = kP3, G3k = 0, g = 0;
          if (act) {
            const int y = s3[k] & 31;
            G3k = G3[k];
            g = s_r[0][y];
            // fill_parallel (:2840-2858) then fill_moved (:2812-2833), strict <
            v = up[k] + s1gg;
            int tt = pv[k] + gs2g;
            if (tt < v) { v = tt; code = kP1; }
            tt = dg[k] + s1s2g;
            if (tt < v) { v = tt; code = kP2; }
            if (k > 0) {
              tt = up[k - 1] + s_r[1][y];
              if (tt < v) { v = tt; code = kS3; }
              tt = pv[k - 1] + s_r[2][y];
              if (tt < v) { v = tt; code = kS1; }
              tt = dg[k - 1] + s_r[3][y];
              if (tt < v) { v = tt; code = kS2; }
            }
          }
          const ChainOut o = c_chain(v, act, G3k, g, carry_mm, carry_g3, k == 0);
          if (act) {
            cur[k] = o.mm;
            dc[k] = (uint8_t)(o.ss ? kSS : code);
          }
        }
      }
    }
    // the reference returns the last cell of the last row written; every
    // lane stores the same value (no lane-divergent code at the end of the
    // item loop body, which keeps the loop scalar)
    c_wave_fence();
    cost_out[t] = ROW(n1 * n2 - 1)[n3 - 1];
    c_wave_fence();
#undef ROW
  }
}

// ---------------------------------------------------------------------------
// Block kernel: a workgroup of kWaves waves (8 or 2) fills one cube, a wave two
// consecutive rows at a time.  Lane L owns the R consecutive cells k = L*R ..
// L*R+R-1 of a row (n3 <= 64*R), so a row is one pass: six candidate moves per
// cell as ranked keys (value*8 + move index; the minimum key is the
// reference's first minimum), then the self pass along s3 as one prefix
// minimum (mm[k] = min(v[k], mm[k-1] + g[k]) equals G3[k] + min_{j<=k}(v[j] -
// G3[j]) with G3 the prefix sums of g; the self move wins exactly where
// mm[k-1] + g[k] < v[k]).
//
// The reference's row pointers lag (see the top of this file): row `out` of
// plane p >= 1 reads rows out-(n2+p-1) ("upper", or "diagonal" on line 0),
// out-(n2+p) ("diagonal") and out-(p+1) ("previous").  So p + 1 consecutive
// lines of plane p depend on none of each other: the workgroup computes chunks
// of min(p + 1, 2 kWaves) lines, one barrier a chunk, and from plane
// 6 kWaves on the inputs of the next chunk are stored before the current one
// starts and are loaded while it is computed.  Plane 0 (each line reads the
// one before) is the first wave's.  Rows live in a ring of n1 + n2 + 2
// kWaves rows per workgroup (a chunk's stores never reach a row another
// wave still reads); T is int16_t when every cell value is provably below 2^15
// (checked on the host), else int32_t.
//
// Bound by VALU issue (about 25 operations a cell) and, where the longest
// triples run out, by their chunks.  One wave per triple, row after row, took 1
// us a row whatever the batch: 1,024 triples of 100-500 took 268 ms, here 67 (for
// costs that leave the packed kernel's range), 53 in the packed kernel below.
constexpr int kBig3 = 1 << 28;
constexpr int kTop3 = 0x7fffffff;
constexpr int cube_lines(int waves) { return 2 * waves; }         // lines of a full chunk
constexpr int cube_ahead(int waves) { return 3 * cube_lines(waves); }   // first plane whose chunks' inputs are three chunks old

__device__ __forceinline__ int c_shr1(int v, int fill) {
  return __builtin_amdgcn_update_dpp(fill, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
}

template <typename T, int R>
struct RingRow {
  static constexpr int kWords = R * (int)sizeof(T) / 4;
  uint32_t w[kWords];
  __device__ __forceinline__ void load(const T *p) {
    static_assert(kWords % 2 == 0, "rows are loaded in 8-byte pieces");
    const uint2 *q = (const uint2 *)p;
#pragma unroll
    for (int i = 0; i < kWords / 2; ++i) {
      const uint2 v = q[i];
      w[2 * i] = v.x;
      w[2 * i + 1] = v.y;
    }
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < kWords; ++i) w[i] = 0;
  }
  // cell j as a non-negative int (inactive cells may hold anything)
  __device__ __forceinline__ int get(int j) const {
    if constexpr (sizeof(T) == 2) return (int)((w[j >> 1] >> (16 * (j & 1))) & 0xffffu);
    else return (int)w[j];
  }
};

template <typename T, int R>
__device__ __forceinline__ void store_ring(T *p, const int (&mm)[R]) {
  constexpr int kWords = R * (int)sizeof(T) / 4;
  uint32_t w[kWords];
#pragma unroll
  for (int i = 0; i < kWords; ++i) {
    if constexpr (sizeof(T) == 2)
      w[i] = __builtin_amdgcn_perm((uint32_t)mm[2 * i + 1], (uint32_t)mm[2 * i], 0x05040100u);
    else
      w[i] = (uint32_t)mm[i];
  }
  uint2 *q = (uint2 *)p;
#pragma unroll
  for (int i = 0; i < kWords / 2; ++i) q[i] = make_uint2(w[2 * i], w[2 * i + 1]);
}

// R 4-bit codes (R/2 bytes at p, aligned to R/2 bytes)
template <int R>
__device__ __forceinline__ void store_codes(uint8_t *p, const uint32_t (&c)[(R + 7) / 8]) {
  if constexpr (R == 4) {
    *(uint16_t *)p = (uint16_t)c[0];
  } else if constexpr (R == 8) {
    *(uint32_t *)p = c[0];
  } else if constexpr (R == 12) {
    uint16_t *q = (uint16_t *)p;
    q[0] = (uint16_t)c[0];
    q[1] = (uint16_t)(c[0] >> 16);
    q[2] = (uint16_t)c[1];
  } else {
    static_assert(R == 16, "row widths are 4, 8, 12 or 16 cells per lane");
    *(uint2 *)p = make_uint2(c[0], c[1]);
  }
}

// One row.  kKind 0: plane 0, line >= 1 (previous-row moves only); 1: line 0
// of a plane >= 1 (upper moves only, the upper row being the reference's
// diagonal pointer there); 2: every other row.  U, D, P: raw values of the
// upper, diagonal and previous rows; tab: the LDS cost table row of s2[r]; z: the
// cells' S3 terms.
// Out: mm (raw values) and the packed move codes.
template <int R, int kKind>
__device__ __forceinline__ void cube_row(const int (&U)[R], const int (&D)[R], const int (&P)[R],
                                         const int (&G3s)[R], const int (&yo)[R], const int2 *tab, const int (&z)[R],
                                         int cP3, int cP1, int cP2, int (&mm)[R], uint32_t (&codes)[(R + 7) / 8]) {
  // cell k-1 of lane 0's first cell does not exist: the fill value makes its
  // moves lose to every real key
  constexpr int kNone = kBig3 >> 3;
  int Ul = 0, Dl = 0, Pl = 0;
  c_dpp_guard();
  if (kKind != 0) Ul = c_shr1(U[R - 1], kNone);
  if (kKind == 2) Dl = c_shr1(D[R - 1], kNone);
  if (kKind != 1) Pl = c_shr1(P[R - 1], kNone);
  int key[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    int2 tb = make_int2(0, 0);
    if (kKind != 1) tb = tab[yo[j]];
    const int ul = j ? U[j - 1] : Ul, dl = j ? D[j - 1] : Dl, pl = j ? P[j - 1] : Pl;
    int k;
    if (kKind == 0) {
      k = min((P[j] << 3) + cP1, (pl << 3) + tb.x);
    } else if (kKind == 1) {
      k = min((U[j] << 3) + cP3, (ul << 3) + z[j]);
    } else {
      k = min(min((U[j] << 3) + cP3, (P[j] << 3) + cP1), (D[j] << 3) + cP2);
      k = min(min(k, (ul << 3) + z[j]), min((pl << 3) + tb.x, (dl << 3) + tb.y));
    }
    key[j] = k;
  }
  // self pass along s3
  int wv[R], lp[R];
  int run = kTop3;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    wv[j] = (key[j] & ~7) - G3s[j];
    run = min(run, wv[j]);
    lp[j] = run;
  }
  const int incl = c_prefix_min(run);
  c_dpp_guard();
  const int excl = c_shr1(incl, kTop3);
  int prev = excl;
#pragma unroll
  for (int j = 0; j < (R + 7) / 8; ++j) codes[j] = 0;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int pm = min(excl, lp[j]);
    const bool ss = prev < wv[j];
    mm[j] = (G3s[j] + pm) >> 3;
    const uint32_t c = ss ? (uint32_t)kSS : (uint32_t)(key[j] & 7);
    codes[j >> 3] |= c << (4 * (j & 7));
    prev = pm;
  }
}

// Inclusive prefix minimum over the wave without the EXEC guard (for use
// inside a block whose EXEC is unchanged since its one guard).
__device__ __forceinline__ int c_prefix_min_ng(int v) {
  constexpr int I = 0x7fffffff;
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x111, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x112, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x114, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x118, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x142, 0xa, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x143, 0xc, 0xf, false));
  return v;
}

// Two consecutive rows of one plane (lines r and r+1 >= 1): independent of
// each other (the lag puts every input of either at least two rows back),
// computed in one block with one EXEC guard so that their dependent chains
// interleave.  The second row's diagonal row is the first row's upper row.
template <int R>
__device__ __forceinline__ void cube_row_pair(const int (&U0)[R], const int (&D0)[R], const int (&P0)[R],
                                              const int2 *tab0, int cP1a, int cP2a, const int (&U1)[R],
                                              const int (&P1)[R], const int2 *tab1, int cP1b, int cP2b,
                                              const int (&G3s)[R], const int (&yo)[R], const int (&z)[R], int cP3,
                                              int (&mm0)[R], uint32_t (&codes0)[(R + 7) / 8], int (&mm1)[R],
                                              uint32_t (&codes1)[(R + 7) / 8]) {
  constexpr int kNone = kBig3 >> 3;
  c_dpp_guard();
  const int Ul0 = c_shr1(U0[R - 1], kNone), Dl0 = c_shr1(D0[R - 1], kNone), Pl0 = c_shr1(P0[R - 1], kNone);
  const int Ul1 = c_shr1(U1[R - 1], kNone), Pl1 = c_shr1(P1[R - 1], kNone);
  int key0[R], key1[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int2 ta = tab0[yo[j]], tb = tab1[yo[j]];
    const int ul0 = j ? U0[j - 1] : Ul0, dl0 = j ? D0[j - 1] : Dl0, pl0 = j ? P0[j - 1] : Pl0;
    const int ul1 = j ? U1[j - 1] : Ul1, dl1 = ul0, pl1 = j ? P1[j - 1] : Pl1;
    int k0 = min(min((U0[j] << 3) + cP3, (P0[j] << 3) + cP1a), (D0[j] << 3) + cP2a);
    k0 = min(min(k0, (ul0 << 3) + z[j]), min((pl0 << 3) + ta.x, (dl0 << 3) + ta.y));
    int k1 = min(min((U1[j] << 3) + cP3, (P1[j] << 3) + cP1b), (U0[j] << 3) + cP2b);
    k1 = min(min(k1, (ul1 << 3) + z[j]), min((pl1 << 3) + tb.x, (dl1 << 3) + tb.y));
    key0[j] = k0;
    key1[j] = k1;
  }
  int wv0[R], lp0[R], wv1[R], lp1[R];
  int run0 = kTop3, run1 = kTop3;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    wv0[j] = (key0[j] & ~7) - G3s[j];
    wv1[j] = (key1[j] & ~7) - G3s[j];
    run0 = min(run0, wv0[j]);
    run1 = min(run1, wv1[j]);
    lp0[j] = run0;
    lp1[j] = run1;
  }
  const int excl0 = c_shr1(c_prefix_min_ng(run0), kTop3);
  const int excl1 = c_shr1(c_prefix_min_ng(run1), kTop3);
  int prev0 = excl0, prev1 = excl1;
#pragma unroll
  for (int j = 0; j < (R + 7) / 8; ++j) codes0[j] = codes1[j] = 0;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int pm0 = min(excl0, lp0[j]), pm1 = min(excl1, lp1[j]);
    const bool ss0 = prev0 < wv0[j], ss1 = prev1 < wv1[j];
    mm0[j] = (G3s[j] + pm0) >> 3;
    mm1[j] = (G3s[j] + pm1) >> 3;
    codes0[j >> 3] |= (ss0 ? (uint32_t)kSS : (uint32_t)(key0[j] & 7)) << (4 * (j & 7));
    codes1[j >> 3] |= (ss1 ? (uint32_t)kSS : (uint32_t)(key1[j] & 7)) << (4 * (j & 7));
    prev0 = pm0;
    prev1 = pm1;
  }
}

template <typename T, int R, int kWaves>
__global__ __launch_bounds__(64 * kWaves, kWaves == kCubeWaves || R < 16 ? 2 : 1) void cube_block_kernel(
    const TripleMeta *__restrict__ meta, const int32_t *__restrict__ order, int n, int *counter,
    const uint8_t *__restrict__ seq, const DevTcm3 *__restrict__ tcm, uint8_t *dm_base, T *scratch,
    int64_t scratch_per_group, int32_t *cost_out) {
  // [b][y] of the planes of one parity: x = cost(gap, b, y)*8 + S1, y = cost(a, b, y)*8 + S2 for the plane's s1
  // symbol a; s_z: cost(a, gap, y)*8 + S3
  __shared__ int2 s_tab[2][32 * 32];
  __shared__ int s_z[2][32];
  __shared__ int s_item;
  constexpr int RS = 64 * R;   // ring row stride (elements)
  constexpr int kThreads = 64 * kWaves, kLines = cube_lines(kWaves), kAhead = cube_ahead(kWaves);
  constexpr int kPer = 1024 / kThreads;   // table entries per thread
  const int lane = c_lane(), wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  T *const ring = scratch + (size_t)blockIdx.x * scratch_per_group;
  const int gap = tcm->gap;
  for (int e = threadIdx.x; e < 1024; e += kThreads)
    s_tab[0][e].x = s_tab[1][e].x = (tcm->cost[gap * 1024 + e] << 3) | kS1;
  for (;;) {
    __syncthreads();   // the previous triple is done in every wave
    if (threadIdx.x == 0) s_item = atomicAdd(counter, 1);
    __syncthreads();
    const int kk = __builtin_amdgcn_readfirstlane(s_item);
    if (kk >= n) break;
    const int t = __builtin_amdgcn_readfirstlane(order[kk]);
    const int64_t off1 = c_uniform64(meta[t].off1), off2 = c_uniform64(meta[t].off2),
                  off3 = c_uniform64(meta[t].off3), dm_off = c_uniform64(meta[t].dm_off);
    const int n1 = __builtin_amdgcn_readfirstlane(meta[t].l1), n2 = __builtin_amdgcn_readfirstlane(meta[t].l2),
              n3 = __builtin_amdgcn_readfirstlane(meta[t].l3),
              dstride = __builtin_amdgcn_readfirstlane(meta[t].dstride);
    // the triples with the most rows bound the launch: their waves issue first
    const int prio = (__builtin_amdgcn_readfirstlane(meta[t].flags) >> 1) & 3;
    if (prio >= 2) __builtin_amdgcn_s_setprio(2);
    else if (prio == 1) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
    const uint8_t *s1 = seq + off1, *s2 = seq + off2, *s3 = seq + off3;
    uint8_t *dm = dm_base + dm_off;
    const int W = n1 + n2 + kLines;
    const int s30 = __builtin_amdgcn_readfirstlane((int)(s3[0] & 31));
    const bool act = lane * R < n3;   // lane holds at least one cell
    // the table of plane p (its part of 1,024 entries per thread)
    int tv[kPer], tz = 0;
    auto table_load = [&](int p) {
      const int a = __builtin_amdgcn_readfirstlane((int)(s1[p] & 31));
#pragma unroll
      for (int q = 0; q < kPer; ++q) tv[q] = tcm->cost[a * 1024 + q * kThreads + (int)threadIdx.x];
      tz = tcm->cost[(a * 32 + gap) * 32 + (lane & 31)];
    };
    auto table_store = [&](int p) {
#pragma unroll
      for (int q = 0; q < kPer; ++q) s_tab[p & 1][q * kThreads + (int)threadIdx.x].y = (tv[q] << 3) | kS2;
      if (threadIdx.x < 32) s_z[p & 1][lane] = (tz << 3) | kS3;
    };
    if (n1 > 1) table_load(1);
    // per-cell symbols of s3 (inactive cells: the gap) and prefix sums of
    // cost(gap, gap, s3[k]) for k >= 1
    int yo[R], G3s[R], z[R];
    {
      int g[R], sum = 0;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int k = lane * R + j;
        const int y = k < n3 ? (int)(s3[k] & 31) : gap;
        yo[j] = y;
        g[j] = (k >= 1 && k < n3) ? (s_tab[0][gap * 32 + y].x >> 3) : 0;
        sum += g[j];
        G3s[j] = sum;
        z[j] = 0;
      }
      const int ex = c_prefix_sum(sum) - sum;
#pragma unroll
      for (int j = 0; j < R; ++j) G3s[j] = (G3s[j] + ex) << 3;
    }
    int mm[R];
    uint32_t codes[(R + 7) / 8];
    // row f (ring row rr) from mm and codes; the last row's last cell is the cost
    const int total = n1 * n2;
    auto store_row = [&](int rr, int f) {
      if (act) {
        store_ring<T, R>(ring + (size_t)rr * RS + lane * R, mm);
        store_codes<R>(dm + (size_t)f * dstride + lane * (R / 2), codes);
      }
      if (f == total - 1) {
        const int jl = (n3 - 1) % R;
        int v = 0;
#pragma unroll
        for (int j = 0; j < R; ++j) v = j == jl ? mm[j] : v;
        cost_out[t] = __builtin_amdgcn_readlane(v, (n3 - 1) / R);   // every lane stores the same value
      }
    };
    if (wv == 0) {
      // plane 0, line 0: the self pass from 0
#pragma unroll
      for (int j = 0; j < R; ++j) mm[j] = G3s[j] >> 3;
#pragma unroll
      for (int j = 0; j < (R + 7) / 8; ++j) codes[j] = kSS * 0x11111111u;
      if (lane == 0) codes[0] = (codes[0] & ~0xfu) | kS2;   // the origin's code is never read
      store_row(0, 0);
      // lines r >= 1 (the previous row is the one just computed)
      for (int r = 1; r < n2; ++r) {
        const int b = __builtin_amdgcn_readfirstlane((int)(s2[r] & 31));
        const int2 *tab = s_tab[0] + b * 32;
        const int cP1 = __builtin_amdgcn_readfirstlane(tab[s30].x) - (kS1 - kP1);
        int P[R];
#pragma unroll
        for (int j = 0; j < R; ++j) P[j] = mm[j];
        cube_row<R, 0>(P, P, P, G3s, yo, tab, z, 0, cP1, 0, mm, codes);
        store_row(r, r);
      }
    }
    if (n1 > 1) table_store(1);
    __syncthreads();
    // planes p >= 1.  in: the inputs of the wave's lines r, r + 1 of a chunk
    // (d: the diagonal row of line r; that of line r + 1 is u0).
    struct Inputs {
      RingRow<T, R> d, u0, u1, p0, p1;
      int b0, b1;
    } in;
    in.d.zero();
    in.u0.zero();
    in.u1.zero();
    in.p0.zero();
    in.p1.zero();
    in.b0 = in.b1 = 0;
    // the chunk's first ring row; lines of the wave
    auto load_inputs = [&](int p, int r, int rr, int lines) {
      if (lines <= 0) return;
      auto row = [&](RingRow<T, R> &x, int back) {
        int i = rr - back;
        i += i < 0 ? W : 0;
        i -= i >= W ? W : 0;
        if (act) x.load(ring + (size_t)i * RS + lane * R);
      };
      row(in.u0, n2 + p - 1);
      if (r >= 1) {
        row(in.d, n2 + p);
        row(in.p0, p + 1);
      }
      in.b0 = s2[r];
      if (lines > 1) {
        row(in.u1, n2 + p - 2);
        row(in.p1, p);
        in.b1 = s2[r + 1];
      }
    };
    int rb = n2;         // ring row of the chunk's first line
    bool ready = false;   // `in` holds the chunk's inputs
    for (int p = 1; p < n1; ++p) {
      const int buf = p & 1;
#pragma unroll
      for (int j = 0; j < R; ++j) z[j] = s_z[buf][yo[j]];
      const int cP3 = __builtin_amdgcn_readfirstlane(s_z[buf][s30]) - (kS3 - kP3);
      if (p + 1 < n1) table_load(p + 1);
      const int B = min(p + 1, kLines);
      for (int r0 = 0; r0 < n2; r0 += B) {
        const int len = min(B, n2 - r0);
        const int r = r0 + 2 * wv, lines = len - 2 * wv;
        int rr = rb + 2 * wv;
        rr -= rr >= W ? W : 0;
        if (!ready) load_inputs(p, r, rr, lines);
        Inputs now = in;
        // the next chunk
        int np = p, nr0 = r0 + B, nrb = rb + len;
        nrb -= nrb >= W ? W : 0;
        if (nr0 >= n2) {
          np = p + 1;
          nr0 = 0;
        }
        ready = np < n1 && np >= kAhead;
        if (ready) {
          const int nlen = min(kLines, n2 - nr0);
          int nrr = nrb + 2 * wv;
          nrr -= nrr >= W ? W : 0;
          load_inputs(np, nr0 + 2 * wv, nrr, nlen - 2 * wv);
        }
        if (lines > 0) {
          const int b0 = __builtin_amdgcn_readfirstlane(now.b0) & 31;
          const int b1 = __builtin_amdgcn_readfirstlane(now.b1) & 31;
          const int2 *tab0 = s_tab[buf] + b0 * 32, *tab1 = s_tab[buf] + b1 * 32;
          const int2 c0 = tab0[s30], c1 = tab1[s30];
          const int cP1a = __builtin_amdgcn_readfirstlane(c0.x) - (kS1 - kP1);
          const int cP2a = __builtin_amdgcn_readfirstlane(c0.y) - (kS2 - kP2);
          const int cP1b = __builtin_amdgcn_readfirstlane(c1.x) - (kS1 - kP1);
          const int cP2b = __builtin_amdgcn_readfirstlane(c1.y) - (kS2 - kP2);
          int U0[R], D0[R], P0[R], U1[R], P1[R];
#pragma unroll
          for (int j = 0; j < R; ++j) {
            U0[j] = now.u0.get(j);
            D0[j] = now.d.get(j);
            P0[j] = now.p0.get(j);
            U1[j] = now.u1.get(j);
            P1[j] = now.p1.get(j);
          }
          const int f = p * n2 + r;
          int rr1 = rr + 1;
          rr1 -= rr1 >= W ? W : 0;
          if (r >= 1 && lines > 1) {
            int mm1[R];
            uint32_t codes1[(R + 7) / 8];
            cube_row_pair<R>(U0, D0, P0, tab0, cP1a, cP2a, U1, P1, tab1, cP1b, cP2b, G3s, yo, z, cP3, mm, codes, mm1,
                             codes1);
            store_row(rr, f);
#pragma unroll
            for (int j = 0; j < R; ++j) mm[j] = mm1[j];
#pragma unroll
            for (int q = 0; q < (R + 7) / 8; ++q) codes[q] = codes1[q];
            store_row(rr1, f + 1);
          } else {
            if (r == 0) cube_row<R, 1>(U0, U0, U0, G3s, yo, tab0, z, cP3, 0, 0, mm, codes);
            else cube_row<R, 2>(U0, D0, P0, G3s, yo, tab0, z, cP3, cP1a, cP2a, mm, codes);
            store_row(rr, f);
            if (lines > 1) {
              cube_row<R, 2>(U1, U0, P1, G3s, yo, tab1, z, cP3, cP1b, cP2b, mm, codes);
              store_row(rr1, f + 1);
            }
          }
        }
        if (r0 + B >= n2 && p + 1 < n1) table_store(p + 1);   // (its buffer was plane p - 1's)
        rb = nrb;
        __syncthreads();
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The block kernel in packed 16-bit halves, for triples whose every cell value
// stays below kPackMax: a register holds one cell of the wave's two lines (the
// first in the low half), so that the six candidates, the minima and the
// prefix minimum serve both.  A line without previous or diagonal rows (line 0
// of a plane, plane 0) reads kPackNone in their place, whose candidates lose to
// every real one.  At R = 8 a chunk of two lines takes 307 vector and 117
// scalar instructions of a wave (VALU in use 55% of the time, with two waves a
// SIMD; the rows, 175 GB to and from memory for 1,024 triples, are not the
// bound).  What it took: 66 ms with the same waits as the unpacked kernel (the
// barrier of every chunk then waited for its stores), 55 with counted waits,
// 52 with the chunk's loop free of branches and copies.
// ---------------------------------------------------------------------------
constexpr int kPackMax = 8000, kPackCost = 64, kPackNone = 8100;   // 8 kPackNone + 8 kPackCost + 7 < 2^16
typedef short c3s __attribute__((ext_vector_type(2)));
typedef unsigned short c3u __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t p3_min_u(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(c3u, a), __builtin_bit_cast(c3u, b)));
}
__device__ __forceinline__ uint32_t p3_min_i(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(c3s, a), __builtin_bit_cast(c3s, b)));
}
__device__ __forceinline__ uint32_t p3_add(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(c3u, a) + __builtin_bit_cast(c3u, b));
}
__device__ __forceinline__ uint32_t p3_sub(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(c3u, a) - __builtin_bit_cast(c3u, b));
}
// per half: 8 v + c (c may be uniform)
__device__ __forceinline__ uint32_t p3_key(uint32_t v, uint32_t c) {
  uint32_t r;
  asm("v_pk_mad_u16 %0, %1, 8, %2 op_sel_hi:[1,0,1]" : "=v"(r) : "v"(v), "v"(c));
  return r;
}
__device__ __forceinline__ uint32_t p3_key_s(uint32_t v, uint32_t c) {
  uint32_t r;
  asm("v_pk_mad_u16 %0, %1, 8, %2 op_sel_hi:[1,0,1]" : "=v"(r) : "v"(v), "s"(c));
  return r;
}
// per half: all ones where a < b, signed (written out: the compiler makes two
// compares and selects of it)
__device__ __forceinline__ uint32_t p3_lt(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_sub_i16 %0, %1, %2 clamp" : "=v"(r) : "v"(a), "v"(b));
  asm("v_pk_ashrrev_i16 %0, 15, %0 op_sel_hi:[0,1]" : "+v"(r));
  return r;
}
__device__ __forceinline__ uint32_t p3_lo(uint32_t first, uint32_t second) {   // low halves
  return __builtin_amdgcn_perm(second, first, 0x05040100u);
}
__device__ __forceinline__ uint32_t p3_hi(uint32_t first, uint32_t second) {
  return __builtin_amdgcn_perm(second, first, 0x07060302u);
}
__device__ __forceinline__ uint32_t p3_prefix_min(uint32_t v) {
  constexpr int I = 0x7fff7fff;
  v = p3_min_i(v, (uint32_t)__builtin_amdgcn_update_dpp(I, (int)v, 0x111, 0xf, 0xf, false));
  v = p3_min_i(v, (uint32_t)__builtin_amdgcn_update_dpp(I, (int)v, 0x112, 0xf, 0xf, false));
  v = p3_min_i(v, (uint32_t)__builtin_amdgcn_update_dpp(I, (int)v, 0x114, 0xf, 0xf, false));
  v = p3_min_i(v, (uint32_t)__builtin_amdgcn_update_dpp(I, (int)v, 0x118, 0xf, 0xf, false));
  v = p3_min_i(v, (uint32_t)__builtin_amdgcn_update_dpp(I, (int)v, 0x142, 0xa, 0xf, false));
  v = p3_min_i(v, (uint32_t)__builtin_amdgcn_update_dpp(I, (int)v, 0x143, 0xc, 0xf, false));
  return v;
}

// Two lines.  U, D, P: their upper, diagonal and previous rows; tab0 / tab1:
// the table rows of their s2 symbols (S1 term | S2 term << 16); mm: the values;
// codes[q]: move codes of cells 4q .. 4q + 3 of both lines.
template <int R>
__device__ __forceinline__ void cube_lines(const uint32_t (&U)[R], const uint32_t (&D)[R], const uint32_t (&P)[R],
                                           const uint32_t (&G3)[R], const uint32_t (&z)[R], const int (&yo)[R],
                                           const uint32_t *tab0, const uint32_t *tab1, uint32_t cP3, uint32_t cP1,
                                           uint32_t cP2, uint32_t (&mm)[R], uint32_t (&codes)[R / 4]) {
  constexpr int kNone = kPackNone * 0x00010001;
  c_dpp_guard();
  const uint32_t Ul = (uint32_t)c_shr1((int)U[R - 1], kNone), Dl = (uint32_t)c_shr1((int)D[R - 1], kNone),
                 Pl = (uint32_t)c_shr1((int)P[R - 1], kNone);
  uint32_t key[R], wv[R], lp[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const uint32_t e0 = *(const uint32_t *)((const char *)tab0 + yo[j]), e1 = *(const uint32_t *)((const char *)tab1 + yo[j]);
    const uint32_t ul = j ? U[j ? j - 1 : 0] : Ul, dl = j ? D[j ? j - 1 : 0] : Dl, pl = j ? P[j ? j - 1 : 0] : Pl;
    const uint32_t a = p3_min_u(p3_min_u(p3_key_s(U[j], cP3), p3_key_s(P[j], cP1)), p3_key_s(D[j], cP2));
    const uint32_t b = p3_min_u(p3_min_u(p3_key(ul, z[j]), p3_key(pl, p3_lo(e0, e1))), p3_key(dl, p3_hi(e0, e1)));
    key[j] = p3_min_u(a, b);
  }
  // self pass along s3
  uint32_t run = 0x7fff7fffu;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const c3u v = __builtin_bit_cast(c3u, key[j]) >> (c3u){3, 3};
    wv[j] = p3_sub(__builtin_bit_cast(uint32_t, v), G3[j]);
    run = p3_min_i(run, wv[j]);
    lp[j] = run;
  }
  const uint32_t excl = (uint32_t)c_shr1((int)p3_prefix_min(run), 0x7fff7fff);
  uint32_t prev = excl;
#pragma unroll
  for (int j = 0; j < R / 4; ++j) codes[j] = 0;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const uint32_t pm = p3_min_i(excl, lp[j]);
    // all ones where the cell before plus the self cost is smaller
    const uint32_t m = p3_lt(prev, wv[j]);
    mm[j] = p3_add(G3[j], pm);
    const uint32_t code = ((m & (kSS * 0x00010001u)) | (~m & key[j])) & 0x00070007u;
    codes[j >> 2] |= code << (4 * (j & 3));
    prev = pm;
  }
}

// LDS of a workgroup.  tab: [b][y] of the planes of one parity, cost(gap, b,
// y)*8 + S1 | (cost(a, b, y)*8 + S2) << 16 for the plane's s1 symbol a; z:
// cost(a, gap, y)*8 + S3.
struct CubeLds {
  uint32_t tab[2][32 * 32];
  uint32_t z[2][32];
  int item;
  uint8_t s2[kPackMax];   // (n2 < kPackMax: every cost bound is at least 1)
};

// One triple by the workgroup; tx: the S1 terms of this thread's table entries.
template <int R, int kWaves>
__device__ __forceinline__ void cube_packed_triple(int t, const TripleMeta *__restrict__ meta,
                                                   const uint8_t *__restrict__ seq, const DevTcm3 *__restrict__ tcm,
                                                   uint8_t *dm_base, uint16_t *const ring, int32_t *cost_out, CubeLds &L,
                                                   const uint32_t (&tx)[1024 / (64 * kWaves)], int gap) {
  constexpr int RS = 64 * R;   // ring row stride (elements)
  constexpr int kThreads = 64 * kWaves, kLines = cube_lines(kWaves), kAhead = cube_ahead(kWaves);
  constexpr int kPer = 1024 / kThreads;   // table entries per thread
  uint32_t(&s_tab)[2][32 * 32] = L.tab;
  uint32_t(&s_z)[2][32] = L.z;
  const int lane = c_lane(), wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int64_t off1 = c_uniform64(meta[t].off1), off2 = c_uniform64(meta[t].off2),
                off3 = c_uniform64(meta[t].off3), dm_off = c_uniform64(meta[t].dm_off);
  const int n1 = __builtin_amdgcn_readfirstlane(meta[t].l1), n2 = __builtin_amdgcn_readfirstlane(meta[t].l2),
            n3 = __builtin_amdgcn_readfirstlane(meta[t].l3),
            dstride = __builtin_amdgcn_readfirstlane(meta[t].dstride);
  // the triples with the most rows bound the launch: their waves issue first
  const int prio = (__builtin_amdgcn_readfirstlane(meta[t].flags) >> 1) & 3;
  if (prio >= 2) __builtin_amdgcn_s_setprio(2);
  else if (prio == 1) __builtin_amdgcn_s_setprio(1);
  else __builtin_amdgcn_s_setprio(0);
  const uint8_t *s1 = seq + off1, *s2 = seq + off2, *s3 = seq + off3;
  uint8_t *dm = dm_base + dm_off;
  const int W = n1 + n2 + kLines;
  const int s30 = __builtin_amdgcn_readfirstlane((int)(s3[0] & 31));
  const bool act = lane * R < n3;   // lane holds at least one cell
  int tv[kPer], tz = 0;
  auto table_load = [&](int p) {
    const int a = __builtin_amdgcn_readfirstlane((int)(s1[p] & 31));
#pragma unroll
    for (int q = 0; q < kPer; ++q) tv[q] = tcm->cost[a * 1024 + q * kThreads + (int)threadIdx.x];
    tz = tcm->cost[(a * 32 + gap) * 32 + (lane & 31)];
  };
  auto table_store = [&](int p) {
#pragma unroll
    for (int q = 0; q < kPer; ++q)
      s_tab[p & 1][q * kThreads + (int)threadIdx.x] = tx[q] | ((uint32_t)((tv[q] << 3) | kS2) << 16);
    if (threadIdx.x < 32) s_z[p & 1][lane] = (uint32_t)((tz << 3) | kS3) & 0xffffu;
  };
  for (int k = threadIdx.x; k < n2; k += kThreads) L.s2[k] = s2[k];   // (read after the next barrier)
  if (n1 > 1) table_load(1);
  // byte offsets of the cells' s3 symbols in a table row (inactive cells:
  // the gap), prefix sums of cost(gap, gap, s3[k]) for k >= 1, S3 terms
  int yo[R];
  uint32_t G3[R], z[R];
  {
    int g[R], sum = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int k = lane * R + j;
      const int y = k < n3 ? (int)(s3[k] & 31) : gap;
      yo[j] = 4 * y;
      sum += (k >= 1 && k < n3) ? (int)((s_tab[0][gap * 32 + y] & 0xffffu) >> 3) : 0;
      g[j] = sum;
      z[j] = 0;
    }
    const int ex = c_prefix_sum(sum) - sum;
#pragma unroll
    for (int j = 0; j < R; ++j) G3[j] = (uint32_t)(g[j] + ex) * 0x00010001u;
  }
  constexpr uint32_t kNone2 = kPackNone * 0x00010001u;
  uint32_t mm[R], codes[R / 4];
  const int total = n1 * n2;
  using Low = std::integral_constant<int, 0>;
  using High = std::integral_constant<int, 1>;
  // the last cell of a line of mm
  auto last_cell = [&](auto half) {
    const int jl = (n3 - 1) % R;
    int v = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) v = j == jl ? (int)((mm[j] >> (16 * decltype(half)::value)) & 0xffffu) : v;
    return __builtin_amdgcn_readlane(v, (n3 - 1) / R);
  };
  // plane 0's line f (the low halves)
  auto store_line = [&](int f) {
    uint32_t w[R / 2], c[(R + 7) / 8];
#pragma unroll
    for (int i = 0; i < R / 2; ++i) w[i] = p3_lo(mm[2 * i], mm[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < (R + 7) / 8; ++i) c[i] = p3_lo(codes[2 * i], 2 * i + 1 < R / 4 ? codes[2 * i + 1 < R / 4 ? 2 * i + 1 : 0] : 0u);
    if (act) {
      uint2 *q = (uint2 *)(ring + (size_t)f * RS + lane * R);
#pragma unroll
      for (int i = 0; i < R / 4; ++i) q[i] = make_uint2(w[2 * i], w[2 * i + 1]);
      store_codes<R>(dm + (size_t)f * dstride + lane * (R / 2), c);
    }
    if (f == total - 1) cost_out[t] = last_cell(Low{});   // every lane stores the same value
  };
  if (wv == 0) {
    uint32_t none[R];
    // plane 0, line 0: the self pass from 0
#pragma unroll
    for (int j = 0; j < R; ++j) {
      none[j] = kNone2;
      mm[j] = G3[j];
    }
#pragma unroll
    for (int j = 0; j < R / 4; ++j) codes[j] = kSS * 0x11111111u;
    if (lane == 0) codes[0] = (codes[0] & ~0xfu) | kS2;   // the origin's code is never read
    store_line(0);
    // lines r >= 1 (the previous row is the one just computed)
    for (int r = 1; r < n2; ++r) {
      const int b = __builtin_amdgcn_readfirstlane((int)(s2[r] & 31));
      const uint32_t *tab = s_tab[0] + b * 32;
      const uint32_t cP1 = (__builtin_amdgcn_readfirstlane(tab[s30]) & 0xffffu) - (kS1 - kP1);
      uint32_t P[R];
#pragma unroll
      for (int j = 0; j < R; ++j) P[j] = mm[j];
      cube_lines<R>(none, none, P, G3, z, yo, tab, tab, 0u, cP1, 0u, mm, codes);
      store_line(r);
    }
  }
  if (n1 > 1) table_store(1);
  __syncthreads();
  // Planes p >= 1.  Every chunk of every wave issues the same loads and stores
  // (lanes and lines it does not have are dropped by their offsets), so that the
  // waits can count them: with the next chunk's inputs three chunks old (from
  // plane 6 kWaves on) a wave waits, before its stores, for those of the chunk
  // before -- all older than the loads just issued -- and the barrier waits for
  // nothing else.
  constexpr int kW = R / 2;                  // words of a row per lane
  constexpr int kRowLoads = R <= 8 ? 1 : 2;   // loads of a row
  constexpr int kDrop = 0x7ffffff0;
  const __amdgpu_buffer_rsrc_t rring = __builtin_amdgcn_make_buffer_rsrc(ring, 0, W * RS * 2, 0x00020000);
  const int vring = act ? lane * R * 2 : kDrop, vcode = act ? lane * (R / 2) : kDrop;
  // the inputs of the wave's lines r, r + 1 of a chunk (d: the diagonal row of
  // line r; that of line r + 1 is u0)
  uint32_t iu0[kW], iu1[kW], id[kW], ip0[kW], ip1[kW];
  int ib0 = 0, ib1 = 0;
  auto up = [&](int i) { return i + ((i >> 31) & W); };          // -W .. W - 1 to 0 .. W - 1
  auto down = [&](int i) { return i >= W ? i - W : i; };          // 0 .. 2 W - 1 to 0 .. W - 1
  auto load_row = [&](uint32_t (&w)[kW], int row) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    const int at = row * (RS * 2);
    if constexpr (R == 4) {
      const u2 v = __builtin_amdgcn_raw_buffer_load_b64(rring, vring, at, 0);
      w[0] = v.x;
      w[1] = v.y;
    } else {
      const u4 v = __builtin_amdgcn_raw_buffer_load_b128(rring, vring, at, 0);
      w[0] = v.x;
      w[1] = v.y;
      w[2] = v.z;
      w[3] = v.w;
      if constexpr (R == 12) {
        const u2 x = __builtin_amdgcn_raw_buffer_load_b64(rring, vring + 16, at, 0);
        w[4] = x.x;
        w[5] = x.y;
      } else if constexpr (R == 16) {
        const u4 x = __builtin_amdgcn_raw_buffer_load_b128(rring, vring + 16, at, 0);
        w[4] = x.x;
        w[5] = x.y;
        w[6] = x.z;
        w[7] = x.w;
      }
    }
  };
  auto load_inputs = [&](int p, int r, int rr) {
    const int u = up(rr - (n2 + p - 1)), q = up(rr - (p + 1));
    load_row(iu0, u);
    load_row(id, up(u - 1));
    load_row(ip0, q);
    load_row(iu1, down(u + 1));
    load_row(ip1, down(q + 1));
    ib0 = L.s2[min(r, n2 - 1)];
    ib1 = L.s2[min(r + 1, n2 - 1)];
  };
  // line kHalf of mm and codes: ring row rr, line r of the plane (dropped: off)
  auto store_half = [&](auto half, __amdgpu_buffer_rsrc_t rcode, int rr, int r, bool on) {
    constexpr int kHalf = decltype(half)::value;
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    uint32_t w[kW], c[(R + 7) / 8];
#pragma unroll
    for (int i = 0; i < kW; ++i) w[i] = kHalf ? p3_hi(mm[2 * i], mm[2 * i + 1]) : p3_lo(mm[2 * i], mm[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < (R + 7) / 8; ++i) {
      const uint32_t second = 2 * i + 1 < R / 4 ? codes[2 * i + 1 < R / 4 ? 2 * i + 1 : 0] : 0u;
      c[i] = kHalf ? p3_hi(codes[2 * i], second) : p3_lo(codes[2 * i], second);
    }
    const int vr = on ? vring : kDrop, vc = on ? vcode : kDrop, at = rr * (RS * 2), ac = r * dstride;
    if constexpr (R == 4) __builtin_amdgcn_raw_buffer_store_b64(u2{w[0], w[1]}, rring, vr, at, 0);
    else __builtin_amdgcn_raw_buffer_store_b128(u4{w[0], w[1], w[2], w[3]}, rring, vr, at, 0);
    if constexpr (R == 12) __builtin_amdgcn_raw_buffer_store_b64(u2{w[4], w[5]}, rring, vr + 16, at, 0);
    if constexpr (R == 16) __builtin_amdgcn_raw_buffer_store_b128(u4{w[4], w[5], w[6], w[7]}, rring, vr + 16, at, 0);
    if constexpr (R == 4) {
      __builtin_amdgcn_raw_buffer_store_b16((uint16_t)c[0], rcode, vc, ac, 0);
    } else if constexpr (R == 12) {   // (lanes' codes start at multiples of 6 bytes)
      __builtin_amdgcn_raw_buffer_store_b16((uint16_t)c[0], rcode, vc, ac, 0);
      __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(c[0] >> 16), rcode, vc + 2, ac, 0);
      __builtin_amdgcn_raw_buffer_store_b16((uint16_t)c[1], rcode, vc + 4, ac, 0);
    } else if constexpr (R == 8) {
      __builtin_amdgcn_raw_buffer_store_b32(c[0], rcode, vc, ac, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b64(u2{c[0], c[1]}, rcode, vc, ac, 0);
    }
  };
  int rb = n2;   // ring row of the chunk's first line
  // planes p0 .. p1 - 1; kPrefetch: the first chunk's inputs are on their way,
  // and each chunk issues the loads of the next one (past the last plane: rows
  // that nothing reads)
  auto planes = [&](auto prefetch, int first, int last) {
    constexpr bool kPrefetch = decltype(prefetch)::value;
    for (int p = first; p < last; ++p) {
      const int buf = p & 1;
#pragma unroll
      for (int j = 0; j < R; ++j) z[j] = *(const uint32_t *)((const char *)s_z[buf] + yo[j]) * 0x00010001u;
      const uint32_t cP3 = (__builtin_amdgcn_readfirstlane(s_z[buf][s30]) - (kS3 - kP3)) * 0x00010001u;
      const int cline = (int)s_tab[buf][(lane & 31) * 32 + s30];   // lane b: the table entry of s2 symbol b and s3[0]
      if (p + 1 < n1) table_load(p + 1);
      const __amdgpu_buffer_rsrc_t rcode =
          __builtin_amdgcn_make_buffer_rsrc(dm + (int64_t)p * n2 * dstride, 0, n2 * dstride, 0x00020000);
      const int B = kPrefetch ? kLines : min(p + 1, kLines);
      for (int r0 = 0; r0 < n2; r0 += B) {
        const int len = min(B, n2 - r0);
        const int r = r0 + 2 * wv, lines = len - 2 * wv;
        const int rr = down(rb + 2 * wv);
        if constexpr (!kPrefetch) load_inputs(p, r, rr);
        // line 0 has no previous and no diagonal row (a branch here would copy every input)
        const uint32_t keep = r == 0 ? 0u : 0xffffffffu, none = kNone2 & ~keep;
        uint32_t U[R], D[R], P[R];
#pragma unroll
        for (int i = 0; i < kW; ++i) {
          const uint32_t d = (id[i] & keep) | none, p0 = (ip0[i] & keep) | none;
          U[2 * i] = p3_lo(iu0[i], iu1[i]);
          U[2 * i + 1] = p3_hi(iu0[i], iu1[i]);
          D[2 * i] = p3_lo(d, iu0[i]);
          D[2 * i + 1] = p3_hi(d, iu0[i]);
          P[2 * i] = p3_lo(p0, ip1[i]);
          P[2 * i + 1] = p3_hi(p0, ip1[i]);
        }
        const int b0 = __builtin_amdgcn_readfirstlane(ib0) & 31, b1 = __builtin_amdgcn_readfirstlane(ib1) & 31;
        const int nrb = down(rb + len);
        if constexpr (kPrefetch) {
          __builtin_amdgcn_sched_barrier(0);   // the loads reuse the inputs' registers
          const bool turn = r0 + B >= n2;
          load_inputs(turn ? p + 1 : p, (turn ? 0 : r0 + B) + 2 * wv, down(nrb + 2 * wv));
        }
        if (lines > 0) {
          const uint32_t c0 = (uint32_t)__builtin_amdgcn_readlane(cline, b0), c1 = (uint32_t)__builtin_amdgcn_readlane(cline, b1);
          const uint32_t cP1 = ((c0 & 0xffffu) | (c1 << 16)) - (kS1 - kP1) * 0x00010001u;
          const uint32_t cP2 = ((c0 >> 16) | (c1 & 0xffff0000u)) - (kS2 - kP2) * 0x00010001u;
          cube_lines<R>(U, D, P, G3, z, yo, s_tab[buf] + b0 * 32, s_tab[buf] + b1 * 32, cP3, cP1, cP2, mm, codes);
        }
        if constexpr (kPrefetch) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(5 * kRowLoads) : "memory");
        store_half(Low{}, rcode, rr, r, lines > 0);
        store_half(High{}, rcode, down(rr + 1), r + 1, lines > 1);
        if (r0 + B >= n2 && p + 1 < n1) table_store(p + 1);   // (its buffer was plane p - 1's)
        rb = nrb;
        if constexpr (kPrefetch) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else __syncthreads();
      }
    }
  };
  planes(std::false_type{}, 1, min(n1, kAhead));
  if (n1 > kAhead) {
    load_inputs(kAhead, 2 * wv, down(rb + 2 * wv));
    planes(std::true_type{}, kAhead, n1);
    __syncthreads();   // the last stores
  }
  if (n1 > 1) {   // the last row is still in its wave's mm
    const int at = (n2 - 1) % min(n1, kLines);
    if (wv == at >> 1) {
      const int c = at & 1 ? last_cell(High{}) : last_cell(Low{});
      cost_out[t] = c;   // every lane stores the same value
    }
  }
}

// Every triple of the plan whose n3 <= 64 kMaxR in one work list, the largest
// first: workgroups of different row widths in launches of their own, side by
// side, left a few wide triples waiting for the narrow launch's workgroups (100
// ms against 70).  kMaxR 8: two workgroups a compute unit, 16: one.
template <int kMaxR, int kWaves>
__global__ __launch_bounds__(64 * kWaves, kMaxR <= 8 ? 4 : 2) void cube_packed_kernel(
    const TripleMeta *__restrict__ meta, const int32_t *__restrict__ order, int n, int *counter,
    const uint8_t *__restrict__ seq, const DevTcm3 *__restrict__ tcm, uint8_t *dm_base, uint16_t *scratch,
    int64_t scratch_per_group, int32_t *cost_out) {
  __shared__ CubeLds L;
  uint16_t *const ring = scratch + (size_t)blockIdx.x * scratch_per_group;
  const int gap = tcm->gap;
  constexpr int kPer = 1024 / (64 * kWaves);
  uint32_t tx[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int e = q * 64 * kWaves + (int)threadIdx.x;
    tx[q] = (uint32_t)((tcm->cost[gap * 1024 + e] << 3) | kS1) & 0xffffu;
    L.tab[0][e] = tx[q];   // (plane 0 reads no S2 term that counts)
  }
  for (;;) {
    __syncthreads();   // the previous triple is done in every wave
    if (threadIdx.x == 0) L.item = atomicAdd(counter, 1);
    __syncthreads();
    const int kk = __builtin_amdgcn_readfirstlane(L.item);
    if (kk >= n) break;
    const int t = __builtin_amdgcn_readfirstlane(order[kk]);
    const int c = (__builtin_amdgcn_readfirstlane(meta[t].l3) + 255) >> 8;   // cube_class
    if (c <= 1) cube_packed_triple<4, kWaves>(t, meta, seq, tcm, dm_base, ring, cost_out, L, tx, gap);
    else if (c == 2) cube_packed_triple<8, kWaves>(t, meta, seq, tcm, dm_base, ring, cost_out, L, tx, gap);
    if constexpr (kMaxR > 8) {
      if (c == 3) cube_packed_triple<12, kWaves>(t, meta, seq, tcm, dm_base, ring, cost_out, L, tx, gap);
      else if (c == 4) cube_packed_triple<16, kWaves>(t, meta, seq, tcm, dm_base, ring, cost_out, L, tx, gap);
    }
  }
}

__device__ __forceinline__ void rev_put(uint8_t *base, int &pos, uint32_t &acc, int v) {
  --pos;
  acc |= (uint32_t)(v & 0xff) << (8 * (pos & 3));
  if ((pos & 3) == 0) {
    *(uint32_t *)(base + pos) = acc;
    acc = 0;
  }
}
__device__ __forceinline__ void rev_flush(uint8_t *base, int pos, uint32_t acc) {
  if (pos & 3) *(uint32_t *)(base + (pos & ~3)) = acc;
}

// backtrack_3d + algn_get_median_3d; slots: aligned s1, s2, s3, median.
__global__ void cube_trace_kernel(const TripleMeta *__restrict__ meta, const int32_t *__restrict__ order, int n,
                                  const uint8_t *__restrict__ seq, const DevTcm3 *__restrict__ tcm,
                                  const uint8_t *__restrict__ dm_base, uint8_t *out, int32_t *out_len,
                                  int32_t *status) {
  const int tt = blockIdx.x * blockDim.x + threadIdx.x;
  if (tt >= n) return;
  const int t = order[tt];
  const TripleMeta m = meta[t];
  const uint8_t *s1 = seq + m.off1, *s2 = seq + m.off2, *s3 = seq + m.off3;
  const int l1 = m.l1, l2 = m.l2, l3 = m.l3, gap = tcm->gap;
  const uint8_t *dm = dm_base + m.dm_off;
  uint8_t *o = out + m.out_off;
  int pos[3] = {m.cap, m.cap, m.cap};
  uint32_t acc[3] = {0, 0, 0};
  const bool nib = m.flags & 1;   // e counts cells; a row holds dstride bytes
  const int64_t a_line = nib ? 2 * (int64_t)m.dstride : m.dstride, a_plane = (int64_t)l2 * a_line;
  int64_t e = ((int64_t)l1 * l2 - 1) * a_line + (l3 - 1);
  int i1 = l1 - 1, i2 = l2 - 1, i3 = l3 - 1, len = 0, bad = 0;
  int last[3] = {gap, gap, gap};
  // per move index: which sequences advance (bits 0-2) -- P3, P1, P2, S3, S1, S2, SS
  constexpr uint32_t kUse = 1u | (2u << 3) | (3u << 6) | (5u << 9) | (6u << 12) | (7u << 15) | (4u << 18);
  while (e > 0) {
    const int d = nib ? (dm[e >> 1] >> (4 * (e & 1))) & 15 : dm[e];
    if (d > kSS) { bad = 1; break; }
    const uint32_t u = (kUse >> (3 * d)) & 7u;
    const bool m1 = u & 1u, m2 = u & 2u, m3 = u & 4u;
    if ((m1 && i1 < 0) || (m2 && i2 < 0) || (m3 && i3 < 0)) { bad = 1; break; }
    const int x1 = m1 ? (int)s1[i1--] : gap, x2 = m2 ? (int)s2[i2--] : gap, x3 = m3 ? (int)s3[i3--] : gap;
    e -= (m1 ? a_plane : 0) + (m2 ? a_line : 0) + (m3 ? 1 : 0);
    if (len == 0) { last[0] = x1; last[1] = x2; last[2] = x3; }
    rev_put(o, pos[0], acc[0], x1);
    rev_put(o + m.cap, pos[1], acc[1], x2);
    rev_put(o + 2 * m.cap, pos[2], acc[2], x3);
    ++len;
    if (i1 < -1 || i2 < -1 || i3 < -1 || len > m.cap) { bad = 1; break; }
  }
  for (int q = 0; q < 3; ++q) rev_flush(o + q * m.cap, pos[q], acc[q]);
  // median_3 over the aligned triple: a constant sequence (the reference
  // never moves its end pointers), one symbol per column
  const int med = len > 0 ? tcm->median[((last[0] & 31) * 32 + (last[1] & 31)) * 32 + (last[2] & 31)] : 0;
  int mp = m.cap;
  uint32_t ma = 0;
  for (int q = 0; q < len; ++q) rev_put(o + 3 * m.cap, mp, ma, med);
  rev_flush(o + 3 * m.cap, mp, ma);
  for (int q = 0; q < 3; ++q) out_len[4 * t + q] = len;
  out_len[4 * t + 3] = len;
  if (bad) atomicAdd(status, 1);
}

hipError_t launch_reset(int *counters, int n, hipStream_t s);

}  // namespace poyg

using namespace poyg;

#define HIP_TRY3(expr)                                                               \
  do {                                                                               \
    hipError_t e_ = (expr);                                                          \
    if (e_ != hipSuccess) {                                                          \
      set_error("%s failed: %s", #expr, hipGetErrorString(e_));                      \
      return POYG_EDEVICE;                                                           \
    }                                                                                \
  } while (0)

// Triple plans are kept apart from pair plans; the C ABI shares poyg_plan
// through a tagged wrapper defined here.
//
// Row classes: a triple with n3 <= 64*R (R = 4, 8, 12, 16) runs in the block
// kernel of that R; longer s3 fall back to cube_fill_kernel (64-cell chunks).
constexpr int kCubeClasses = 5;   // 0: chunked fallback, c >= 1: block kernel with R = 4c
struct TriplePlan {
  poyg_ctx *ctx;
  int n;
  std::vector<int32_t> order;
  std::vector<TripleMeta> meta;
  std::vector<std::pair<int, int>> batches;   // [begin, end) in `order`
  std::vector<int64_t> out_off;
  int64_t out_bytes = 0, cells = 0, dm_bytes = 0;
  int64_t scratch_bytes_per_wave = 0;
  int waves = kCubeWaves;   // of a block kernel's workgroup: kCubeWaves or kCubeFew
  int grid = 1;        // workgroups of a block kernel launch
  int fill_grid = 0;   // waves of the chunked fallback; its scratch follows the fill_at rings of the block kernels
  int fill_at = 0;
  bool narrow = false;   // int16 ring rows
  bool packed = false;   // ... and the packed kernel: one launch for every row class
  bool wide = false;     // ... with triples of more than 512 cells a row
  int group(int k) const { return packed ? std::min(cls[k], 1) : cls[k]; }   // launch of triple k
  std::vector<int> cls;  // row class per triple
  void *d_tcm = nullptr, *d_meta = nullptr, *d_order = nullptr, *d_dm = nullptr, *d_scratch = nullptr,
       *d_ctr = nullptr, *d_status = nullptr;
  hipStream_t stream = nullptr, side = nullptr, side2 = nullptr;
  hipStream_t last_stream = nullptr;   // the stream of the last run (its status is read there)
  hipEvent_t fork = nullptr, join = nullptr, join2 = nullptr;   // row classes run on three streams
  ~TriplePlan() {
    for (void *p : {d_tcm, d_meta, d_order, d_dm, d_scratch, d_ctr, d_status})
      if (p) (void)hipFree(p);
    for (hipEvent_t e : {fork, join, join2})
      if (e) (void)hipEventDestroy(e);
  }
};

static int cube_class(int l3) { return l3 > 1024 ? 0 : (l3 + 255) / 256; }

// Launch ri of a batch uses scratch region ri (launches run side by side).
template <typename T, int R, int kWaves>
static hipError_t launch_rows(const TriplePlan *P, int ri, const int32_t *ord, int nb, int *ctr,
                              const uint8_t *d_seq, int32_t *d_cost, hipStream_t s) {
  const int grid = std::max(1, std::min(P->grid, nb));
  T *scratch = (T *)((uint8_t *)P->d_scratch + (size_t)ri * P->grid * P->scratch_bytes_per_wave);
  hipLaunchKernelGGL((cube_block_kernel<T, R, kWaves>), dim3(grid), dim3(64 * kWaves), 0, s, (const TripleMeta *)P->d_meta, ord, nb, ctr,
                     d_seq, (const DevTcm3 *)P->d_tcm, (uint8_t *)P->d_dm, scratch,
                     (int64_t)(P->scratch_bytes_per_wave / (int64_t)sizeof(T)), d_cost);
  return hipGetLastError();
}

template <typename T, int kWaves>
static hipError_t launch_class(const TriplePlan *P, int c, int ri, const int32_t *ord, int nb, int *ctr,
                               const uint8_t *d_seq, int32_t *d_cost, hipStream_t s) {
  switch (c) {
    case 1: return launch_rows<T, 4, kWaves>(P, ri, ord, nb, ctr, d_seq, d_cost, s);
    case 2: return launch_rows<T, 8, kWaves>(P, ri, ord, nb, ctr, d_seq, d_cost, s);
    case 3: return launch_rows<T, 12, kWaves>(P, ri, ord, nb, ctr, d_seq, d_cost, s);
    default: return launch_rows<T, 16, kWaves>(P, ri, ord, nb, ctr, d_seq, d_cost, s);
  }
}

static hipError_t launch_packed(const TriplePlan *P, int ri, const int32_t *ord, int nb, int *ctr, const uint8_t *d_seq,
                                int32_t *d_cost, hipStream_t s) {
  const int grid = std::max(1, std::min(P->grid, nb));
  uint16_t *scratch = (uint16_t *)((uint8_t *)P->d_scratch + (size_t)ri * P->grid * P->scratch_bytes_per_wave);
  auto *k = P->waves == kCubeWaves ? (P->wide ? cube_packed_kernel<16, kCubeWaves> : cube_packed_kernel<8, kCubeWaves>)
                                   : (P->wide ? cube_packed_kernel<16, kCubeFew> : cube_packed_kernel<8, kCubeFew>);
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * P->waves), 0, s, (const TripleMeta *)P->d_meta, ord, nb, ctr, d_seq,
                     (const DevTcm3 *)P->d_tcm, (uint8_t *)P->d_dm, scratch, P->scratch_bytes_per_wave / 2, d_cost);
  return hipGetLastError();
}

extern "C" {

int poyg_triple_plan_create(poyg_ctx *ctx, const poyg_cm3 *cm3, int32_t n, const int64_t *off_1,
                            const int32_t *len_1, const int64_t *off_2, const int32_t *len_2,
                            const int64_t *off_3, const int32_t *len_3, int device, int cus, void *stream,
                            void *side, void *side2, int64_t dm_budget, int waves_per_cu, void **out) {
  if (!cm3 || n < 0 || !out) return POYG_EINVAL;
  if (cm3->lcm != 5 || cm3->gap != kGap) {
    set_error("poyg_plan_triples: 5-bit DNA matrices only");
    return POYG_EUNSUPPORTED;
  }
  HIP_TRY3(hipSetDevice(device));
  DevTcm3 *dt = new DevTcm3;
  to_dev_tcm3(cm3, dt);
  // cost bounds of the masks a sequence can hold (1..31)
  int64_t maxc = 0, minc = 0;
  for (int a = 1; a < 32; ++a)
    for (int b = 1; b < 32; ++b)
      for (int c = 1; c < 32; ++c) {
        const int64_t v = dt->cost[(a * 32 + b) * 32 + c];
        maxc = std::max(maxc, v);
        minc = std::min(minc, v);
      }
  TriplePlan *P = new TriplePlan;
  P->ctx = ctx;
  P->n = n;
  P->stream = (hipStream_t)stream;
  P->side = (hipStream_t)side;
  P->side2 = (hipStream_t)side2;
  P->meta.resize(n);
  P->out_off.resize(n);
  P->cls.resize(n);
  std::vector<int64_t> cells(n), dmb(n);
  int64_t max_sum = 0;
  for (int k = 0; k < n; ++k) {
    TripleMeta &m = P->meta[k];
    if (len_1[k] < 1 || len_2[k] < 1 || len_3[k] < 1) {
      delete P;
      delete dt;
      set_error("poyg_plan_triples: empty sequence in triple %d", k);
      return POYG_EINVAL;
    }
    m.off1 = off_1[k]; m.off2 = off_2[k]; m.off3 = off_3[k];
    m.l1 = len_1[k]; m.l2 = len_2[k]; m.l3 = len_3[k];
    m.cap = (int32_t)(((int64_t)m.l1 + m.l2 + m.l3 + 1 + 15) & ~15);
    m.out_off = P->out_bytes;
    P->out_off[k] = P->out_bytes;
    P->out_bytes += 4 * (int64_t)m.cap;
    cells[k] = (int64_t)m.l1 * m.l2 * m.l3;
    P->cells += cells[k];
    max_sum = std::max(max_sum, (int64_t)m.l1 + m.l2 + m.l3);
  }
  // every cell value is at most (l1 + l2 + l3) * maxc (a path of single
  // moves), so the row kernel's keys (value * 8 + move) stay below 2^28 and,
  // for non-negative costs below 2^15, the ring rows fit int16
  const bool rows_ok = minc >= 0 && max_sum * std::max<int64_t>(maxc, 1) < (int64_t(1) << 24);
  P->narrow = rows_ok && max_sum * maxc < 32767;
  P->packed = rows_ok && maxc <= kPackCost && max_sum * std::max<int64_t>(maxc, 1) < kPackMax;
  int64_t need = 0;
  for (int k = 0; k < n; ++k) {
    TripleMeta &m = P->meta[k];
    const int c = rows_ok ? cube_class(m.l3) : 0;
    P->cls[k] = c;
    P->wide = P->wide || c > 2;
    // row kernel: 4-bit codes, rows padded to whole lanes' cells; fallback: bytes
    m.dstride = c ? (m.l3 + 4 * c - 1) / (4 * c) * (2 * c) : m.l3;
    m.flags = c ? 1 : 0;
    dmb[k] = (int64_t)m.l1 * m.l2 * m.dstride;
    const int64_t w = (int64_t)m.l1 + m.l2;
    const int64_t bytes = c ? (w + cube_lines(kCubeWaves)) * 64 * 4 * c * (P->narrow ? 2 : 4)
                            : 4 * (w * m.l3 + m.l3 + 64);
    need = std::max(need, bytes);
  }
  P->scratch_bytes_per_wave = (need + 255) & ~(int64_t)255;
  // wave priority: the triples with the most rows (each is one workgroup's serial work)
  {
    int64_t max_rows = 1;
    for (int k = 0; k < n; ++k) max_rows = std::max(max_rows, (int64_t)P->meta[k].l1 * P->meta[k].l2);
    for (int k = 0; k < n; ++k) {
      const int64_t rows = (int64_t)P->meta[k].l1 * P->meta[k].l2;
      const int prio = rows * 2 >= max_rows ? 2 : rows * 4 >= max_rows ? 1 : 0;
      P->meta[k].flags |= prio << 1;
    }
  }
  P->order.resize(n);
  std::iota(P->order.begin(), P->order.end(), 0);
  std::stable_sort(P->order.begin(), P->order.end(), [&](int a, int b) {
    return P->group(a) != P->group(b) ? P->group(a) > P->group(b) : cells[a] > cells[b];
  });
  // split into batches whose direction cubes fit the budget
  int64_t cur = 0;
  int begin = 0;
  for (int q = 0; q < n; ++q) {
    const int k = P->order[q];
    if (cur > 0 && cur + dmb[k] > dm_budget) {
      P->batches.push_back({begin, q});
      begin = q;
      cur = 0;
    }
    P->meta[k].dm_off = cur;
    cur += (dmb[k] + 15) & ~(int64_t)15;
    P->dm_bytes = std::max(P->dm_bytes, cur);
  }
  if (n) P->batches.push_back({begin, n});
  const char *wv = getenv("POYG_CUBE_WAVES_PER_CU");
  const int asked = waves_per_cu > 0 ? waves_per_cu : (wv ? std::max(1, atoi(wv)) : 0);
  const bool one_per_cu = P->packed && P->wide;
  std::vector<CubeRows> rows;
  for (int k = 0; k < n; ++k)
    if (P->cls[k]) rows.push_back(CubeRows{P->meta[k].l1, P->meta[k].l2});
  P->waves = cube_group_waves(rows, cus, asked, one_per_cu);
  const CubeGrid shape = cube_grid(n, cus, asked, one_per_cu, P->waves);
  P->grid = shape.rows;
  hipError_t e = hipSuccess;
  auto A = [&](void **p, size_t b) { if (e == hipSuccess) e = hipMalloc(p, b ? b : 16); };
  A(&P->d_tcm, sizeof(DevTcm3));
  A(&P->d_meta, sizeof(TripleMeta) * (size_t)n);
  A(&P->d_order, sizeof(int32_t) * (size_t)n);
  A(&P->d_dm, (size_t)P->dm_bytes);
  // one scratch region per row class (a batch runs its classes side by side),
  // the chunked fallback's, the last in the order, after the others
  {
    bool seen[kCubeClasses] = {};
    for (int k = 0; k < n; ++k) seen[P->group(k)] = true;
    if (seen[0]) P->fill_grid = shape.fill;
    for (int c = 1; c < kCubeClasses; ++c) P->fill_at += seen[c] ? P->grid : 0;
  }
  A(&P->d_scratch, (size_t)P->scratch_bytes_per_wave * (P->fill_at + P->fill_grid));
  A(&P->d_ctr, 64);
  A(&P->d_status, 64);
  for (hipEvent_t *ev : {&P->fork, &P->join, &P->join2})
    if (e == hipSuccess) e = hipEventCreateWithFlags(ev, hipEventDisableTiming);
  if (e == hipSuccess) e = hipMemcpy(P->d_tcm, dt, sizeof(DevTcm3), hipMemcpyHostToDevice);
  if (e == hipSuccess && n) e = hipMemcpy(P->d_meta, P->meta.data(), sizeof(TripleMeta) * n, hipMemcpyHostToDevice);
  if (e == hipSuccess && n) e = hipMemcpy(P->d_order, P->order.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice);
  delete dt;
  if (e != hipSuccess) {
    set_error("poyg_plan_triples: device setup failed: %s", hipGetErrorString(e));
    delete P;
    return POYG_ENOMEM;
  }
  *out = P;
  return POYG_OK;
}

void poyg_triple_plan_destroy(void *p) { delete (TriplePlan *)p; }
int64_t poyg_triple_plan_out_bytes(void *p) { return ((TriplePlan *)p)->out_bytes; }
int64_t poyg_triple_plan_cells(void *p) { return ((TriplePlan *)p)->cells; }
int poyg_triple_plan_out_offsets(void *p, int64_t *o) {
  TriplePlan *P = (TriplePlan *)p;
  std::copy(P->out_off.begin(), P->out_off.end(), o);
  return POYG_OK;
}

int poyg_triple_plan_run(void *pp, const uint8_t *d_seq, int32_t *d_cost, uint8_t *d_out, int32_t *d_out_len,
                         void *stream, float *fill_ms, float *trace_ms) {
  TriplePlan *P = (TriplePlan *)pp;
  if (!P || !d_seq || !d_cost || !d_out || !d_out_len) return POYG_EINVAL;
  hipStream_t s = stream ? (hipStream_t)stream : P->stream;
  hipEvent_t ev[3];
  const bool timing = fill_ms || trace_ms;
  if (timing)
    for (auto &x : ev) HIP_TRY3(hipEventCreate(&x));
  float f_tot = 0, t_tot = 0;
  // the status counts the failed triples of the whole run (every batch)
  HIP_TRY3(launch_reset((int *)P->d_status, 4, s));
  P->last_stream = s;
  for (auto &b : P->batches) {
    const int nb = b.second - b.first;
    const int32_t *ord = (const int32_t *)P->d_order + b.first;
    if (timing) HIP_TRY3(hipEventRecord(ev[0], s));
    HIP_TRY3(launch_reset((int *)P->d_ctr, 16, s));
    // one launch per row class present in the batch (the order is sorted by
    // class), the classes side by side: the first on the third stream, the
    // last on the run stream, any others on the second
    std::vector<std::pair<int, int>> runs;
    for (int q = b.first; q < b.second;) {
      int q2 = q;
      while (q2 < b.second && P->group(P->order[q2]) == P->group(P->order[q])) ++q2;
      runs.push_back({q, q2});
      q = q2;
    }
    const bool fan = runs.size() > 1 && P->side && P->side2;
    bool used_side = false, used_side2 = false;
    if (fan) {
      HIP_TRY3(hipEventRecord(P->fork, s));
      HIP_TRY3(hipStreamWaitEvent(P->side, P->fork, 0));
      HIP_TRY3(hipStreamWaitEvent(P->side2, P->fork, 0));
    }
    for (size_t ri = 0; ri < runs.size(); ++ri) {
      const int q = runs[ri].first, q2 = runs[ri].second;
      const int c = P->cls[P->order[q]];
      hipStream_t ls = s;
      if (fan && ri + 1 < runs.size()) {
        ls = ri == 0 ? P->side2 : P->side;
        (ri == 0 ? used_side2 : used_side) = true;
      }
      const int32_t *o2 = (const int32_t *)P->d_order + q;
      int *ctr = (int *)P->d_ctr + ri;
      if (c == 0) {
        const int grid = std::max(1, std::min(P->fill_grid, q2 - q));
        hipLaunchKernelGGL(cube_fill_kernel, dim3(grid), dim3(64), 0, ls, (const TripleMeta *)P->d_meta, o2,
                           q2 - q, ctr, d_seq, (const DevTcm3 *)P->d_tcm, (uint8_t *)P->d_dm,
                           (int *)P->d_scratch + (size_t)P->fill_at * (P->scratch_bytes_per_wave / 4),
                           P->scratch_bytes_per_wave / 4, d_cost);
        HIP_TRY3(hipGetLastError());
      } else if (P->packed) {
        HIP_TRY3(launch_packed(P, (int)ri, o2, q2 - q, ctr, d_seq, d_cost, ls));
      } else if (P->waves == kCubeWaves) {
        auto *launch = P->narrow ? launch_class<int16_t, kCubeWaves> : launch_class<int32_t, kCubeWaves>;
        HIP_TRY3(launch(P, c, ri, o2, q2 - q, ctr, d_seq, d_cost, ls));
      } else {
        auto *launch = P->narrow ? launch_class<int16_t, kCubeFew> : launch_class<int32_t, kCubeFew>;
        HIP_TRY3(launch(P, c, ri, o2, q2 - q, ctr, d_seq, d_cost, ls));
      }
    }
    if (used_side) {
      HIP_TRY3(hipEventRecord(P->join, P->side));
      HIP_TRY3(hipStreamWaitEvent(s, P->join, 0));
    }
    if (used_side2) {
      HIP_TRY3(hipEventRecord(P->join2, P->side2));
      HIP_TRY3(hipStreamWaitEvent(s, P->join2, 0));
    }
    if (timing) HIP_TRY3(hipEventRecord(ev[1], s));
    hipLaunchKernelGGL(cube_trace_kernel, dim3((nb + 63) / 64), dim3(64), 0, s, (const TripleMeta *)P->d_meta, ord,
                       nb, d_seq, (const DevTcm3 *)P->d_tcm, (const uint8_t *)P->d_dm, d_out, d_out_len,
                       (int32_t *)P->d_status);
    HIP_TRY3(hipGetLastError());
    if (timing) {
      HIP_TRY3(hipEventRecord(ev[2], s));
      HIP_TRY3(hipEventSynchronize(ev[2]));
      float a = 0, c = 0;
      HIP_TRY3(hipEventElapsedTime(&a, ev[0], ev[1]));
      HIP_TRY3(hipEventElapsedTime(&c, ev[1], ev[2]));
      f_tot += a;
      t_tot += c;
    }
  }
  if (timing) {
    for (auto &x : ev) (void)hipEventDestroy(x);
    if (fill_ms) *fill_ms = f_tot;
    if (trace_ms) *trace_ms = t_tot;
  }
  return POYG_OK;
}

// Failed triples of the last run, read on the stream that run was queued on.
int poyg_triple_plan_status(void *pp, int32_t *bad) {
  TriplePlan *P = (TriplePlan *)pp;
  *bad = 0;
  if (!P->last_stream) return POYG_OK;
  HIP_TRY3(hipMemcpyAsync(bad, P->d_status, sizeof(int32_t), hipMemcpyDeviceToHost, P->last_stream));
  HIP_TRY3(hipStreamSynchronize(P->last_stream));
  return POYG_OK;
}

}  // extern "C"
