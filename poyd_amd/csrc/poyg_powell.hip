// Powell's three-way alignment with affine gaps (powell_3D_align,
// src/ukkCommon.c:110-151): the reference's check-point Ukkonen search
// (src/ukk.checkp.c) as level-synchronous device passes.
//
// A level is one cost d of one search range (doUkkInLimits): 16 consecutive
// lanes per diagonal within the range's reach at cost d.  A cell's value is
// calcUkk's (src/ukk.checkp.c:608-781) over the levels already stored: the
// state's neighbour diagonal at every previous state (the cost without the
// second mismatch when whichCharCost says 1, else one mismatch lower for
// states with a second cost), the same state one cost lower, and for the
// all-match state the furthest state of this level extended along equal
// characters; a candidate wins only when strictly further, in that order.
// The winner's code is stored beside the dist, so the "from" records the
// reference keeps (coordinates in a base case; the check-point cell above the
// band) are walks over the stored levels.
//
// What bounds it is latency: a level depends on the one before, and a search
// of a hundred levels has a few to a hundred thousand diagonals a level, so
// the chip fills only near the end of the first pass.  So a level is one
// launch for all ranges of a depth of the recursion (they do not depend on
// each other), and its chain of memory accesses is short: descriptors of the
// ten levels a cell can reach as uniform loads, then every candidate's cell at
// once, then every candidate's characters at once, then the run of equal
// characters sixteen at a time.  Three sequences of 300 at 10% substitutions
// (cost 126): a search took 35.7 ms with a launch per range and level (844
// of 24.6 us, each candidate read after the one before was judged); it takes
// 5.8 ms, in 295 level launches of 9 us (5.5 us the small ones) and 127 of
// the evaluation sweep of 7.7 us (25.7).
//
// The first pass also finds the reference's check-point cost: the first
// cost d after whose top-level call the cells evaluated so far reach |A| / 2
// (src/ukk.checkp.c:152-170).  The cells Ukk evaluates up to that call are
// those some chain of calls reaches from the end diagonal's all-match cell
// at a cost of at most d: ukk_esweep_kernel gives every cell the least such
// d (its callers are the cell one cost higher, the all-match cell of its
// level, and the cells whose transition lowers the cost onto it), from the
// top level down.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <mutex>
#include <utility>

#include "poyg_internal.h"
#include "poyg_ukk.h"
#include "poyg_wave.h"

namespace poyg {

// The model tables of setup (src/ukkCommon.c:247-330).
void uk_model(int mm, int go, int ge, UkModel *M) {
  int ns = 0;
  int st[kUkStates][3];
  for (int s = 0; s < 27; ++s) {
    const int t[3] = {s % 3, (s / 3) % 3, (s / 9) % 3};   // match 0, del 1, ins 2
    int nm = 0, ni = 0;
    for (int q = 0; q < 3; ++q) {
      nm += t[q] == 0;
      ni += t[q] == 2;
    }
    if (nm == 0 || ni > 1) continue;   // at least one match, at most one insert
    for (int q = 0; q < 3; ++q) st[ns][q] = t[q];
    ++ns;
  }
  M->ns = ns;
  M->mis = mm;
  M->go = go;
  M->ge = ge;
  for (int s = 0; s < ns; ++s) {
    int nm = 0, nd = 0, ni = 0;
    for (int q = 0; q < 3; ++q) {
      nm += st[s][q] == 0;
      nd += st[s][q] == 1;
      ni += st[s][q] == 2;
    }
    // no insert: the matching sequences advance; one insert: only it does
    int nb = 0;
    for (int q = 0; q < 3; ++q) nb |= (ni ? st[s][q] == 2 : st[s][q] == 0) << q;
    M->nb[s] = nb;
    if (ni) {
      M->cont[s] = ge;
      M->second[s] = 0;
    } else if (nm == 3) {
      M->cont[s] = mm;
      M->second[s] = 1;
    } else if (nd == 1) {
      M->cont[s] = ge;
      M->second[s] = 1;
    } else {
      M->cont[s] = 2 * ge;
      M->second[s] = 0;
    }
  }
  int max_step = 0;
  for (int a = 0; a < ns; ++a)
    for (int b = 0; b < ns; ++b) {
      int c = 0, nm = 0;
      for (int q = 0; q < 3; ++q) {
        if (st[b][q] != 0 && st[b][q] != st[a][q]) c += go;
        nm += st[b][q] == 0;
      }
      M->trans[a][b] = c;
      max_step = std::max(max_step, c + M->cont[b] + mm * (nm - 1));
    }
  M->max_step = max_step;
}

namespace {

// A workgroup takes 16 diagonals of 16 states, a row of 16 lanes each.
constexpr int kUkBlock = 256;
constexpr int kUkDiags = kUkBlock / kUkStates;

// Row-wise (16 lanes) exchange partners whose masks generate all lanes of a row.
__device__ __forceinline__ int row_x8(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x128 /* row_ror:8 */, 0xf, 0xf, false); }
__device__ __forceinline__ int row_x7(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x141 /* row_half_mirror */, 0xf, 0xf, false); }
__device__ __forceinline__ int row_x2(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x4e /* quad_perm 2,3,0,1 */, 0xf, 0xf, false); }
__device__ __forceinline__ int row_x1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0xb1 /* quad_perm 1,0,3,2 */, 0xf, 0xf, false); }

// v[s] of lane l is l's part of result s; lane s of each row of 16 gets result
// s.  Each step halves the results a lane still holds: 15 exchanges, against
// the 64 of sixteen separate row reductions.
template <typename Op>
__device__ __forceinline__ int row_transpose_reduce(int (&v)[16], int l, Op op) {
  dpp_exec_guard();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int lo = v[i], hi = v[i + 8];
    const int keep = l & 8 ? hi : lo, give = l & 8 ? lo : hi;
    v[i] = op(keep, row_x8(give));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lo = v[i], hi = v[i + 4];
    const int keep = l & 4 ? hi : lo, give = l & 4 ? lo : hi;
    v[i] = op(keep, row_x7(give));
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int lo = v[i], hi = v[i + 2];
    const int keep = l & 2 ? hi : lo, give = l & 2 ? lo : hi;
    v[i] = op(keep, row_x2(give));
  }
  const int lo = v[0], hi = v[1];
  const int keep = l & 1 ? hi : lo, give = l & 1 ? lo : hi;
  return op(keep, row_x1(give));
}

__device__ __forceinline__ int row_max(int v) {
  dpp_exec_guard();
  v = max(v, row_x8(v));
  v = max(v, row_x7(v));
  v = max(v, row_x2(v));
  return max(v, row_x1(v));
}

struct OpMax { __device__ __forceinline__ int operator()(int a, int b) const { return max(a, b); } };
struct OpMin { __device__ __forceinline__ int operator()(int a, int b) const { return min(a, b); } };

// State s's three digits, two bits a state, as constants indexed by a lane's state.
constexpr uint32_t uk_digits(int q) {
  uint32_t v = 0;
  for (int s = 0; s < kUkStates; ++s) v |= (uint32_t)kUkTable.t[s][q] << (2 * s);
  return v;
}
constexpr uint64_t uk_steps() {
  uint64_t v = 0;
  for (int s = 0; s < kUkStates; ++s) v |= (uint64_t)uk_step(s) << (4 * s);
  return v;
}
constexpr uint32_t uk_kinds() {
  uint32_t v = 0;
  for (int s = 0; s < kUkStates; ++s) v |= (uint32_t)uk_cont_kind(s) << (2 * s);
  return v;
}
constexpr int uk_bits(int nb) { return (nb & 1) + ((nb >> 1) & 1) + ((nb >> 2) & 1); }

// A level as the candidates see it: uniform, in scalar registers.
typedef int i32x4 __attribute__((ext_vector_type(4)));
struct UkView {
  int64_t org;
  int nac;
  int reach;   // -1: the level lies below the range
};

__device__ __forceinline__ UkView uk_view(const UkLevel *lev, int t) {
  const i32x4 v = *(const i32x4 *)(lev + max(t, 0));
  // (one load of sixteen bytes; here, so that all levels' loads are issued before the first use)
  return UkView{(int64_t)((uint64_t)(uint32_t)v.x | ((uint64_t)(uint32_t)v.y << 32)), v.z, t < 0 ? -1 : v.w};
}

// withinMatrix: the range's start can reach diagonal (ab, ac) at cost c.
__device__ __forceinline__ bool uk_within(const UkRange &r, int go, int ge, int ab, int ac, int c) {
  int x = abs(r.sab - ab), y = abs(r.sac - ac), z = abs((r.sac - r.sab) - (ac - ab));
  // the two smallest of three
  const int g = min(x, min(y, z));
  const int h = max(min(x, y), min(max(x, y), z));
  const int open = r.sstate == 0 ? go : 0;
  const int cheapest = (g ? open : 0) + (h ? open : 0) + (g + h) * ge;
  return cheapest + r.scost <= c;
}

// What a lane knows of its diagonal, as previous state `fs` (its lane in the row).
struct UkLane {
  int fs, ab, ac;
  int neq[3][3];        // neq[q][v]: this lane's state differs from v in sequence q
  int m[8];             // m[nb]: the further offset from the start of the diagonal a step nb back; INT_MAX outside the ends
};

// Previous cell of state S at one level: three levels, by how many of S's
// gaps the lane's state would have to open.
template <int S>
__device__ __forceinline__ uint32_t uk_cand(const UkLane &z, const UkView (&V)[3], const uint32_t *U) {
  constexpr int nb = uk_step(S);
  int k = 0;
#pragma unroll
  for (int q = 0; q < 3; ++q)
    if (kUkTable.t[S][q] != 0) k += z.neq[q][kUkTable.t[S][q]];
  const UkView a = V[0], b = V[1], c = V[2];
  const int reach = k == 0 ? a.reach : k == 1 ? b.reach : c.reach;
  const int nac = k == 0 ? a.nac : k == 1 ? b.nac : c.nac;
  const int64_t org = k == 0 ? a.org : k == 1 ? b.org : c.org;
  const int ab1 = z.ab - (nb & 1) + ((nb >> 1) & 1), ac1 = z.ac - (nb & 1) + ((nb >> 2) & 1);
  // (no branch, so that all candidates' loads are in flight together: a cell
  // outside the level is the store's first word, which is zero)
  return U[z.m[nb] <= reach ? org + ((int64_t)ab1 * nac + ac1) * kUkStates + z.fs : 0];
}

// The candidate's column fits: what okIndex says of the previous cell's dist a.
template <int NB>
__device__ __forceinline__ bool uk_fits(const UkLane &z, const UkRange &r, int a) {
  constexpr int da = NB & 1, db = (NB >> 1) & 1, dc = (NB >> 2) & 1;
  const int b = a - (z.ab - da + db), c = a - (z.ac - da + dc);
  return (min(a, min(b, c)) >= 0) & (a <= r.endA - da) & (b <= r.endB - db) & (c <= r.endC - dc);
}

template <int S>
__device__ __forceinline__ int uk_key(const UkLane &z, const UkRange &r, int a, int v) {
  constexpr int nb = uk_step(S);
  return uk_fits<nb>(z, r, a) ? ((a + (nb & 1) + 1) << 5) | ((15 - z.fs) << 1) | v : 0;
}

// The characters of a column that advances two or three sequences, at the
// cost without the second mismatch.
struct UkColumn {
  int x, y, w;
};

template <int S>
__device__ __forceinline__ UkColumn uk_column(const UkLane &z, const UkRange &r, int a, const char *A, const char *B,
                                              const char *C) {
  constexpr int nb = uk_step(S);
  constexpr int da = nb & 1, db = (nb >> 1) & 1, dc = (nb >> 2) & 1;
  const bool ok = uk_fits<nb>(z, r, a);
  const int b = a - (z.ab - da + db), c = a - (z.ac - da + dc);
  UkColumn o{0, 0, 0};
  if (da) o.x = A[ok ? a : 0];
  if (db) o.y = B[ok ? b : 0];
  if (dc) o.w = C[ok ? c : 0];
  return o;
}

template <int S>
__device__ __forceinline__ bool uk_one_mismatch(const UkColumn &o) {
  constexpr int nb = uk_step(S);
  if (nb == 7) return (int)(o.x == o.y) + (int)(o.x == o.w) + (int)(o.y == o.w) == 1;
  return !(nb & 1) ? o.y == o.w : !(nb & 2) ? o.x == o.w : o.x == o.y;
}

template <int S>
__device__ __forceinline__ void uk_read_state(const UkLane &z, const UkView (&V)[5][3], const uint32_t *U,
                                              uint32_t (&x1)[16], uint32_t (&x2)[16]) {
  // V: the level a mismatch, one and two gap extensions below, and for the
  // first two another mismatch below
  constexpr int kind = uk_cont_kind(S);
  x1[S] = uk_cand<S>(z, V[kind], U);
  if (uk_bits(uk_step(S)) > 1) x2[S] = uk_cand<S>(z, V[3 + (kind == 1)], U);
}

template <int S>
__device__ __forceinline__ void uk_read_column(const UkLane &z, const UkRange &r, const char *A, const char *B,
                                               const char *C, const uint32_t (&x1)[16], UkColumn (&col)[16]) {
  if (uk_bits(uk_step(S)) > 1) col[S] = uk_column<S>(z, r, (int)(x1[S] & 0xffffu) - 1, A, B, C);
}

template <int S>
__device__ __forceinline__ void uk_eval_state(const UkLane &z, const UkRange &r, const UkColumn (&col)[16],
                                              const uint32_t (&x1)[16], const uint32_t (&x2)[16], int (&key)[16]) {
  const int a1 = (int)(x1[S] & 0xffffu) - 1;
  key[S] = uk_key<S>(z, r, a1, 0);
  if (uk_bits(uk_step(S)) > 1) {
    // (a column of one sequence against two gaps always costs one mismatch)
    const int second = uk_key<S>(z, r, (int)(x2[S] & 0xffffu) - 1, 1);
    key[S] = key[S] != 0 && uk_one_mismatch<S>(col[S]) ? key[S] : second;
  }
}

template <int... S>
__device__ __forceinline__ void uk_read_all(std::integer_sequence<int, S...>, const UkLane &z,
                                            const UkView (&V)[5][3], const uint32_t *U, uint32_t (&x1)[16],
                                            uint32_t (&x2)[16]) {
  (uk_read_state<S>(z, V, U, x1, x2), ...);
}

template <int... S>
__device__ __forceinline__ void uk_eval_all(std::integer_sequence<int, S...>, const UkLane &z, const UkRange &r,
                                            const char *A, const char *B, const char *C, const uint32_t (&x1)[16],
                                            const uint32_t (&x2)[16], int (&key)[16]) {
  UkColumn col[16];
  (uk_read_column<S>(z, r, A, B, C, x1, col), ...);
  (uk_eval_state<S>(z, r, col, x1, x2, key), ...);
}

}  // namespace

// Level t (cost scost + t) of every range of the batch (blockIdx.y).  The
// first level at which the range's end condition holds goes to w->reached;
// levels after it are not searched.
//
// A lane is a previous state while the candidates are read (the sixteen lanes
// of a row read one diagonal's sixteen words of at most three levels), and
// the state itself from the transposing reduction on.
__global__ __launch_bounds__(kUkBlock) void ukk_level_kernel(int mis, int go, int ge, const UkJob *__restrict__ jobs,
                                                             int t, const UkLevel *__restrict__ levs,
                                                             int stride, uint32_t *U, const char *__restrict__ A,
                                                             const char *__restrict__ B, const char *__restrict__ C,
                                                             UkWalk *walks) {
  const UkJob J = jobs[blockIdx.y];
  const UkRange r = J.r;
  UkWalk *w = walks + blockIdx.y;
  const UkLevel *lev = levs + (int64_t)blockIdx.y * stride;
  const int c = r.scost + t;
  const UkLevel L = lev[t];
  const int reached = w->reached;
  UkView V[5][3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    V[1][k] = uk_view(lev, t - ge - k * go);
    V[2][k] = uk_view(lev, t - 2 * ge - k * go);
  }
  V[0][0] = uk_view(lev, t - mis);
  V[3][0] = uk_view(lev, t - 2 * mis);
  V[4][0] = uk_view(lev, t - ge - mis);
  V[4][1] = uk_view(lev, t - ge - mis - go);
  // states that open at most none (all match) or one gap never take these
  V[0][1] = V[0][2] = V[0][0];
  V[3][1] = V[3][2] = V[3][0];
  V[4][2] = V[4][1];
  const UkView low = uk_view(lev, t - 1);
  // the descriptors are read before the way out is looked at: one wait, not three
  asm volatile("" ::"s"(V[0][0].org), "s"(V[3][0].org), "s"(V[1][0].org), "s"(V[1][1].org), "s"(V[1][2].org),
               "s"(V[2][0].org), "s"(V[2][1].org), "s"(V[2][2].org), "s"(V[4][0].org), "s"(V[4][1].org),
               "s"(low.org), "s"(reached), "s"(L.org));
  if ((t >= J.nlev) | (reached < c) | ((int64_t)blockIdx.x * kUkDiags >= (int64_t)L.nab * L.nac)) return;
  const int l = (int)threadIdx.x & 15;
  const int64_t diag = (int64_t)blockIdx.x * kUkDiags + ((int)threadIdx.x >> 4);
  const bool act = diag < (int64_t)L.nab * L.nac;
  UkLane z;
  z.fs = l;
  const uint32_t di = (uint32_t)diag;   // (a level holds fewer than 2^32 diagonals)
  z.ab = L.ab_lo + (int)(di / (uint32_t)L.nac);
  z.ac = L.ac_lo + (int)(di % (uint32_t)L.nac);
  const bool in = act & uk_within(r, go, ge, z.ab, z.ac, c);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int d = (int)(uk_digits(q) >> (2 * l)) & 3;
#pragma unroll
    for (int v = 0; v < 3; ++v) z.neq[q][v] = d != v;
  }
#pragma unroll
  for (int nb = 0; nb < 8; ++nb) {
    const int ab1 = z.ab - (nb & 1) + ((nb >> 1) & 1), ac1 = z.ac - (nb & 1) + ((nb >> 2) & 1);
    z.m[nb] = in & (ab1 >= -r.endB) & (ab1 <= r.endA) & (ac1 >= -r.endC) & (ac1 <= r.endA)
                  ? max(abs(ab1 - r.sab), abs(ac1 - r.sac))
                  : INT_MAX;
  }
  uint32_t x1[16], x2[16];
  uk_read_all(std::make_integer_sequence<int, kUkStates>(), z, V, U, x1, x2);
  const bool below = in && max(abs(z.ab - r.sab), abs(z.ac - r.sac)) <= low.reach;
  const uint32_t xl = U[below ? low.org + ((int64_t)z.ab * low.nac + z.ac) * kUkStates + l : 0];
  int key[16];
  uk_eval_all(std::make_integer_sequence<int, kUkStates>(), z, r, A, B, C, x1, x2, key);
  // from here the lane is the state: dist -1 stands for -INFINITY
  const int s = l;
  const int top = row_transpose_reduce(key, l, OpMax());
  int best = (top >> 5) - 1;
  int code = top ? 2 * (15 - ((top >> 1) & 15)) + (top & 1) : kUkNone;
  const int d1 = (int)(xl & 0xffffu) - 1;
  if (d1 > best && d1 - z.ab >= 0 && d1 - z.ac >= 0 && d1 <= r.endA && d1 - z.ab <= r.endB && d1 - z.ac <= r.endC) {
    best = d1;
    code = kUkLower;
  }
  const bool at_start = t == 0 && in && z.ab == r.sab && z.ac == r.sac;
  if (at_start && s == r.sstate) {
    best = r.sdist;
    code = kUkStart;
  }
  // the furthest state of the level (the first of the furthest), extended
  // along equal characters: the row looks at sixteen columns at a time
  const int far = row_max(((best + 1) << 4) | (15 - s));
  int dist = (far >> 4) - 1;
  bool run = in && dist >= 0 && !(at_start && r.sstate == 0);
  while (__ballot(run)) {
    const int a = dist + s, b = a - z.ab, d = a - z.ac;
    const bool eq = run && a < r.endA && b >= 0 && b < r.endB && d >= 0 && d < r.endC && A[a] == B[b] && A[a] == C[d];
    const uint32_t row = (uint32_t)(__ballot(eq) >> (threadIdx.x & 48)) & 0xffffu;
    const int n = __builtin_ctz(~row);
    if (run) dist += n;
    run = run && n == 16;
  }
  if (in && s == 0 && dist > best && !(at_start && r.sstate == 0)) {
    best = dist;
    if ((far & 15) != 15) code = kUkExt + 15 - (far & 15);
  }
  if (in && z.ab == r.fab && z.ac == r.fac) {
    const bool hit = J.target_state < 0 ? s == 0 && t > 0 && dist >= r.fdist   // doUkk's loop starts at cost 1
                                        : s == J.target_state && best >= r.fdist;
    if (hit) atomicMin(&w->reached, c);
  }
  if (act) U[L.base + diag * kUkStates + s] = ((uint32_t)code << 16) | (uint32_t)(best + 1);
}

// First pass, one level from the top down: every cell's first top-level
// cost at which the recursion evaluates it (E), and the least such cost over
// the cells that reach |A| / 2 (w->dstar).  E keeps ring_n levels.
//
// A lane is a calling state while the callers' costs are read: three levels
// (by how many gaps the called state leaves it to open) hold all its words.
__global__ __launch_bounds__(kUkBlock) void ukk_esweep_kernel(int mis, int go, int ge, const UkJob *__restrict__ jobs,
                                                              int t, int final_cost,
                                                              const UkLevel *__restrict__ levs,
                                                              const uint32_t *__restrict__ U, int *E,
                                                              int64_t ring_words, int ring_n, int half, UkWalk *w) {
  __shared__ int s_least[kUkBlock / 64];
  const UkRange r = jobs[0].r;
  const UkLevel *lev = levs;
  const UkLevel L = lev[t];
  const int last = final_cost - r.scost;
  const int seen = w->dstar;
  const int slot = t % ring_n;
  const int l = (int)threadIdx.x & 15;
  const int64_t diag = (int64_t)blockIdx.x * kUkDiags + ((int)threadIdx.x >> 4);
  const bool act = diag < (int64_t)L.nab * L.nac;
  const uint32_t di = (uint32_t)diag;
  const int ab = L.ab_lo + (int)(di / (uint32_t)L.nac), ac = L.ac_lo + (int)(di % (uint32_t)L.nac);
  const int c = r.scost + t;
  const bool in = act & uk_within(r, go, ge, ab, ac, c);
  const int nb = (int)(uk_steps() >> (4 * l)) & 7, kind = (int)(uk_kinds() >> (2 * l)) & 3;
  const int yab = ab + (nb & 1) - ((nb >> 1) & 1), yac = ac + (nb & 1) - ((nb >> 2) & 1);
  const bool inside = in & (yab >= -r.endB) & (yab <= r.endA) & (yac >= -r.endC) & (yac <= r.endA);
  const int m = inside ? max(abs(yab - r.sab), abs(yac - r.sac)) : INT_MAX;
  int x[3], xok = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    int reach = 0, nac = 0;
    int64_t org = 0;
#pragma unroll
    for (int kd = 0; kd < 3; ++kd) {
      const int up = (kd == 0 ? mis : kd * ge) + k * go;   // (at most max_step: fewer than ring_n)
      const UkLevel X = lev[min(t + up, last)];
      const int ring = slot + up >= ring_n ? slot + up - ring_n : slot + up;
      if (kd == kind) {
        reach = t + up <= last ? (int)X.reach : -1;
        nac = X.nac;
        org = X.org - X.base + (int64_t)ring * ring_words;
      }
    }
    // the all-match state opens no gap
    const bool has = m <= reach && (k == 0 || kind != 0);
    xok |= has << k;
    x[k] = E[has ? org + ((int64_t)yab * nac + yac) * kUkStates + l : 0];
  }
  const bool above = in && t + 1 <= last;
  const UkLevel X1 = lev[min(t + 1, last)];
  const int ring1 = slot + 1 == ring_n ? 0 : slot + 1;
  int own = E[above ? (int64_t)ring1 * ring_words + X1.org - X1.base + ((int64_t)ab * X1.nac + ac) * kUkStates + l : 0];
  const uint32_t cell = U[act ? L.base + diag * kUkStates + l : 0] & 0xffffu;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (!((xok >> k) & 1)) x[k] = INT_MAX;
  if (!above) own = INT_MAX;
  int e[16];
#pragma unroll
  for (int s = 0; s < kUkStates; ++s) {
    int k = 0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int d = (int)(uk_digits(q) >> (2 * l)) & 3;
      k += d != 0 && d != kUkTable.t[s][q];
    }
    const int x0 = x[0], x1 = x[1], x2 = x[2];
    e[s] = k == 0 ? x0 : k == 1 ? x1 : x2;
  }
  const int s = l;
  int least = min(row_transpose_reduce(e, l, OpMin()), own);
  if (in && s == 0 && ab == r.fab && ac == r.fac && c >= 1) least = c;   // doUkk's call at cost c (all others are later)
  if (!in) least = INT_MAX;
  // the preset start cell is never evaluated and calls nothing
  const bool at_start = t == 0 && ab == r.sab && ac == r.sac;
  // the all-match cell of this level evaluates every other state of it
  const int match = __shfl(least, threadIdx.x & 48);
  if (s != 0 && !(at_start && r.sstate == 0)) least = min(least, match);
  if (act) E[(int64_t)slot * ring_words + diag * kUkStates + s] = least;
  const bool far = in && !(at_start && s == r.sstate) && (int)cell - 1 >= half && cell != 0;
  const int part = wave_prefix_min(far ? least : INT_MAX);
  if ((threadIdx.x & 63) == 63) s_least[threadIdx.x >> 6] = part;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int all = min(min(s_least[0], s_least[1]), min(s_least[2], s_least[3]));
    if (all < seen) atomicMin(&w->dstar, all);
  }
}

namespace {

// The candidate a cell's code names.
__device__ __forceinline__ void uk_pred(const UkModel &M, int code, int &ab, int &ac, int &c, int &s) {
  if (code < kUkLower) {
    const int fs = code >> 1, v = code & 1;
    const int nb = M.nb[s];
    const int da = nb & 1, db = (nb >> 1) & 1, dc = (nb >> 2) & 1;
    c = c - M.trans[fs][s] - M.cont[s] - v * M.mis;
    ab = ab - da + db;
    ac = ac - da + dc;
    s = fs;
  } else if (code == kUkLower) {
    c -= 1;
  } else {
    s = code - kUkExt;
  }
}

// A range's levels as its walks read them: the descriptors staged in LDS (a
// walk is a serial chain of cells; each then costs one access to memory).
constexpr int kUkStaged = 512;

struct UkCells {
  const UkLevel *lds, *lev;
  const uint32_t *U;
  int scost, nlev;
};

__device__ __forceinline__ uint32_t uk_word(const UkCells &S, int ab, int ac, int c, int s) {
  const int t = c - S.scost;
  if (t < 0 || t >= S.nlev) return (uint32_t)kUkNone << 16;
  const UkLevel L = t < kUkStaged ? S.lds[t] : S.lev[t];
  if (ab < L.ab_lo || ab >= L.ab_lo + L.nab || ac < L.ac_lo || ac >= L.ac_lo + L.nac) return (uint32_t)kUkNone << 16;
  return S.U[L.org + ((int64_t)ab * L.nac + ac) * kUkStates + s];
}

// The check-point split of a range (getSplitRecurse, src/ukk.checkp.c:
// 324-368): from the end cell at the level its loop stopped at, back along
// the winning candidates to the first cell inside [cpcost, cpcost + cpw)
// -- the end cell's "from" record.  first_pass: the end state is the first
// best one and cpcost = dstar + 1 (src/ukk.checkp.c:160-187).
__device__ void uk_split(const UkModel &M, const UkRange &r, const UkCells &S, int cpcost, int cpw, int first_pass,
                         UkWalk *w) {
  const int end = w->reached;
  if (end == INT_MAX || end < r.scost) {
    w->error = 1;
    return;
  }
  int st = r.fstate;
  if (first_pass) {
    int best = -kUkInf;
    st = -1;
    for (int s = 0; s < M.ns; ++s) {
      const uint32_t x = uk_word(S, r.fab, r.fac, end, s) & 0xffffu;
      const int d = x ? (int)x - 1 : -kUkInf;
      if (d > best) {
        best = d;
        st = s;
      }
    }
    w->fstate = st;
    if (w->dstar == INT_MAX) {
      w->error = 2;
      return;
    }
    cpcost = w->dstar + 1;
    if (st < 0) {
      w->error = 3;
      return;
    }
  }
  int ab = r.fab, ac = r.fac, c = end, s = st;
  for (int steps = 0; steps < (1 << 26); ++steps) {
    if (c < cpcost) return;   // no check point: the range is searched whole
    const uint32_t x = uk_word(S, ab, ac, c, s);
    if (c < cpcost + cpw) {
      w->f_ab = ab;
      w->f_ac = ac;
      w->f_cost = c;
      w->f_state = s;
      w->f_dist = (int)(x & 0xffffu) - 1;
      return;
    }
    const int code = (int)(x >> 16);
    if (code == kUkNone || code == kUkStart) return;
    uk_pred(M, code, ab, ac, c, s);
  }
  w->error = 4;
}

// The traceback of a base-case range (traceBack, src/ukk.checkp.c:370-454):
// from the end cell back to the start cell, a run of all-match columns down
// to each candidate's dist, then one column of the cell's state; the range's
// columns go out last first.
__device__ void uk_traceback(const UkModel &M, const UkRange &r, const UkCells &S, const char *A, const char *B,
                             const char *C, char *cols, int cap, UkWalk *w) {
  const int end = w->reached;
  if (end == INT_MAX || end < r.scost) {
    w->error = 5;
    return;
  }
  int n = 0;
  int ab = r.fab, ac = r.fac, c = end, s = r.fstate;
  auto emit = [&](char x, char y, char z) {
    if (n >= cap) return false;
    cols[3 * (int64_t)n] = x;
    cols[3 * (int64_t)n + 1] = y;
    cols[3 * (int64_t)n + 2] = z;
    ++n;
    return true;
  };
  uint32_t x = uk_word(S, ab, ac, c, s);
  while (ab != r.sab || ac != r.sac || c != r.scost || s != r.sstate) {
    const int code = (int)(x >> 16);
    if (code == kUkNone || code == kUkStart || !(x & 0xffffu)) {
      w->error = 6;
      w->ncols = n;
      return;
    }
    int a = (int)(x & 0xffffu) - 1;
    int nab = ab, nac = ac, nc = c, ns = s;
    uk_pred(M, code, nab, nac, nc, ns);
    const uint32_t y = uk_word(S, nab, nac, nc, ns);
    if (!(y & 0xffffu)) {
      w->error = 7;
      w->ncols = n;
      return;
    }
    const int a1 = (int)(y & 0xffffu) - 1;
    int b = a - ab, cc = a - ac;
    const int b1 = a1 - nab, c1 = a1 - nac;
    bool ok = true;
    while (ok && a > a1 && b > b1 && cc > c1) {
      --a;
      --b;
      --cc;
      ok = emit(A[a], B[b], C[cc]);
    }
    if (ok && (a != a1 || b != b1 || cc != c1)) {
      const char p = a > a1 ? A[--a] : '-';
      const char q = b > b1 ? B[--b] : '-';
      const char t = cc > c1 ? C[--cc] : '-';
      ok = emit(p, q, t);
    }
    if (!ok || a != a1 || b != b1 || cc != c1) {
      w->error = 8;
      w->ncols = n;
      return;
    }
    ab = nab;
    ac = nac;
    c = nc;
    s = ns;
    x = y;
  }
  w->ncols = n;
}

}  // namespace

// After a batch's levels: the traceback of each base-case range, the split of
// each other one.  One workgroup a range; its first thread walks.
__global__ __launch_bounds__(kUkBlock) void ukk_walk_kernel(const UkModel *__restrict__ Mg,
                                                            const UkJob *__restrict__ jobs, int cpw,
                                                            const UkLevel *__restrict__ levs, int stride,
                                                            const uint32_t *__restrict__ U,
                                                            const char *__restrict__ A, const char *__restrict__ B,
                                                            const char *__restrict__ C, char *cols, int first_pass,
                                                            UkWalk *walks) {
  __shared__ UkModel M;
  __shared__ UkLevel s_lev[kUkStaged];
  const UkJob J = jobs[blockIdx.x];
  UkWalk *w = walks + blockIdx.x;
  const UkLevel *lev = levs + (int64_t)blockIdx.x * stride;
  for (int e = threadIdx.x; e < (int)(sizeof(UkModel) / 4); e += kUkBlock) ((int *)&M)[e] = ((const int *)Mg)[e];
  for (int e = threadIdx.x; e < min(J.nlev, kUkStaged); e += kUkBlock) s_lev[e] = lev[e];
  __syncthreads();
  if (threadIdx.x != 0) return;
  const UkCells S{s_lev, lev, U, J.r.scost, J.nlev};
  if (J.base_case)
    uk_traceback(M, J.r, S, A, B, C, cols + 3 * (int64_t)J.col0, J.col_cap, w);
  else
    uk_split(M, J.r, S, J.cpcost, cpw, first_pass, w);
}

// Searches may run on several host threads at once (a context each); their
// launches go through one lock, so that the launch path sees one thread at a
// time (the waits, where the time goes, stay concurrent).
static std::mutex g_ukk_launch;

// Costs beyond every level there can be (a level's descriptor takes 64 bytes):
// the kernels add up to four of them in 32 bits.
static int uk_cap(int cost) { return std::min(cost, 1 << 28); }

// diags: the most diagonals any of the n ranges has at level t.
hipError_t launch_ukk_level(const UkModel &M, const UkJob *jobs, int n, int t, int64_t diags, const UkLevel *lev,
                            int stride, uint32_t *U, const char *A, const char *B, const char *C, UkWalk *w, hipStream_t s) {
  std::lock_guard<std::mutex> lock(g_ukk_launch);
  if (diags <= 0 || n <= 0) return hipSuccess;
  const int64_t blocks = (diags + kUkDiags - 1) / kUkDiags;
  hipLaunchKernelGGL(ukk_level_kernel, dim3((unsigned)blocks, (unsigned)n), dim3(kUkBlock), 0, s, uk_cap(M.mis), uk_cap(M.go),
                     uk_cap(M.ge), jobs, t, lev, stride, U, A, B, C, w);
  return hipGetLastError();
}

hipError_t launch_ukk_esweep(const UkModel &M, const UkJob *jobs, int t, int final_cost, int64_t diags,
                             const UkLevel *lev, const uint32_t *U, int *E, int64_t ring_words, int ring_n, int half,
                             UkWalk *w, hipStream_t s) {
  std::lock_guard<std::mutex> lock(g_ukk_launch);
  if (diags <= 0) return hipSuccess;
  const int64_t blocks = (diags + kUkDiags - 1) / kUkDiags;
  hipLaunchKernelGGL(ukk_esweep_kernel, dim3((unsigned)blocks), dim3(kUkBlock), 0, s, uk_cap(M.mis), uk_cap(M.go),
                     uk_cap(M.ge), jobs, t,
                     final_cost, lev, U, E, ring_words, ring_n, half, w);
  return hipGetLastError();
}

hipError_t launch_ukk_walk(const UkModel *M, const UkJob *jobs, int n, int cpw, const UkLevel *lev, int stride,
                           const uint32_t *U, const char *A, const char *B, const char *C, char *cols, int first_pass, UkWalk *w,
                           hipStream_t s) {
  std::lock_guard<std::mutex> lock(g_ukk_launch);
  hipLaunchKernelGGL(ukk_walk_kernel, dim3((unsigned)n), dim3(kUkBlock), 0, s, M, jobs, cpw, lev, stride, U, A, B, C, cols,
                     first_pass, w);
  return hipGetLastError();
}

}  // namespace poyg
