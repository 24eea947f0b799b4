// Wave-level helpers shared by the kernel files: lane and wave indexes, packed
// 16-bit arithmetic, cross-lane moves and sums, LDS ordering, wave-uniform
// copies.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "poyg_internal.h"

namespace poyg {

// ---------------------------------------------------------------------------
// wave helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// Separates DPP moves from any EXEC change before them: eight wait states,
// and the scheduler may move nothing across the barrier.  A DPP issued a few
// instructions after an EXEC restore has been seen to treat enabled source
// lanes as disabled (returning the fill value), depending on how waves
// interleave; every DPP sequence below starts with this guard.
__device__ __forceinline__ void dpp_exec_guard() {
  asm volatile("s_nop 7");
  __builtin_amdgcn_sched_barrier(0);
}

// Two unsigned 16-bit halves in one register (v_pk_* operations).
typedef unsigned short c16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ c16x2 c16v(uint32_t x) { return __builtin_bit_cast(c16x2, x); }
__device__ __forceinline__ uint32_t c16u(c16x2 x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ uint32_t c16_add_sat(uint32_t a, uint32_t b) {
  return c16u(__builtin_elementwise_add_sat(c16v(a), c16v(b)));
}
__device__ __forceinline__ uint32_t c16_sub_sat(uint32_t a, uint32_t b) {
  return c16u(__builtin_elementwise_sub_sat(c16v(a), c16v(b)));
}
__device__ __forceinline__ uint32_t c16_min(uint32_t a, uint32_t b) {
  return c16u(__builtin_elementwise_min(c16v(a), c16v(b)));
}
__device__ __forceinline__ uint32_t c16_add(uint32_t a, uint32_t b) { return c16u(c16v(a) + c16v(b)); }
// per half: b where g == 0, 0xffff where g > 0 (g * 0xffff + b, saturated)
__device__ __forceinline__ uint32_t c16_gate(uint32_t g, uint32_t b) {
  uint32_t r;
  asm("v_pk_mad_u16 %0, %1, -1, %2 clamp" : "=v"(r) : "v"(g), "v"(b));
  return r;
}


// Cross-lane operations use DPP (VALU) and v_readlane only: lane i receives
// lane i-1's value (lane 0 receives `fill`).
__device__ __forceinline__ int shfl_up1(int v, int fill) {
  dpp_exec_guard();
  return __builtin_amdgcn_update_dpp(fill, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
}

// Inclusive prefix minimum over the 64 lanes: Hillis-Steele inside 16-lane
// rows (row_shr 1, 2, 4, 8), then row_bcast:15 and row_bcast:31 carry the
// row totals upward.  Disabled DPP lanes return the identity.
__device__ __forceinline__ int wave_prefix_min(int v) {
  constexpr int I = 0x7fffffff;
  dpp_exec_guard();
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x111, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x112, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x114, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x118, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x142, 0xa, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(I, v, 0x143, 0xc, 0xf, false));
  return v;
}

__device__ __forceinline__ int wave_prefix_sum(int v) {
  dpp_exec_guard();
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

__device__ __forceinline__ int lane63(int v) { return __builtin_amdgcn_readlane(v, kWave - 1); }

// Index of this wave inside its workgroup as a wave-uniform (scalar) value.
// Per-wave LDS regions are addressed from it, so that their base lives in
// scalar registers: a per-lane copy of the base has been seen to go stale in
// some lanes across the divergent code of the fill loops.
__device__ __forceinline__ int wave_in_group() {
  return __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
}

// Orders this wave's LDS traffic across lanes: every LDS access issued
// before the call has completed (s_waitcnt lgkmcnt(0)) before any access
// after it, and the compiler may not move memory operations across it.
// Used between DP rows, where lane j reads what lane j-1 wrote.
__device__ __forceinline__ void wave_sync_mem() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);   // gfx9 encoding of lgkmcnt(0), other counters unchanged
  __builtin_amdgcn_wave_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Ordering of a wave's global row stores before its loads of them on the
// next row, for kernels with one wave per workgroup: workgroup scope needs
// no L2 write-back or invalidate (an agent-scope fence would do both).
__device__ __forceinline__ void wave_fence_global() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup"); }

// Wave-uniform copies of loaded values.  A work item's descriptor is the
// same in every lane; reading it through v_readfirstlane lets the compiler
// keep it in scalar registers and turn every branch on it into a scalar
// branch, instead of EXEC-masked code for control flow that never diverges.
// Together with the rule that no early exit (return, break) of a per-item
// body sits inside lane-divergent code, this keeps the persistent item loops
// scalar.  When that rule was broken (`if (lane == 0) store; return;`), the
// compiler built the item loop as a divergent loop that refreshed VGPR copies
// of the item's geometry under a partial EXEC mask, so some lanes computed
// with the previous item's geometry.
__device__ __forceinline__ int uniform32(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform64(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ PairMeta uniform_meta(const PairMeta *meta, int p) {
  PairMeta m = meta[p];
  m.off_r = uniform64(m.off_r);
  m.off_c = uniform64(m.off_c);
  m.out_off = uniform64(m.out_off);
  m.dm_off = uniform64(m.dm_off);
  m.aux_off = uniform64(m.aux_off);
  m.lr = uniform32(m.lr);
  m.lc = uniform32(m.lc);
  m.stride = uniform32(m.stride);
  m.cap = uniform32(m.cap);
  m.swap = uniform32(m.swap);
  m.p0 = uniform32(m.p0);
  m.p1 = uniform32(m.p1);
  m.p2 = uniform32(m.p2);
  m.p3 = uniform32(m.p3);
  return m;
}

// The one-pair-per-wave fills take the longest pairs, whose run time is
// a chain of dependent steps; when they share SIMDs with the packed
// kernel (whose longest pairs run at priority 2), their waves issue first:
// beside it, the one- and two-set fills of 1,008 long pairs end after 2.6 and
// 4.0 ms, against 4.6 and 6.1 at equal priority.
__device__ __forceinline__ void wave_priority_long_pairs() { __builtin_amdgcn_s_setprio(3); }

__device__ __forceinline__ int next_item(int *counter) {
  int v = 0;
  if (lane_id() == 0) v = atomicAdd(counter, 1);
  return __builtin_amdgcn_readfirstlane(v);
}

}  // namespace poyg
