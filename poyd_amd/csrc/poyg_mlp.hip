// Learned join scorer: 4-mer profiles of sequences, pair features, and a
// 256 -> 256 -> 256 -> 1 ReLU network with bf16 weights and f32
// accumulation, trained and evaluated by the kernels below (bf16 matrix
// products on the MFMA units, 16x16x32 per instruction).  The network only
// orders candidate joins; every join it keeps is scored again by the exact
// alignment DP, so nothing here changes a reported cost.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "poyg_internal.h"

namespace poyg {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kH = 256;   // input width = hidden width

// float -> bf16 with round-to-nearest-even (inputs are finite).
__host__ __device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__host__ __device__ __forceinline__ float bf2f(uint16_t h) {
  const uint32_t u = (uint32_t)h << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// ---------------------------------------------------------------------------
// 4-mer profiles.  A position's base is the lowest base bit of its 5-bit
// mask (A=1, C=2, G=4, T=8); a position with no base bit (the gap) ends
// every window that holds it.  Position 0 (the leading gap) is skipped.
// counts[s][b0*64 + b1*16 + b2*4 + b3] = windows of sequence s.
// One workgroup per sequence, an LDS histogram.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int base_of(uint8_t x) {
  const int b = x & 15;
  return b ? __builtin_ctz(b) : -1;
}

__global__ __launch_bounds__(256) void kmer_count_kernel(const uint8_t *__restrict__ seq,
                                                          const int64_t *__restrict__ off,
                                                          const int32_t *__restrict__ len, int n,
                                                          float *__restrict__ counts) {
  __shared__ int hist[256];
  for (int s = blockIdx.x; s < n; s += gridDim.x) {
    hist[threadIdx.x] = 0;
    __syncthreads();
    const uint8_t *p = seq + off[s];
    const int L = len[s];
    for (int i = 1 + (int)threadIdx.x; i + 3 < L; i += blockDim.x) {
      const int a = base_of(p[i]), b = base_of(p[i + 1]), c = base_of(p[i + 2]), d = base_of(p[i + 3]);
      if ((a | b | c | d) >= 0) atomicAdd(&hist[(a << 6) | (b << 4) | (c << 2) | d], 1);
    }
    __syncthreads();
    counts[(int64_t)s * 256 + threadIdx.x] = (float)hist[threadIdx.x];
    __syncthreads();
  }
}

// x[p][k] = bf16(|counts[ia[p]][k] - counts[ib[p]][k]| * scale).  Half a wave
// takes one pair, eight columns per lane (two 16-byte reads of each profile,
// one 16-byte store): bound by the 512 bytes written per pair and the 2 KB
// read from the profiles in L2.  1,048,576 pairs over 3,000 profiles: 609 us
// with one 2-byte store per thread, 182 us now.
__global__ __launch_bounds__(256) void pair_feature_kernel(const float *__restrict__ counts,
                                                            const int32_t *__restrict__ ia,
                                                            const int32_t *__restrict__ ib, int64_t n,
                                                            float scale, uint16_t *__restrict__ x) {
  const int c = (threadIdx.x & 31) * 8;
  const int64_t step = (int64_t)gridDim.x * 8;
  for (int64_t p = blockIdx.x * (int64_t)8 + (threadIdx.x >> 5); p < n; p += step) {
    const float4 *a = (const float4 *)(counts + (int64_t)ia[p] * 256 + c);
    const float4 *b = (const float4 *)(counts + (int64_t)ib[p] * 256 + c);
    const float4 a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1];
    auto two = [&](float u, float v, float w, float z) {
      return (uint32_t)f2bf(fabsf(u - v) * scale) | ((uint32_t)f2bf(fabsf(w - z) * scale) << 16);
    };
    *(uint4 *)(x + p * 256 + c) = make_uint4(two(a0.x, b0.x, a0.y, b0.y), two(a0.z, b0.z, a0.w, b0.w),
                                             two(a1.x, b1.x, a1.y, b1.y), two(a1.z, b1.z, a1.w, b1.w));
  }
}

// The same one element per thread, for buffers that are not 16-byte aligned.
__global__ __launch_bounds__(256) void pair_feature_any_kernel(const float *__restrict__ counts,
                                                                const int32_t *__restrict__ ia,
                                                                const int32_t *__restrict__ ib, int64_t n,
                                                                float scale, uint16_t *__restrict__ x) {
  for (int64_t p = blockIdx.x; p < n; p += gridDim.x) {
    const float a = counts[(int64_t)ia[p] * 256 + threadIdx.x];
    const float b = counts[(int64_t)ib[p] * 256 + threadIdx.x];
    x[p * 256 + threadIdx.x] = f2bf(fabsf(a - b) * scale);
  }
}

// ---------------------------------------------------------------------------
// C[i][j] = sum_k A(i, k) B(k, j) over bf16 operands with f32 accumulation,
// A(i, k) = A[i*a_rs + k*a_cs], B(k, j) = B[k*b_rs + j*b_cs].  A workgroup
// (four waves) computes a 64 x 64 tile of C; each wave a 32 x 32 quadrant
// as 2 x 2 blocks of v_mfma_f32_16x16x32_bf16.  Operand tiles of 32 k pass
// through LDS in k-contiguous rows (A as [i][k], B as [j][k]), so that the
// MFMA operands are one 16-byte LDS read per lane: lane l holds
// A[l%16][8*(l/16) .. +7] and B[8*(l/16) .. +7][l%16], and receives
// C[4*(l/16) + r][l%16], r = 0..3.  Rows i >= M, columns j >= N and k >= K
// read as zero and are not stored.
// ---------------------------------------------------------------------------
constexpr int kTM = 64, kTN = 64, kTK = 32, kLdsK = kTK + 8;   // row pad: 16 bytes

__device__ __forceinline__ void load_tile(uint16_t (*dst)[kLdsK], const uint16_t *__restrict__ src, int64_t rs,
                                          int64_t cs, int r0, int rmax, int k0, int kmax) {
  const int t = threadIdx.x;
  if (cs == 1 && (rs & 7) == 0 && k0 + kTK <= kmax) {
    // 16-byte loads: thread t takes row t / 4, k chunk (t % 4) * 8
    const int r = t >> 2, kc = (t & 3) * 8;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (r0 + r < rmax) v = *(const uint4 *)(src + (int64_t)(r0 + r) * rs + k0 + kc);
    *(uint4 *)&dst[r][kc] = v;
  } else {
    // element loads; consecutive threads take consecutive rows
    for (int e = t; e < kTM * kTK; e += 256) {
      const int r = e & (kTM - 1), k = e >> 6;
      uint16_t v = 0;
      if (r0 + r < rmax && k0 + k < kmax) v = src[(int64_t)(r0 + r) * rs + (int64_t)(k0 + k) * cs];
      dst[r][k] = v;
    }
  }
}

__global__ __launch_bounds__(256) void gemm_bf16_kernel(int M, int N, int K, const uint16_t *__restrict__ A,
                                                        int64_t a_rs, int64_t a_cs, const uint16_t *__restrict__ B,
                                                        int64_t b_rs, int64_t b_cs, float *__restrict__ out,
                                                        int64_t ldc) {
  __shared__ __attribute__((aligned(16))) uint16_t As[kTM][kLdsK];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[kTN][kLdsK];
  const int i0 = blockIdx.x * kTM, j0 = blockIdx.y * kTN;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int qi = (wv >> 1) * 32, qj = (wv & 1) * 32;
  f32x4 acc[2][2];
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += kTK) {
    __syncthreads();
    load_tile(As, A, a_rs, a_cs, i0, M, k0, K);
    // B(k, j): rows of the LDS tile are columns j, k contiguous
    load_tile(Bs, B, b_cs, b_rs, j0, N, k0, K);
    __syncthreads();
    const int kk = 8 * (lane >> 4);
    bf16x8 av[2], bv[2];
    for (int a = 0; a < 2; ++a) av[a] = *(const bf16x8 *)&As[qi + 16 * a + (lane & 15)][kk];
    for (int b = 0; b < 2; ++b) bv[b] = *(const bf16x8 *)&Bs[qj + 16 * b + (lane & 15)][kk];
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[a], bv[b], acc[a][b], 0, 0, 0);
  }
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + qi + 16 * a + 4 * (lane >> 4) + r;
        const int j = j0 + qj + 16 * b + (lane & 15);
        if (i < M && j < N) out[(int64_t)i * ldc + j] = acc[a][b][r];
      }
}

// ---------------------------------------------------------------------------
// The whole network in one kernel: y = w3 . relu(W2^T relu(W1^T x + b1) + b2)
// + b3.  A workgroup of eight waves takes tiles of 16 RB rows; wave w owns the
// hidden columns 32w .. 32w+31 of both layers and holds its slices of W1 and
// W2 as MFMA operands in 128 VGPRs for the whole launch, so only the rows
// move: x (the next tile loaded while this one is computed) and the first
// layer's activations pass through LDS.  The weights are the A operand, so a
// lane receives four consecutive columns of one row and stores them as one
// 8-byte LDS write.  Bound by LDS reads of the row operand (256 KB per tile
// and layer of RB = 4, as many cycles as the MFMAs take).  The products, their
// order over k and the roundings of the activations are those of one
// v_mfma_f32_16x16x32_bf16 chain per output; the output layer sums in f32.
// RB = 4 for large batches; 1 where tiles of 64 rows would leave compute units
// idle.  1,048,576 rows: 5.6 ms as two products and an output kernel per
// 4,096 rows, 0.29 ms here (950 TFLOP/s).
// ---------------------------------------------------------------------------
constexpr int kNetWaves = 8;
constexpr int kRowPad = kH + 8;   // LDS row of 256 bf16 and 16 bytes of padding

// The bf16 copies of the hidden layers' weights lie in MFMA operand order:
// element (n, k) of the operand A(n, k) = W[k][n] (W[n][k] for the backward
// product) at the place of its 16 x 32 block, lane and half word, so that a
// wave reads an operand as one contiguous kilobyte.
__device__ __forceinline__ int frag_at(int n, int k) {
  return ((n >> 4) * 8 + (k >> 5)) * 512 + (((k >> 3) & 3) * 16 + (n & 15)) * 8 + (k & 7);
}

// A wave's 32 columns of one layer: the A operands of two 16-column blocks.
struct NetSlice {
  bf16x8 a[2][8];
  __device__ __forceinline__ void load(const uint16_t *__restrict__ w, int n0) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int k = 0; k < 8; ++k)
        a[b][k] = *(const bf16x8 *)(w + ((n0 >> 4) + b) * 4096 + 512 * k + 8 * (threadIdx.x & 63));
  }
  // acc[b] = the slice's block b times the 16 rows at `rows` (LDS)
  __device__ __forceinline__ void mul(const uint16_t (*rows)[kRowPad], f32x4 (&acc)[2]) const {
    const int lane = threadIdx.x & 63;
    acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bf16x8 x = *(const bf16x8 *)&rows[lane & 15][32 * k + 8 * (lane >> 4)];
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0][k], x, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1][k], x, acc[1], 0, 0, 0);
    }
  }
};

__device__ __forceinline__ uint2 pack_relu(const f32x4 &v, const float4 &bias) {
  const uint32_t q0 = f2bf(fmaxf(v[0] + bias.x, 0.f)), q1 = f2bf(fmaxf(v[1] + bias.y, 0.f));
  const uint32_t q2 = f2bf(fmaxf(v[2] + bias.z, 0.f)), q3 = f2bf(fmaxf(v[3] + bias.w, 0.f));
  return make_uint2(q0 | (q1 << 16), q2 | (q3 << 16));
}
__device__ __forceinline__ float bf_lo(uint32_t u) { return bf2f((uint16_t)u); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return bf2f((uint16_t)(u >> 16)); }
__device__ __forceinline__ float dot4(const uint2 &h, const float4 &w) {
  return (bf_lo(h.x) * w.x + bf_hi(h.x) * w.y) + (bf_lo(h.y) * w.z + bf_hi(h.y) * w.w);
}
__device__ __forceinline__ float4 load4_bf(const uint16_t *w) {
  const uint2 u = *(const uint2 *)w;
  return make_float4(bf_lo(u.x), bf_hi(u.x), bf_lo(u.y), bf_hi(u.y));
}
// four floats of the parameter vector (its sections are 4-byte aligned only)
__device__ __forceinline__ float4 load4_f(const float *p) { return make_float4(p[0], p[1], p[2], p[3]); }

template <int RB>
__global__ __launch_bounds__(64 * kNetWaves, 2) void net_forward_kernel(
    int64_t n, const uint16_t *__restrict__ x, const uint16_t *__restrict__ w1t, const float *__restrict__ b1,
    const uint16_t *__restrict__ w2t, const float *__restrict__ b2, const uint16_t *__restrict__ w3,
    const float *__restrict__ b3, float *__restrict__ y) {
  constexpr int kRows = 16 * RB;
  constexpr int kChunks = kRows * (kH / 8) / (64 * kNetWaves);   // 16-byte pieces of a tile per thread
  __shared__ __attribute__((aligned(16))) uint16_t xs[2][kRows][kRowPad];
  __shared__ __attribute__((aligned(16))) uint16_t hs[kRows][kRowPad];
  __shared__ float part[kNetWaves][kRows];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int n0 = 32 * wv, c0 = n0 + 4 * (lane >> 4), row = lane & 15;
  NetSlice s1, s2;
  s1.load(w1t, n0);
  s2.load(w2t, n0);
  float4 bias1[2], bias2[2], wo[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    bias1[b] = load4_f(b1 + c0 + 16 * b);
    bias2[b] = load4_f(b2 + c0 + 16 * b);
    wo[b] = load4_bf(w3 + c0 + 16 * b);
  }
  const float bo = b3[0];
  uint4 pre[kChunks];
  auto fetch = [&](int64_t r0) {
#pragma unroll
    for (int q = 0; q < kChunks; ++q) {
      const int e = t + 64 * kNetWaves * q;
      const int64_t r = r0 + (e >> 5);
      pre[q] = r < n ? *(const uint4 *)(x + r * kH + 8 * (e & 31)) : make_uint4(0, 0, 0, 0);
    }
  };
  auto commit = [&](int buf) {
#pragma unroll
    for (int q = 0; q < kChunks; ++q) {
      const int e = t + 64 * kNetWaves * q;
      *(uint4 *)&xs[buf][e >> 5][8 * (e & 31)] = pre[q];
    }
  };
  const int64_t step = (int64_t)gridDim.x * kRows;
  int64_t r0 = (int64_t)blockIdx.x * kRows;
  fetch(r0);
  commit(0);
  __syncthreads();
  int cur = 0;
  for (; r0 < n; r0 += step, cur ^= 1) {
    fetch(r0 + step);   // (rows past the last one read as zero)
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      f32x4 acc[2];
      s1.mul(&xs[cur][16 * m], acc);
#pragma unroll
      for (int b = 0; b < 2; ++b) *(uint2 *)&hs[16 * m + row][c0 + 16 * b] = pack_relu(acc[b], bias1[b]);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      f32x4 acc[2];
      s2.mul(&hs[16 * m], acc);
      float s = dot4(pack_relu(acc[0], bias2[0]), wo[0]) + dot4(pack_relu(acc[1], bias2[1]), wo[1]);
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (lane < 16) part[wv][16 * m + row] = s;
    }
    commit(cur ^ 1);
    __syncthreads();
    if (t < kRows && r0 + t < n) {
      float s = bo;
#pragma unroll
      for (int w = 0; w < kNetWaves; ++w) s += part[w][t];
      y[r0 + t] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// One training step in four launches: net_grad (forward, loss, back-propagated
// errors), net_wgrad (both weight gradients), net_reduce (their partial sums
// and the biases', in a fixed order) and adam (below).  A batch of 4,096 rows
// is too little work for the chip to hide 17 dependent launches (170 us a
// step; the weight gradients' products alone 47 us, reading both operands
// against their layout one element at a time).  Now 38 us: net_grad 16 (bound
// by the 384 KB of weights every workgroup reads from L2; 23 while each product
// waited for its own in 64-byte pieces), net_wgrad 10, net_reduce 7, adam 4.
//
// net_grad: a workgroup of eight waves takes 16 rows (256 workgroups for 4,096
// rows) as net_forward does, keeps both layers' activations in LDS, and goes
// back: with e = y - t, dy = 2 e / n (mean squared error), dZ2[m][k] =
// bf16(dy[m] w3[k]) where H2[m][k] > 0, dZ1 = bf16(dZ2 W2^T) where H1 > 0.
// X, H1, dZ1 and dZ2 are stored transposed (column k: ldt rows, contiguous),
// so that the weight gradients read both operands along their sum; rows n ..
// 16 gridDim.x - 1 are stored as zeros.  Per workgroup, the sums over its rows
// of dZ1, dZ2 and H2 dy go to colpart[block][3][256], those of dy and of the
// loss e^2 / n to rowpart[block][2].
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64 * kNetWaves, 2) void net_grad_kernel(
    int n, const uint16_t *__restrict__ x, const float *__restrict__ t, const uint16_t *__restrict__ w1t,
    const float *__restrict__ b1, const uint16_t *__restrict__ w2t, const float *__restrict__ b2,
    const uint16_t *__restrict__ w2b, const uint16_t *__restrict__ w3, const float *__restrict__ b3,
    uint16_t *__restrict__ xT, uint16_t *__restrict__ h1T, uint16_t *__restrict__ dz1T, uint16_t *__restrict__ dz2T,
    int64_t ldt, float *__restrict__ colpart, float *__restrict__ rowpart) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[16][kRowPad], h1[16][kRowPad], h2[16][kRowPad],
      d1[16][kRowPad], d2[16][kRowPad];
  __shared__ float part[kNetWaves][16], dy[16];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int n0 = 32 * wv, c0 = n0 + 4 * (lane >> 4), row = lane & 15;
  const int r0 = 16 * blockIdx.x;
  const bool live = r0 + row < n;
  NetSlice s1, s2, s3;   // one round of loads for the three products
  s1.load(w1t, n0);
  s2.load(w2t, n0);
  s3.load(w2b, n0);
  {
    const int r = tid >> 5;
    *(uint4 *)&xs[r][8 * (tid & 31)] =
        r0 + r < n ? *(const uint4 *)(x + (int64_t)(r0 + r) * kH + 8 * (tid & 31)) : make_uint4(0, 0, 0, 0);
  }
  __syncthreads();
  f32x4 acc[2];
  s1.mul(xs, acc);
#pragma unroll
  for (int b = 0; b < 2; ++b)
    *(uint2 *)&h1[row][c0 + 16 * b] = live ? pack_relu(acc[b], load4_f(b1 + c0 + 16 * b)) : make_uint2(0, 0);
  __syncthreads();
  s2.mul(h1, acc);
  float4 wo[2];
  uint2 h[2];
  float p = 0.f;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    wo[b] = load4_bf(w3 + c0 + 16 * b);
    h[b] = live ? pack_relu(acc[b], load4_f(b2 + c0 + 16 * b)) : make_uint2(0, 0);
    *(uint2 *)&h2[row][c0 + 16 * b] = h[b];
    p += dot4(h[b], wo[b]);
  }
  p += __shfl_xor(p, 16);
  p += __shfl_xor(p, 32);
  if (lane < 16) part[wv][row] = p;
  __syncthreads();
  float y = b3[0];
#pragma unroll
  for (int w = 0; w < kNetWaves; ++w) y += part[w][row];
  const float e = live ? y - t[r0 + row] : 0.f;
  const float g = 2.f * e / (float)n;
  if (wv == 0) {
    if (lane < 16) dy[row] = g;
    float sg = g, sl = e * e / (float)n;
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
      sg += __shfl_xor(sg, d);
      sl += __shfl_xor(sl, d);
    }
    if (lane == 0) {
      rowpart[2 * blockIdx.x] = sg;
      rowpart[2 * blockIdx.x + 1] = sl;
    }
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    auto q = [&](float hv, float w) { return hv > 0.f ? (uint32_t)f2bf(g * w) : 0u; };   // (h is 0 past the last row)
    *(uint2 *)&d2[row][c0 + 16 * b] =
        make_uint2(q(bf_lo(h[b].x), wo[b].x) | (q(bf_hi(h[b].x), wo[b].y) << 16),
                   q(bf_lo(h[b].y), wo[b].z) | (q(bf_hi(h[b].y), wo[b].w) << 16));
  }
  __syncthreads();
  s3.mul(d2, acc);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const uint2 m = *(const uint2 *)&h1[row][c0 + 16 * b];
    auto q = [&](float hv, float v) { return hv > 0.f ? (uint32_t)f2bf(v) : 0u; };
    *(uint2 *)&d1[row][c0 + 16 * b] = make_uint2(q(bf_lo(m.x), acc[b][0]) | (q(bf_hi(m.x), acc[b][1]) << 16),
                                                 q(bf_lo(m.y), acc[b][2]) | (q(bf_hi(m.y), acc[b][3]) << 16));
  }
  __syncthreads();
  // columns: thread 2c + half takes rows 8 half .. +7 of column c
  const int c = tid >> 1, q0 = 8 * (tid & 1);
  const int64_t at = c * ldt + r0 + q0;
  auto column = [&](const uint16_t (*m)[kRowPad], uint16_t *out) {
    uint32_t v[4];
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t lo = m[q0 + 2 * r][c], hi = m[q0 + 2 * r + 1][c];
      v[r] = lo | (hi << 16);
      sum += bf2f((uint16_t)lo) + bf2f((uint16_t)hi);
    }
    *(uint4 *)(out + at) = make_uint4(v[0], v[1], v[2], v[3]);
    return sum + __shfl_xor(sum, 1);
  };
  column(xs, xT);
  column(h1, h1T);
  const float sb1 = column(d1, dz1T), sb2 = column(d2, dz2T);
  float sw = 0.f;
#pragma unroll
  for (int r = 0; r < 8; ++r) sw += bf2f(h2[q0 + r][c]) * dy[q0 + r];
  sw += __shfl_xor(sw, 1);
  if (q0 == 0) {
    float *o = colpart + (int64_t)blockIdx.x * 3 * kH + c;
    o[0] = sb1;
    o[kH] = sb2;
    o[2 * kH] = sw;
  }
}

// Weight gradients dW1 = X^T dZ1 and dW2 = H1^T dZ2 over rows [chunk z,
// chunk (z + 1)) of `rows` (a multiple of 32) for workgroup (tile, matrix, z):
// a 64 x 64 tile of one of them, each wave a 32 x 32 quadrant, MFMA operands
// read straight from the transposed operands (16 contiguous bytes per lane,
// no LDS: every operand line is used by two waves of the workgroup and comes
// from L2).  Splitting the rows gives the 32 tiles enough workgroups for the
// chip.
constexpr int kWgSplits = 8;
__global__ __launch_bounds__(256) void net_wgrad_kernel(int rows, int chunk, int64_t ldt,
                                                        const uint16_t *__restrict__ xT,
                                                        const uint16_t *__restrict__ h1T,
                                                        const uint16_t *__restrict__ dz1T,
                                                        const uint16_t *__restrict__ dz2T,
                                                        float *__restrict__ part) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int i0 = (blockIdx.x >> 2) * 64 + (wv >> 1) * 32, j0 = (blockIdx.x & 3) * 64 + (wv & 1) * 32;
  const bool second = blockIdx.y == 1;
  const int64_t off = (lane & 15) * ldt + 8 * (lane >> 4);
  const uint16_t *A = (second ? h1T : xT) + i0 * ldt + off, *B = (second ? dz2T : dz1T) + j0 * ldt + off;
  const int k1 = min(rows, (int)(blockIdx.z + 1) * chunk);
  f32x4 acc[2][2];
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = blockIdx.z * chunk; k < k1; k += 32) {
    bf16x8 av[2], bv[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      av[a] = *(const bf16x8 *)(A + 16 * a * ldt + k);
      bv[a] = *(const bf16x8 *)(B + 16 * a * ldt + k);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[a], bv[b], acc[a][b], 0, 0, 0);
  }
  float *o = part + ((int64_t)blockIdx.z * 2 + blockIdx.y) * kH * kH;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[(i0 + 16 * a + 4 * (lane >> 4) + r) * kH + j0 + 16 * b + (lane & 15)] = acc[a][b][r];
}

// dst row r = src row idx[r] (rows of `words` 32-bit words): batch
// shuffles of training data on the device.
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint32_t *__restrict__ src, int words,
                                                          const int32_t *__restrict__ idx, int64_t n,
                                                          uint32_t *__restrict__ dst) {
  for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
    const uint32_t *a = src + (int64_t)idx[r] * words;
    uint32_t *b = dst + r * words;
    for (int w = threadIdx.x; w < words; w += blockDim.x) b[w] = a[w];
  }
}

// Adam over the flat parameter vector, and the bf16 copies the products read
// (frag_at): w1t(n, k) = W1[k][n], w2t(n, k) = W2[k][n], w2b(k, n) = W2[k][n],
// w3b = w3.
struct MlpLayout {
  static constexpr int64_t W1 = 0, B1 = W1 + kH * kH, W2 = B1 + kH, B2 = W2 + kH * kH, W3 = B2 + kH,
                           B3 = W3 + kH, N = B3 + 1;
};

// Sums of a step's partials, each in a fixed order: workgroups 0 .. 511 the
// weight gradients (one element per thread over the splits), the next 48 the
// column sums of b1, b2 and w3 (16 columns by 16 interleaved groups of net_grad
// workgroups, then the groups in order), the last one b3's and the loss.
constexpr int kReduceBlocks = 2 * kH + 3 * kH / 16 + 1;
__global__ __launch_bounds__(256) void net_reduce_kernel(int splits, int tiles, const float *__restrict__ part,
                                                         const float *__restrict__ colpart,
                                                         const float *__restrict__ rowpart, float *__restrict__ g,
                                                         float *__restrict__ loss) {
  __shared__ float sum[2][256];
  const int t = threadIdx.x;
  int b = blockIdx.x;
  if (b < 2 * kH) {
    const int64_t e = (int64_t)(b & (kH - 1)) * 256 + t;
    const float *q = part + (b >> 8) * kH * kH + e;
    float s = 0.f;
    for (int z = 0; z < splits; ++z) s += q[(int64_t)z * 2 * kH * kH];
    g[(b >> 8 ? MlpLayout::W2 : MlpLayout::W1) + e] = s;
    return;
  }
  b -= 2 * kH;
  if (b < 3 * kH / 16) {
    const int sec = b >> 4, c = (b & 15) * 16 + (t & 15), grp = t >> 4;
    float s = 0.f;
    for (int m = grp; m < tiles; m += 16) s += colpart[((int64_t)m * 3 + sec) * kH + c];
    sum[0][t] = s;
    __syncthreads();
    if (t < 16) {
      float r = 0.f;
      for (int q = 0; q < 16; ++q) r += sum[0][16 * q + t];
      g[(sec == 0 ? MlpLayout::B1 : sec == 1 ? MlpLayout::B2 : MlpLayout::W3) + c] = r;
    }
    return;
  }
  float s0 = 0.f, s1 = 0.f;
  for (int m = t; m < tiles; m += 256) {
    s0 += rowpart[2 * m];
    s1 += rowpart[2 * m + 1];
  }
  sum[0][t] = s0;
  sum[1][t] = s1;
  __syncthreads();
  for (int d = 128; d >= 1; d >>= 1) {
    if (t < d) {
      sum[0][t] += sum[0][t + d];
      sum[1][t] += sum[1][t + d];
    }
    __syncthreads();
  }
  if (t == 0) {
    g[MlpLayout::B3] = sum[0][0];
    loss[0] = sum[1][0];
  }
}

// The bf16 copies of parameter i that the products read.
__device__ __forceinline__ void cast_param(int64_t i, float v, uint16_t *w1t, uint16_t *w2t, uint16_t *w2b,
                                           uint16_t *w3b) {
  const uint16_t h = f2bf(v);
  if (i < MlpLayout::B1) {
    w1t[frag_at((int)(i % kH), (int)(i / kH))] = h;
  } else if (i >= MlpLayout::W2 && i < MlpLayout::B2) {
    const int e = (int)(i - MlpLayout::W2), in = e / kH, out = e % kH;
    w2t[frag_at(out, in)] = h;
    w2b[frag_at(in, out)] = h;
  } else if (i >= MlpLayout::W3 && i < MlpLayout::B3) {
    w3b[i - MlpLayout::W3] = h;
  }
}

__global__ __launch_bounds__(256) void adam_kernel(int64_t n, float *__restrict__ p, const float *__restrict__ g,
                                                   float *__restrict__ m1, float *__restrict__ m2, float lr,
                                                   float b1, float b2, float eps, float c1, float c2,
                                                   uint16_t *__restrict__ w1t, uint16_t *__restrict__ w2t,
                                                   uint16_t *__restrict__ w2b, uint16_t *__restrict__ w3b) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    const float v = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    p[i] = v;
    cast_param(i, v, w1t, w2t, w2b, w3b);
  }
}

__global__ __launch_bounds__(256) void cast_params_kernel(const float *__restrict__ p, uint16_t *__restrict__ w1t,
                                                          uint16_t *__restrict__ w2t, uint16_t *__restrict__ w2b,
                                                          uint16_t *__restrict__ w3b) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < MlpLayout::N) cast_param(i, p[i], w1t, w2t, w2b, w3b);
}

}  // namespace poyg

using namespace poyg;

#define HIP_TRYM(expr)                                                                           \
  do {                                                                                           \
    hipError_t e_ = (expr);                                                                      \
    if (e_ != hipSuccess) {                                                                      \
      set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__);      \
      return POYG_EDEVICE;                                                                       \
    }                                                                                            \
  } while (0)

struct poyg_mlp {
  int device = 0;
  int batch_max = 0;
  int cus = 256;
  hipStream_t stream = nullptr;
  int step = 0;   // Adam steps taken
  // f32: params, grads, Adam moments; bf16 copies; batch scratch
  float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
  uint16_t *w1t = nullptr, *w2t = nullptr, *w2b = nullptr, *w3b = nullptr;
  uint16_t *xT = nullptr, *h1T = nullptr, *dz2T = nullptr, *dz1T = nullptr;   // transposed, ldt rows a column
  int64_t ldt = 0;
  float *lsum = nullptr;
  float *cpart = nullptr, *rpart = nullptr;   // net_grad's partial sums per workgroup
  float *wpart = nullptr;                     // net_wgrad's partial products
  ~poyg_mlp() {
    for (void *q : {(void *)p, (void *)g, (void *)m1, (void *)m2, (void *)w1t, (void *)w2t, (void *)w2b,
                    (void *)w3b, (void *)xT, (void *)h1T, (void *)dz2T, (void *)dz1T, (void *)lsum, (void *)cpart,
                    (void *)rpart, (void *)wpart})
      if (q) (void)hipFree(q);
  }
};

extern "C" void *poyg_ctx_stream(poyg_ctx *ctx);
extern "C" int poyg_ctx_device(poyg_ctx *ctx);

extern "C" {

int poyg_mlp_set_params(poyg_mlp *m, const float *host, int64_t n);

int64_t poyg_mlp_param_count(void) { return MlpLayout::N; }

int poyg_mlp_create(poyg_ctx *ctx, int batch_max, uint64_t seed, poyg_mlp **out) {
  if (!ctx || !out || batch_max < 1) {
    set_error("poyg_mlp_create: bad arguments");
    return POYG_EINVAL;
  }
  poyg_mlp *m = new poyg_mlp;
  m->device = poyg_ctx_device(ctx);
  m->stream = (hipStream_t)poyg_ctx_stream(ctx);
  m->batch_max = batch_max;
  m->cus = ctx_cus(ctx);
  hipError_t e = hipSetDevice(m->device);
  // rows of a batch, rounded to the weight gradients' 32, and 32 more so that
  // the columns do not all start in the same memory channel
  const size_t np = (size_t)MlpLayout::N, nb = ((size_t)batch_max + 31) / 32 * 32;
  m->ldt = (int64_t)nb + 32;
  auto A = [&](void **q, size_t bytes) {
    if (e == hipSuccess) e = hipMalloc(q, std::max<size_t>(bytes, 16));
  };
  A((void **)&m->p, 4 * np);
  A((void **)&m->g, 4 * np);
  A((void **)&m->m1, 4 * np);
  A((void **)&m->m2, 4 * np);
  A((void **)&m->w1t, 2 * kH * kH);
  A((void **)&m->w2t, 2 * kH * kH);
  A((void **)&m->w2b, 2 * kH * kH);
  A((void **)&m->w3b, 2 * kH);
  for (uint16_t **q : {&m->xT, &m->h1T, &m->dz2T, &m->dz1T}) A((void **)q, 2 * (size_t)m->ldt * kH);
  A((void **)&m->lsum, 16);
  A((void **)&m->cpart, 4 * 3 * (nb / 16) * kH);
  A((void **)&m->rpart, 4 * 2 * (nb / 16));
  A((void **)&m->wpart, 4 * 2 * (size_t)kWgSplits * kH * kH);
  if (e != hipSuccess) {
    delete m;
    set_error("poyg_mlp_create: hipMalloc failed: %s", hipGetErrorString(e));
    return POYG_ENOMEM;
  }
  // He-uniform weights (bound sqrt(6 / fan_in)), zero biases, from a
  // splitmix64 stream of the seed
  std::vector<float> h(np, 0.f);
  uint64_t z = seed;
  auto next = [&]() {
    z += 0x9e3779b97f4a7c15ull;
    uint64_t x = z;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    x ^= x >> 31;
    return (double)(x >> 11) * (1.0 / 9007199254740992.0);
  };
  const float bound = sqrtf(6.f / kH);
  for (int64_t i = 0; i < kH * kH; ++i) h[MlpLayout::W1 + i] = (float)((2 * next() - 1) * bound);
  for (int64_t i = 0; i < kH * kH; ++i) h[MlpLayout::W2 + i] = (float)((2 * next() - 1) * bound);
  for (int64_t i = 0; i < kH; ++i) h[MlpLayout::W3 + i] = (float)((2 * next() - 1) * bound);
  const int rc = poyg_mlp_set_params(m, h.data(), (int64_t)np);
  if (rc) {
    delete m;
    return rc;
  }
  *out = m;
  return POYG_OK;
}

void poyg_mlp_destroy(poyg_mlp *m) { delete m; }

int poyg_mlp_set_params(poyg_mlp *m, const float *host, int64_t n) {
  if (!m || !host || n != MlpLayout::N) return POYG_EINVAL;
  HIP_TRYM(hipSetDevice(m->device));
  HIP_TRYM(hipMemcpyAsync(m->p, host, 4 * (size_t)n, hipMemcpyHostToDevice, m->stream));
  HIP_TRYM(hipMemsetAsync(m->m1, 0, 4 * (size_t)n, m->stream));
  HIP_TRYM(hipMemsetAsync(m->m2, 0, 4 * (size_t)n, m->stream));
  hipLaunchKernelGGL(cast_params_kernel, dim3((MlpLayout::N + 255) / 256), dim3(256), 0, m->stream, m->p, m->w1t,
                     m->w2t, m->w2b, m->w3b);
  HIP_TRYM(hipGetLastError());
  HIP_TRYM(hipStreamSynchronize(m->stream));
  m->step = 0;
  return POYG_OK;
}

int poyg_mlp_get_params(poyg_mlp *m, float *host, int64_t n) {
  if (!m || !host || n != MlpLayout::N) return POYG_EINVAL;
  HIP_TRYM(hipMemcpyAsync(host, m->p, 4 * (size_t)n, hipMemcpyDeviceToHost, m->stream));
  HIP_TRYM(hipStreamSynchronize(m->stream));
  return POYG_OK;
}

int poyg_mlp_get_grads(poyg_mlp *m, float *host, int64_t n) {
  if (!m || !host || n != MlpLayout::N) return POYG_EINVAL;
  HIP_TRYM(hipMemcpyAsync(host, m->g, 4 * (size_t)n, hipMemcpyDeviceToHost, m->stream));
  HIP_TRYM(hipStreamSynchronize(m->stream));
  return POYG_OK;
}

// y[r] for r < n of bf16 feature rows d_x[r][256] (device), one launch: one
// persistent workgroup per compute unit (its LDS and registers leave room for
// one), tiles of 64 rows where every compute unit gets one.
int poyg_mlp_forward(poyg_mlp *m, const uint16_t *d_x, int64_t n, float *d_y, void *stream) {
  if (!m || (n > 0 && (!d_x || !d_y)) || n < 0) return POYG_EINVAL;
  if (n == 0) return POYG_OK;
  hipStream_t s = stream ? (hipStream_t)stream : m->stream;
  const float *p = m->p;
  const int rb = n >= 64 * (int64_t)m->cus ? 4 : 1;
  const unsigned grid = (unsigned)std::min<int64_t>((n + 16 * rb - 1) / (16 * rb), m->cus);
  auto k = rb == 4 ? net_forward_kernel<4> : net_forward_kernel<1>;
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * kNetWaves), 0, s, n, d_x, m->w1t, p + MlpLayout::B1, m->w2t,
                     p + MlpLayout::B2, m->w3b, p + MlpLayout::B3, d_y);
  HIP_TRYM(hipGetLastError());
  return POYG_OK;
}

// Gradient of the mean squared error over one batch (n <= batch_max rows
// of features d_x and targets d_t), kept for poyg_mlp_adam; the batch's
// loss (mean) goes to *loss when given (a synchronisation).
int poyg_mlp_grad(poyg_mlp *m, const uint16_t *d_x, const float *d_t, int n, float *loss) {
  if (!m || !d_x || !d_t || n < 1 || n > m->batch_max) {
    set_error("poyg_mlp_grad: bad arguments (batch of %d rows, at most %d)", n, m ? m->batch_max : 0);
    return POYG_EINVAL;
  }
  hipStream_t s = m->stream;
  const float *p = m->p;
  const int rows = (n + 31) / 32 * 32, tiles = rows / 16;
  hipLaunchKernelGGL(net_grad_kernel, dim3(tiles), dim3(64 * kNetWaves), 0, s, n, d_x, d_t, m->w1t, p + MlpLayout::B1,
                     m->w2t, p + MlpLayout::B2, m->w2b, m->w3b, p + MlpLayout::B3, m->xT, m->h1T, m->dz1T, m->dz2T,
                     m->ldt, m->cpart, m->rpart);
  // at least four steps of 32 rows per split
  const int want = std::max(1, std::min(kWgSplits, rows / 128));
  const int chunk = (rows / 32 + want - 1) / want * 32, splits = (rows + chunk - 1) / chunk;
  hipLaunchKernelGGL(net_wgrad_kernel, dim3(16, 2, splits), dim3(256), 0, s, rows, chunk, m->ldt, m->xT, m->h1T,
                     m->dz1T, m->dz2T, m->wpart);
  hipLaunchKernelGGL(net_reduce_kernel, dim3(kReduceBlocks), dim3(256), 0, s, splits, tiles, m->wpart, m->cpart,
                     m->rpart, m->g, m->lsum);
  HIP_TRYM(hipGetLastError());
  if (loss) {
    HIP_TRYM(hipMemcpyAsync(loss, m->lsum, 4, hipMemcpyDeviceToHost, s));
    HIP_TRYM(hipStreamSynchronize(s));
  }
  return POYG_OK;
}

// One Adam step on the gradient the last poyg_mlp_grad left.
int poyg_mlp_adam(poyg_mlp *m, float lr, float beta1, float beta2, float eps) {
  if (!m) return POYG_EINVAL;
  m->step += 1;
  const float c1 = 1.f - powf(beta1, (float)m->step), c2 = 1.f - powf(beta2, (float)m->step);
  hipLaunchKernelGGL(adam_kernel, dim3(256), dim3(256), 0, m->stream, MlpLayout::N, m->p, m->g, m->m1, m->m2, lr,
                     beta1, beta2, eps, c1, c2, m->w1t, m->w2t, m->w2b, m->w3b);
  HIP_TRYM(hipGetLastError());
  return POYG_OK;
}

// 4-mer profiles (float counts, 256 per sequence) of n device sequences.
int poyg_kmer_counts(poyg_ctx *ctx, const uint8_t *d_seq, const int64_t *d_off, const int32_t *d_len, int32_t n,
                     float *d_counts, void *stream) {
  if (!ctx || n < 0 || (n > 0 && (!d_seq || !d_off || !d_len || !d_counts))) return POYG_EINVAL;
  if (n == 0) return POYG_OK;
  hipStream_t s = stream ? (hipStream_t)stream : (hipStream_t)poyg_ctx_stream(ctx);
  hipLaunchKernelGGL(kmer_count_kernel, dim3(std::min(n, 65536)), dim3(256), 0, s, d_seq, d_off, d_len, n,
                     d_counts);
  HIP_TRYM(hipGetLastError());
  return POYG_OK;
}

// Pair features x[p] = bf16(|counts[ia[p]] - counts[ib[p]]| * scale).
int poyg_pair_features(poyg_ctx *ctx, const float *d_counts, const int32_t *d_ia, const int32_t *d_ib, int64_t n,
                       float scale, uint16_t *d_x, void *stream) {
  if (!ctx || n < 0 || (n > 0 && (!d_counts || !d_ia || !d_ib || !d_x))) return POYG_EINVAL;
  if (n == 0) return POYG_OK;
  hipStream_t s = stream ? (hipStream_t)stream : (hipStream_t)poyg_ctx_stream(ctx);
  if ((((uintptr_t)d_counts | (uintptr_t)d_x) & 15) == 0)
    hipLaunchKernelGGL(pair_feature_kernel, dim3((unsigned)std::min<int64_t>((n + 7) / 8, 1 << 14)), dim3(256), 0, s,
                       d_counts, d_ia, d_ib, n, scale, d_x);
  else
    hipLaunchKernelGGL(pair_feature_any_kernel, dim3((unsigned)std::min<int64_t>(n, 1 << 20)), dim3(256), 0, s,
                       d_counts, d_ia, d_ib, n, scale, d_x);
  HIP_TRYM(hipGetLastError());
  return POYG_OK;
}

// dst[r] = src[idx[r]] for rows of row_bytes (a multiple of 4) bytes.
int poyg_gather_rows(poyg_ctx *ctx, const void *d_src, int64_t row_bytes, const int32_t *d_idx, int64_t n,
                     void *d_dst, void *stream) {
  if (!ctx || n < 0 || row_bytes <= 0 || (row_bytes & 3) || (n > 0 && (!d_src || !d_idx || !d_dst))) {
    set_error("poyg_gather_rows: bad arguments");
    return POYG_EINVAL;
  }
  if (n == 0) return POYG_OK;
  hipStream_t s = stream ? (hipStream_t)stream : (hipStream_t)poyg_ctx_stream(ctx);
  hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)std::min<int64_t>(n, 1 << 20)), dim3(256), 0, s,
                     (const uint32_t *)d_src, (int)(row_bytes / 4), d_idx, n, (uint32_t *)d_dst);
  HIP_TRYM(hipGetLastError());
  return POYG_OK;
}

// A plain bf16 product for tests of the MFMA operand layout: C (f32, ldc) = A B
// with the strides above.
int poyg_gemm_bf16_f32(poyg_ctx *ctx, int M, int N, int K, const uint16_t *d_a, int64_t a_rs, int64_t a_cs,
                       const uint16_t *d_b, int64_t b_rs, int64_t b_cs, float *d_c, int64_t ldc, void *stream) {
  if (!ctx || M < 0 || N < 0 || K < 0) return POYG_EINVAL;
  hipStream_t s = stream ? (hipStream_t)stream : (hipStream_t)poyg_ctx_stream(ctx);
  if (M == 0 || N == 0) return POYG_OK;
  hipLaunchKernelGGL(gemm_bf16_kernel, dim3((M + kTM - 1) / kTM, (N + kTN - 1) / kTN), dim3(256), 0, s, M, N, K, d_a,
                     a_rs, a_cs, d_b, b_rs, b_cs, d_c, ldc);
  HIP_TRYM(hipGetLastError());
  return POYG_OK;
}

}  // extern "C"
