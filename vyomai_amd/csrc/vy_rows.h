// Weight-streaming products of few rows (decode): a workgroup of NW = 4 (or 8) waves takes 16 NT rows of W [N][K] against 16 MB rows of X
// on mfma_f32_16x16x32_bf16 (A = weight rows, B = rows of X), both straight from memory into operand registers: a weight is used
// once, and X is small enough for L2.  The waves split K by whole 128-byte lines (two k-steps of 32); every wave requests its
// loads of up to STEPS k-steps before the first product, so a pass over K = 32 NW STEPS costs one memory latency.  W is streamed
// past the caches (non-temporal) unless other workgroups read it too.
#pragma once
#include "vy_common.h"

namespace vy_rows {

template <int NT, int MB, int NW = 4> constexpr int RED = (NW - 1) * NT * MB * 64;   // f32x4 of LDS that stream() needs
template <int NT, int MB, int NW = 4> constexpr int DENSE_RED = NW * NT * MB * 64;   // and dense()
template <int NT, int MB> constexpr int STEPS = NT * MB == 1 ? 16 : NT + MB <= 3 ? 8 : 4;

// acc[t][j] = 16 rows ws[t] x 16 rows xs[j] over the wave's share of K; a lane's pointers are its row (lane & 15) + 8 (lane >> 4).
// D: a lane owns row lane & 15 of X and rows 4 (lane >> 4) .. + 3 of W.
// APART: whole passes over K in code of their own, whose loads have no conditions.  dense() gains by it (decoder of width 2048, steps of 5 / 32
// sequences 602 -> 572 us, 756 -> 690); the experts, whose kernels hold a dense product's code as well, lose (2 layers of width 2048 and 64
// experts, 16 / 32 sequences: 321 -> 329 us, 411 -> 416).  Behind whole passes each load has a condition of its own: all of a step's
// behind one branch came one step after the other (16 sequences 338 us, 32 433).
// HALF: the last eight lanes of the last weight rows have none; up to 16 rows of X they load nothing (5 x 5984, K = 7424, 29.4 -> 26.7 us, 8 x 12511,
// K = 7936, 74.5 -> 69.5), above that the other eight lanes' rows again (32 x 6144, K = 1024, 6.9 us, with conditions 7.2).
template <int NT, int MB, bool ONCE, int NW, int U = STEPS<NT, MB>, bool APART = true, bool HALF = false>
__device__ __forceinline__ void share(const bf16* const (&ws)[NT], const bf16* const (&xs)[MB], int K, f32x4 (&acc)[NT][MB]) {
  const int kq = (threadIdx.x & 63) >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool there = !HALF || MB > 1 || (threadIdx.x & 15) < 8;   // the last weight row, of this lane
  const bf16x8 zero8 = {(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 64 * wave; k0 < K; k0 += 32 * NW * U) {
    bf16x8 w[U][NT], x[U][MB];
    auto request = [&](int u, int k) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16x8* at = reinterpret_cast<const bf16x8*>(ws[t] + k);
        if constexpr (HALF && MB == 1) {
          if (t == NT - 1) { w[u][t] = there ? __builtin_nontemporal_load(at) : zero8; continue; }
        }
        if constexpr (ONCE) w[u][t] = __builtin_nontemporal_load(at);
        else w[u][t] = *at;
      }
#pragma unroll
      for (int j = 0; j < MB; ++j) x[u][j] = *reinterpret_cast<const bf16x8*>(xs[j] + k);
    };
    if (APART && k0 + 64 * NW * ((U - 1) >> 1) + 64 <= K) {
#pragma unroll
      for (int u = 0; u < U; ++u) request(u, k0 + 64 * NW * (u >> 1) + 32 * (u & 1));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + 64 * NW * (u >> 1) + 32 * (u & 1);
        const bool in = k + 8 * kq < K;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const bf16x8* at = reinterpret_cast<const bf16x8*>(ws[t] + k);
          const bool row = in && (t < NT - 1 || there);
          if constexpr (ONCE) w[u][t] = row ? __builtin_nontemporal_load(at) : zero8;
          else w[u][t] = row ? *at : zero8;
        }
#pragma unroll
        for (int j = 0; j < MB; ++j) x[u][j] = in ? *reinterpret_cast<const bf16x8*>(xs[j] + k) : zero8;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][t], x[u][j], acc[t][j], 0, 0, 0);
  }
}

// share() and, in wave 0, the waves' sums
template <int NT, int MB, bool ONCE = true, int NW = 4>
__device__ __forceinline__ void stream(const bf16* const (&ws)[NT], const bf16* const (&xs)[MB], int K, f32x4 (&acc)[NT][MB],
                                       f32x4* red) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  share<NT, MB, ONCE, NW, STEPS<NT, MB>, false>(ws, xs, K, acc);
  __syncthreads();   // (red may still be read from the pass before)
  if (wave)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < MB; ++j) red[((wave - 1) * NT * MB + t * MB + j) * 64 + lane] = acc[t][j];
  __syncthreads();
  if (wave == 0)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < MB; ++j)
#pragma unroll
        for (int s = 0; s < NW - 1; ++s) {
          const f32x4 v = red[(s * NT * MB + t * MB + j) * 64 + lane];
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][j][r] += v[r];
        }
}

struct Dense {
  const bf16* x; int64_t ldx; int M;   // M <= 16 MB
  const bf16* w; int N, K;             // [N][K]
  void* y; int64_t ldy; int f32;       // f32: fp32 results
  const bf16* bias; float act_arg;     // of bf16 results: act(x W^T + bias)
};

// rows R tile .. + R - 1 of W against all of X, R = 16 NT (HALF: - 8, the last eight lanes' rows twice).  What the waves add up goes through
// LDS, and each wave finishes blocks of its own, biases requested ahead of the stream: finished by the first wave alone, element by
// element with a wait for each bias and a switch over the activations, a workgroup ran through 3300 instructions behind its last
// product, 3 of 8.6 us (32 rows, 6144 x 1024).
template <int MB, int NW = 4, int NT = 1, bool HALF = false, int ACT = VY_ACT_NONE, int U = STEPS<NT, MB>>
__device__ __forceinline__ void dense(const Dense& a, f32x4* red, int tile, int K) {   // K: columns of x and w that count
  constexpr int R = 16 * NT - (HALF ? 8 : 0), BLOCKS = NT * MB, MINE = (BLOCKS + NW - 1) / NW;
  const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bf16* ws[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int r = HALF && t == NT - 1 ? r16 & 7 : r16;
    ws[t] = a.w + (int64_t)min(R * tile + 16 * t + r, a.N - 1) * a.K + 8 * kq;
  }
  const bf16* xs[MB];
#pragma unroll
  for (int j = 0; j < MB; ++j) xs[j] = a.x + (int64_t)min(16 * j + r16, a.M - 1) * a.ldx + 8 * kq;
  bf16 bias[MINE][4];   // (as they come: a conversion here waits for them ahead of the stream)
  if (a.bias) {   // (uniform)
#pragma unroll
    for (int b = 0; b < MINE; ++b)
      if (wave + NW * b < BLOCKS)
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[b][r] = a.bias[min(R * tile + 16 * ((wave + NW * b) / MB) + 4 * kq + r, a.N - 1)];
  }
  f32x4 acc[NT][MB];
  share<NT, MB, true, NW, U, true, HALF>(ws, xs, K, acc);
  __syncthreads();   // (red may still be read from the pass before)
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i) red[(wave * BLOCKS + i) * 64 + lane] = acc[i / MB][i % MB];
  __syncthreads();
#pragma unroll
  for (int b = 0; b < MINE; ++b) {
    const int i = wave + NW * b, m = 16 * (i % MB) + r16, n = R * tile + 16 * (i / MB) + 4 * kq;
    if (i >= BLOCKS || m >= a.M || n >= a.N || (HALF && i / MB == NT - 1 && kq >= 2)) continue;
    f32x4 v = red[i * 64 + lane];
#pragma unroll
    for (int s = 1; s < NW; ++s) {
      const f32x4 p = red[(s * BLOCKS + i) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] += p[r];
    }
    if (a.f32) {
      float* y = (float*)a.y + (int64_t)m * a.ldy + n;
      if (n + 4 <= a.N && (uintptr_t)y % 16 == 0) {
        *reinterpret_cast<f32x4*>(y) = v;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < a.N) y[r] = v[r];
      }
      continue;
    }
    bf16x4 w4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float z = v[r];
      if (a.bias) z += (float)bias[b][r];
      if constexpr (ACT != VY_ACT_NONE) z = vy_act_fwd<ACT>(z, a.act_arg);
      w4[r] = (bf16)z;
    }
    bf16* y = (bf16*)a.y + (int64_t)m * a.ldy + n;
    if (n + 4 <= a.N) {
      *reinterpret_cast<bf16x4*>(y) = w4;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < a.N) y[r] = w4[r];
    }
  }
}

template <int MB, int NW = 4, int NT = 1>
__device__ __forceinline__ void dense(const Dense& a, f32x4* red, int tile) { dense<MB, NW, NT>(a, red, tile, a.K); }

// ---- one row of X: a wave per two weight rows ---------------------------------------------------
// Whole 1 KiB pieces of a row per instruction and no sharing between waves: many small, even pieces of work, which a single
// token's stream needs to reach every CU equally (16-row tiles leave some with half as much again as others).
__device__ __forceinline__ float dot8(const bf16x8 a, const bf16x8 b, float s) {
#pragma unroll
  for (int i = 0; i < 8; i += 2) s = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{a[i], a[i + 1]}, bf16x2{b[i], b[i + 1]}, s, false);
  return s;
}
__device__ __forceinline__ void gemv2(const bf16* w0, const bf16* w1, const bf16* x, int K, float& s0, float& s1) {
  constexpr int U = 4;
  const int lane = threadIdx.x & 63;
  s0 = s1 = 0.f;
  int k = lane * 8;
  for (; k - lane * 8 + 512 * U <= K; k += 512 * U) {   // (wave-uniform)
    bf16x8 a[U], b[U], v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      a[u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(w0 + k + 512 * u));
      b[u] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(w1 + k + 512 * u));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const bf16x8*>(x + k + 512 * u);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s0 = dot8(a[u], v[u], s0);
      s1 = dot8(b[u], v[u], s1);
    }
  }
#pragma unroll 2
  for (; k < K; k += 512) {
    const bf16x8 a = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(w0 + k));
    const bf16x8 b = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(w1 + k));
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(x + k);
    s0 = dot8(a, v, s0);
    s1 = dot8(b, v, s1);
  }
  s0 = vy_wave_sum(s0);
  s1 = vy_wave_sum(s1);
}

// rows 8 tile .. + 7 of W against the one row of X
__device__ __forceinline__ void dense1(const Dense& a, int tile) {
  const int n = 8 * tile + 2 * (threadIdx.x >> 6);
  if (n >= a.N) return;
  const bf16* w = a.w + (int64_t)n * a.K;
  float s0, s1;
  gemv2(w, n + 1 < a.N ? w + a.K : w, a.x, a.K, s0, s1);
  if (threadIdx.x & 63) return;
  if (a.f32) {
    ((float*)a.y)[n] = s0;
    if (n + 1 < a.N) ((float*)a.y)[n + 1] = s1;
  } else {
    ((bf16*)a.y)[n] = (bf16)s0;
    if (n + 1 < a.N) ((bf16*)a.y)[n + 1] = (bf16)s1;
  }
}

}  // namespace vy_rows
