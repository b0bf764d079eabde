// Weight-streaming products of few rows (decode): a workgroup of NW = 4 (or 8) waves takes 16 NT rows of W [N][K] against 16 MB rows of X
// on mfma_f32_16x16x32_bf16 (A = weight rows, B = rows of X).  The waves split K by whole 128-byte lines (two k-steps of 32).  Two ways for
// the operands: through LDS, line by line (share_lds), or straight from memory into operand registers (share) -- every wave requests
// its loads of up to STEPS k-steps before the first product, W past the caches (non-temporal).  A
// load into registers is 16 rows with 16 bytes a lane, no two neighbouring lanes on a line, and a CU takes in 25 to 30 KB of them a
// microsecond; of whole lines, 8 lanes each, 60.
#pragma once
#include "vy_common.h"

namespace vy_rows {

template <int NT, int MB> constexpr int RED = 3 * NT * MB * 64;   // f32x4 of LDS that stream() needs
template <int NT, int MB, int NW = 4> constexpr int DENSE_RED = NW * NT * MB * 64;   // and dense()
constexpr int vy_max2(int a, int b) { return a > b ? a : b; }
template <int NT, int MB> constexpr int STEPS = NT * MB == 1 ? 16 : NT + MB <= 3 ? 8 : 4;

// acc[t][j] = 16 rows ws[t] x 16 rows xs[j] over the wave's share of K; a lane's pointers are its row (lane & 15) + 8 (lane >> 4).
// D: a lane owns row lane & 15 of X and rows 4 (lane >> 4) .. + 3 of W.  Each load has a condition of its own: all of a step's behind one
// branch came one step after the other (experts of 16 sequences 338 us, 32 433, instead of 321 and 411).
template <int NT, int MB>
__device__ __forceinline__ void share(const bf16* const (&ws)[NT], const bf16* const (&xs)[MB], int K, f32x4 (&acc)[NT][MB]) {
  constexpr int U = STEPS<NT, MB>, NW = 4;
  const int kq = (threadIdx.x & 63) >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bf16x8 zero8 = {(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 64 * wave; k0 < K; k0 += 32 * NW * U) {
    bf16x8 w[U][NT], x[U][MB];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 64 * NW * (u >> 1) + 32 * (u & 1);
      const bool in = k + 8 * kq < K;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16x8* at = reinterpret_cast<const bf16x8*>(ws[t] + k);
        w[u][t] = in ? __builtin_nontemporal_load(at) : zero8;
      }
#pragma unroll
      for (int j = 0; j < MB; ++j) x[u][j] = in ? *reinterpret_cast<const bf16x8*>(xs[j] + k) : zero8;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][t], x[u][j], acc[t][j], 0, 0, 0);
  }
}

// share() with the operands' way through LDS: a wave's share of K is whole 128-byte lines, and it brings each line of its rows -- 8 rows a
// load, 8 lanes side by side on a row's line -- into a ring of its own, D lines deep, and multiplies out of it.  No other wave is waited
// for, and the products and their order are share()'s.  first, rows, count: rows of W from `first`, R of them, below count.
template <int MB, int R> constexpr int LINE = (2 * MB + R / 8) * 1024;   // bytes of a line of all rows
template <int NT, int MB, int NW, int D, int R>
__device__ __forceinline__ void share_lds(const bf16* x, int64_t ldx, int M, const bf16* w, int64_t ldw, int first, int count, int K, char* ring,
                                          f32x4 (&acc)[NT][MB]) {
  constexpr int PX = 2 * MB, PW = R / 8, P = PX + PW;
  static_assert(R % 8 == 0 && R > 16 * (NT - 1) && P * (D - 1) < 64, "vmcnt counts to 63");
  const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bf16* at[P];
  int col[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int row = 8 * (p < PX ? p : p - PX) + (lane >> 3);
    col[p] = 8 * ((lane & 7) ^ ((row >> 1) & 7));
    at[p] = (p < PX ? x + min(row, M - 1) * ldx : w + min(first + row, count - 1) * ldw) + col[p];
  }
  const bf16* zero = reinterpret_cast<const bf16*>(vy_zero16);
  const int lines = K > 64 * wave ? (K - 64 * wave + 64 * NW - 1) / (64 * NW) : 0;
  char* mine = ring + wave * D * P * 1024;
  auto request = [&](int i, int slot) {
    const int k = 64 * wave + 64 * NW * i;
#pragma unroll
    for (int p = 0; p < P; ++p)
      __builtin_amdgcn_global_load_lds((const VY_GLOBAL void*)(k + col[p] < K ? at[p] + k : zero), (VY_LDS void*)(mine + (slot * P + p) * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < D; ++i)
    if (i < lines) request(i, i);
  unsigned xa[2][MB], wa[2][NT];   // of the two k-steps of a line in slot 0
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
    for (int j = 0; j < MB; ++j) xa[ks][j] = vy_lds_addr(mine) + (16 * j + r16) * 128 + (((4 * ks + kq) ^ ((r16 >> 1) & 7)) << 4);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int r = 16 * t + (16 * t + 16 > R ? r16 & 7 : r16);
      wa[ks][t] = vy_lds_addr(mine) + PX * 1024 + r * 128 + (((4 * ks + kq) ^ ((r >> 1) & 7)) << 4);
    }
  }
  int slot = 0;
  for (int i = 0; i < lines; ++i) {
    // line i has landed: the younger ones, D - 1 of them or what is left, may be on their way
    const int younger = min(D - 1, lines - 1 - i);
    vy_static_for<D>([&](auto n_c) {
      constexpr int n = decltype(n_c)::value;
      if (younger == n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * n) : "memory");
    });
    const unsigned off = (unsigned)slot * P * 1024;
    bf16x8 xf[2][MB], wf[2][NT];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[ks][t] = vy_lds_read128_off<0>(wa[ks][t] + off);
#pragma unroll
      for (int j = 0; j < MB; ++j) xf[ks][j] = vy_lds_read128_off<0>(xa[ks][j] + off);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int t = 0; t < NT; ++t) vy_tie(wf[ks][t]);
#pragma unroll
      for (int j = 0; j < MB; ++j) vy_tie(xf[ks][j]);
    }
    if (i + D < lines) request(i + D, slot);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ks][t], xf[ks][j], acc[t][j], 0, 0, 0);
    slot = slot + 1 == D ? 0 : slot + 1;
  }
}

// share() and, in wave 0, the waves' sums
template <int NT, int MB>
__device__ __forceinline__ void stream(const bf16* const (&ws)[NT], const bf16* const (&xs)[MB], int K, f32x4 (&acc)[NT][MB],
                                       f32x4* red) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  share<NT, MB>(ws, xs, K, acc);
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
        for (int s = 0; s < 3; ++s) {
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
// red: LDS of DENSE bytes, the ring of share_lds before what the waves add up.
template <int MB, int NW, int NT, bool HALF, int D> constexpr int DENSE = vy_max2(D * NW * LINE<MB, 16 * NT - (HALF ? 8 : 0)>, DENSE_RED<NT, MB, NW> * 16);
template <int MB, int NW = 4, int NT = 1, bool HALF = false, int ACT = VY_ACT_NONE, int D = 2>
__device__ __forceinline__ void dense(const Dense& a, char* lds, int tile, int K) {   // K: columns of x and w that count
  constexpr int R = 16 * NT - (HALF ? 8 : 0), BLOCKS = NT * MB, MINE = (BLOCKS + NW - 1) / NW;
  const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  f32x4* red = reinterpret_cast<f32x4*>(lds);
  // biases of the wave's blocks, a quad each: as they come, since what unpacks them here waits for them ahead of the stream
  uint2 bias[MINE];
  if (a.bias && (uintptr_t)a.bias % 8 == 0 && R * tile + 16 * NT <= a.N) {   // (uniform)
#pragma unroll
    for (int b = 0; b < MINE; ++b)
      if (wave + NW * b < BLOCKS) bias[b] = *reinterpret_cast<const uint2*>(a.bias + R * tile + 16 * ((wave + NW * b) / MB) + 4 * kq);
  } else if (a.bias) {
#pragma unroll
    for (int b = 0; b < MINE; ++b)
      if (wave + NW * b < BLOCKS) {
        unsigned v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = reinterpret_cast<const unsigned short*>(a.bias)[min(R * tile + 16 * ((wave + NW * b) / MB) + 4 * kq + r, a.N - 1)];
        bias[b] = make_uint2(v[0] | v[1] << 16, v[2] | v[3] << 16);
      }
  }
  f32x4 acc[NT][MB];
  share_lds<NT, MB, NW, D, R>(a.x, a.ldx, a.M, a.w, a.K, R * tile, a.N, K, lds, acc);
  __syncthreads();   // (red lies over the other waves' rings)
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
      if (a.bias) {
        const unsigned two = r < 2 ? bias[b].x : bias[b].y;
        z += __builtin_bit_cast(float, r & 1 ? two & 0xffff0000u : two << 16);
      }
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

template <int MB>
__device__ __forceinline__ void dense(const Dense& a, char* lds, int tile) { dense<MB>(a, lds, tile, a.K); }

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
