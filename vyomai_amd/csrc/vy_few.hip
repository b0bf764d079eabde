// Decode steps of 1 to 4 sequences: matrix-vector products that make their operand rows themselves.
//
// Such a step is a chain of launches that each move a few MB and take 2 to 4 us, of which the norm between two products is one: a
// single workgroup that waits for the product before it, reduces a row and writes it for the next.  Here every workgroup of the next
// product redoes that norm -- a row is 1.5 to 8 KB out of L2, a wave per row, reductions in registers -- while its weights, which it
// has requested first, are on their way; so the norm costs a launch's tail instead of a launch.  A wave takes R = 1 or 2 weight rows
// (rotary pairs and gate / up pairs are the two rows of a wave) in whole 1 KB pieces.
//
// 12 layers of 768, one sequence behind 70 tokens: 334 -> 249 us a step (62 launches instead of 75, and no products for 32 rows; with the
// output projection inside the attention, PARTS, 50 launches and 215 us);
// 8 layers of width 1024 (latent and lightning attention), 700 tokens: 302 -> 267 us, 2 / 4 rows 414 -> 308 / 482 -> 398 us.
#include "vy_few.h"

namespace vy_few {
namespace {

__device__ __forceinline__ float dot8(const bf16x8 a, const bf16x8 b, float s) {
#pragma unroll
  for (int i = 0; i < 8; i += 2) s = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{a[i], a[i + 1]}, bf16x2{b[i], b[i + 1]}, s, false);
  return s;
}
__device__ __forceinline__ float rsqrt_refined(float ms) {
  const float r = rsqrtf(ms);
  return r * (1.5f - 0.5f * ms * r * r);
}

// (v - mean) rstd of a row of which a lane holds the quads 64 c + lane, over its first n columns (v = 0 in the padding of a LayerNorm
// is not assumed)
template <int KC>
__device__ __forceinline__ void stats(const float (&v)[KC][4], int lane, int n, bool rms, float eps, float& mean, float& rstd) {
  mean = 0.f;
  if (!rms) {
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) s += v[c][e];
    mean = vy_wave_sum(s) / (float)n;
  }
  float q = 0.f;
#pragma unroll
  for (int c = 0; c < KC; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = (64 * c + lane) * 4 + e < n ? v[c][e] - mean : 0.f;
      q += d * d;
    }
  rstd = rsqrt_refined(vy_wave_sum(q) / (float)n + eps);
}

template <int EPI, int PRO, int MR, int KC, int NW>
__global__ __launch_bounds__(64 * NW) void few_kernel(Args a) {
  constexpr int K = 256 * KC, R = (EPI != STORE || KC % 2) ? 2 : 1, P = KC * R / 2;   // columns; weight rows and pieces per wave
  __shared__ __attribute__((aligned(16))) bf16 hs[PRO == PLAIN ? 8 : MR * K];
  constexpr int SHARES = PRO == PARTS ? 4 / MR : 1;   // waves that add up a row, of the first four
  __shared__ __attribute__((aligned(16))) float sums[SHARES > 1 ? 4 * K : 4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int units = EPI == STORE ? (a.N + R - 1) / R : EPI == QKV ? a.N / 2 : a.N;   // of R weight rows
  const int step = (PRO == RMS && a.cache ? gridDim.x - 1 : gridDim.x) * NW;
  int u = blockIdx.x * NW + wave;

  if constexpr (PRO == RMS) {
    if (a.cache && blockIdx.x == gridDim.x - 1) {   // one workgroup more: the new tokens' cache rows, a wave each
      if (wave >= a.M) return;
      constexpr int CH = 2;
      const bf16* src = a.kv + wave * a.ldx;
      float v[CH][8], q = 0.f;
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if ((lane + 64 * c) * 8 < a.np_kv) {
          VyChunk<bf16>::load(src + (lane + 64 * c) * 8, v[c]);
#pragma unroll
          for (int e = 0; e < 8; ++e) q += v[c][e] * v[c][e];
        }
      const int slot = a.slots ? a.slots[wave] : wave, pos = a.start[slot];
      const float rstd = rsqrt_refined(vy_wave_sum(q) / (float)a.n_kv + a.eps);
      if (!a.ring && pos >= a.cap) return;
      bf16* dst = a.cache + slot * a.k_ss + (a.ring ? pos % a.cap : pos) * a.k_st;
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if ((lane + 64 * c) * 8 < a.np_kv) {
          float o[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = v[c][e] * rstd * a.w_kv[(lane + 64 * c) * 8 + e];
          VyChunk<bf16>::store(dst + (lane + 64 * c) * 8, o);
        }
      return;
    }
  }

  auto row_of = [&](int unit, int r) {
    if constexpr (EPI == QKV) return (unit >> 5) * 64 + (unit & 31) + 32 * r;
    else if constexpr (EPI == GATED) return unit + r * a.N;
    else { const int n = unit * R + r; return n < a.N ? n : a.N - 1; }
  };
  // chunk (8 columns) of piece p: which of the wave's rows, and which columns
  bf16x8 w[P];
  auto request = [&](int unit) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int c = 64 * p + lane, r = R == 1 ? 0 : (c >= 32 * KC);
      const bf16x8* at = reinterpret_cast<const bf16x8*>(a.w + (int64_t)row_of(unit, r) * K + (c - r * 32 * KC) * 8);
      if (a.once) w[p] = __builtin_nontemporal_load(at);
      else w[p] = *at;
    }
  };
  // what the epilogue reads besides the product, one lane per (weight row, operand row), and none of it hangs on the product.  QKV requests
  // it behind the norm's operands: behind the norm, the position and then the rotary factors were two more trips to memory (768 columns
  // 3.86 -> 3.68 us).  The others have a bias and a residual at most, which are there before the product is if requested with it; ahead of
  // it they delay weights and operands: text models of 12 layers, steps of 1 / 4 sequences 171.5 -> 168.5 / 207.7 -> 203 us at 512 columns,
  // 194.5 -> 191.5 / 250 -> 244.5 at 768, 250 -> 247 / 302 -> 297 at 1024
  const int er = R == 1 || lane >= R * MR ? 0 : lane / MR, em = R == 1 ? lane : lane % MR;
  float e_bias = 0.f, e_other = 0.f, e_res = 0.f, e_cos = 0.f, e_sin = 0.f;
  int pos = 0;
  auto request_rest = [&](int unit) {
    if (lane >= R * MR || em >= a.M) return;
    const int n = row_of(unit, er);
    if (EPI != GATED && a.bias) e_bias = (float)a.bias[n];
    if (EPI == STORE && a.residual) e_res = (float)a.residual[em * a.ldr + n];
    if (EPI == QKV && a.bias) e_other = (float)a.bias[n ^ 32];   // (of the pair's other column)
    if (EPI == QKV && a.cos_tab) {
      e_cos = a.cos_tab[(int64_t)pos * 32 + (n & 31)];
      e_sin = a.sin_tab[(int64_t)pos * 32 + (n & 31)];
    }
  };
  if constexpr (EPI == QKV) pos = a.pos_dev ? *a.pos_dev : a.pos;
  if (u < units) request(u);
  // PLAIN: the operand rows as well, all together and ahead of the branches below -- left to the place of their use they come one trip to
  // L2 after the other (768 columns, 4 rows of K = 3072 / 4096 with everything in L2 4.6 / 5.5 us, together 3.1 / 3.4; 12 layers of 768, 4
  // sequences behind 790 tokens, the output projection by itself: 394 -> 347 us a step)
  bf16x8 xs[PRO == PLAIN ? P : 1][PRO == PLAIN ? MR : 1];
  if constexpr (PRO == PLAIN) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int c = 64 * p + lane, col = (c - (R == 2 && c >= 32 * KC ? 32 * KC : 0)) * 8;
#pragma unroll
      for (int m = 0; m < MR; ++m) xs[p][m] = *reinterpret_cast<const bf16x8*>(a.x + min(m, a.M - 1) * a.ldx + col);
    }
  }
  const int row = wave / SHARES;   // of the operand, this wave's
  const bool leads = wave % SHARES == 0 && row < a.M;
  if (EPI == QKV && u < units && (PRO == PLAIN || !leads)) request_rest(u);

  if constexpr (PRO != PLAIN) {
    if (a.advance && blockIdx.x == 0)
      for (int i = threadIdx.x; i < a.n_adv; i += 64 * NW) a.advance[a.slots ? a.slots[i] : i] += 1;
    bf16x4 v4[KC], g4[KC], b4[KC], xb4[KC];
    if constexpr (PRO == LAYER || PRO == PARTS) {
      if (leads) {
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const int col = (64 * c + lane) * 4;
          v4[c] = *reinterpret_cast<const bf16x4*>(a.x + row * a.ldx + col);
          g4[c] = *reinterpret_cast<const bf16x4*>(a.ln_g + col);
          b4[c] = *reinterpret_cast<const bf16x4*>(a.ln_b + col);
          xb4[c] = bf16x4{(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
          if (PRO == PARTS && a.x_bias) xb4[c] = *reinterpret_cast<const bf16x4*>(a.x_bias + col);
        }
        if (EPI == QKV && u < units) request_rest(u);
      }
    }
    f32x4 mine[KC];   // PARTS: this wave's share of the row
    if constexpr (PRO == PARTS) {
      constexpr int AHEAD = MR == 4 ? 6 : 4;   // parts requested together: all that a wave has, of 12 heads' two times
#pragma unroll
      for (int c = 0; c < KC; ++c) mine[c] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (row < a.M)
        for (int p0 = wave % SHARES; p0 < a.n_parts; p0 += AHEAD * SHARES) {
          f32x4 part[AHEAD][KC];
#pragma unroll
          for (int i = 0; i < AHEAD; ++i)
#pragma unroll
            for (int c = 0; c < KC; ++c)
              part[i][c] = *reinterpret_cast<const f32x4*>(a.parts + ((int64_t)min(p0 + i * SHARES, a.n_parts - 1) * a.M + row) * K + (64 * c + lane) * 4);
#pragma unroll
          for (int i = 0; i < AHEAD; ++i)
            if (p0 + i * SHARES < a.n_parts)
#pragma unroll
              for (int c = 0; c < KC; ++c) mine[c] += part[i][c];
        }
      if constexpr (SHARES > 1) {
        if (!leads && wave < 4)
#pragma unroll
          for (int c = 0; c < KC; ++c) *reinterpret_cast<f32x4*>(sums + wave * K + (64 * c + lane) * 4) = mine[c];
      }
    }
    if constexpr (SHARES > 1) __syncthreads();
    if constexpr (PRO == RMS) {
      if (leads) {
        // (a lane's quads two by two: the 16-byte chunks, and so the sum's order, of the norm's own kernel)
        auto column = [&](int c) { return ((c >> 1) * 64 + lane) * 8 + (c & 1) * 4; };
        f32x4 w4[KC];
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          v4[c] = *reinterpret_cast<const bf16x4*>(a.x + row * a.ldx + column(c));
          w4[c] = *reinterpret_cast<const f32x4*>(a.w_pre + column(c));
        }
        float q = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) q += (float)v4[c][e] * (float)v4[c][e];
        const float rstd = rsqrt_refined(vy_wave_sum(q) / (float)a.n + a.eps);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (bf16)((float)v4[c][e] * rstd * w4[c][e]);
          *reinterpret_cast<bf16x4*>(hs + row * K + column(c)) = o;
        }
      }
    } else if (leads) {
      const int m = row;
      float v[KC][4], g[KC][4], b[KC][4];
      if constexpr (PRO == LAYER || PRO == PARTS) {
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) { v[c][e] = (float)v4[c][e]; g[c][e] = (float)g4[c][e]; b[c][e] = (float)b4[c][e]; }
        if constexpr (PRO == PARTS) {
#pragma unroll
          for (int c = 0; c < KC; ++c) {
#pragma unroll
            for (int s = 1; s < SHARES; ++s) mine[c] += *reinterpret_cast<const f32x4*>(sums + (wave + s) * K + (64 * c + lane) * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] = vy_round_bf16(mine[c][e] + (float)xb4[c][e] + v[c][e]);
          }
        }
      } else {
        f32x4 s4[KC], p4[KC], g4[KC];
        bf16x4 y4[KC];
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const int col = (64 * c + lane) * 4;
          s4[c] = *reinterpret_cast<const f32x4*>(a.s_in + m * a.lds + col);
          if (a.x) y4[c] = *reinterpret_cast<const bf16x4*>(a.x + m * a.ldx + col);
          if (a.w_post) p4[c] = *reinterpret_cast<const f32x4*>(a.w_post + col);
          if (a.w_pre) g4[c] = *reinterpret_cast<const f32x4*>(a.w_pre + col);
        }
        if (a.x) {
          float mean = 0.f, rstd = 1.f, y[KC][4];
#pragma unroll
          for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) y[c][e] = (float)y4[c][e];
          if (a.w_post) stats<KC>(y, lane, a.n, a.rms, a.eps, mean, rstd);
#pragma unroll
          for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] = s4[c][e] + (a.w_post ? (y[c][e] - mean) * rstd * p4[c][e] : y[c][e]);
        } else {
#pragma unroll
          for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] = s4[c][e];
        }
        if (a.s_out && blockIdx.x == 0)
#pragma unroll
          for (int c = 0; c < KC; ++c) *reinterpret_cast<f32x4*>(a.s_out + m * a.lds + (64 * c + lane) * 4) = f32x4{v[c][0], v[c][1], v[c][2], v[c][3]};
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) { g[c][e] = a.w_pre ? g4[c][e] : 1.f; b[c][e] = 0.f; }
      }
      float mean = 0.f, rstd = 1.f;
      if (PRO != STREAM || a.w_pre) stats<KC>(v, lane, PRO != STREAM ? K : a.n, PRO == STREAM && a.rms, a.eps, mean, rstd);
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const int col = (64 * c + lane) * 4;
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (bf16)((v[c][e] - mean) * rstd * g[c][e] + b[c][e]);
        *reinterpret_cast<bf16x4*>(hs + m * K + col) = o;
        if (a.h && blockIdx.x == 0) *reinterpret_cast<bf16x4*>(a.h + m * a.ldh + col) = o;
      }
    }
    __syncthreads();
  }

  for (; u < units; u += step) {
    if constexpr (EPI != QKV) request_rest(u);
    const bool mine = lane < R * MR && em < a.M;
    const int n = row_of(u, er);
    const bool real = mine && (EPI != STORE || u * R + er < a.N);
    const float bias = e_bias, other_bias = e_other, res = e_res, cs = e_cos, sn = e_sin;
    float acc[R][MR];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < MR; ++m) acc[r][m] = 0.f;
    bf16x8 wv[P];
#pragma unroll
    for (int p = 0; p < P; ++p) wv[p] = w[p];
    if (u + step < units) {
      request(u + step);
      if constexpr (EPI == QKV) request_rest(u + step);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int c = 64 * p + lane;
      const bool second = R == 2 && c >= 32 * KC;
      const int col = (c - (second ? 32 * KC : 0)) * 8;
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        bf16x8 xv;
        if constexpr (PRO == PLAIN) xv = xs[p][m];
        else xv = *reinterpret_cast<const bf16x8*>(hs + m * K + col);
        if (R == 1 || 64 * (p + 1) <= 32 * KC) acc[0][m] = dot8(wv[p], xv, acc[0][m]);
        else if (64 * p >= 32 * KC) acc[R - 1][m] = dot8(wv[p], xv, acc[R - 1][m]);
        else {   // the piece that holds the end of one row and the start of the other
          const float d = dot8(wv[p], xv, 0.f);
          acc[0][m] += second ? 0.f : d;
          acc[R - 1][m] += second ? d : 0.f;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < MR; ++m) acc[r][m] = vy_wave_sum(acc[r][m]);
    float own = 0.f, other = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < MR; ++m)
        if (er == r && em == m) { own = acc[r][m]; other = acc[R - 1 - r][m]; }
    if constexpr (EPI == STORE) {
      float v = own + bias;
      if (a.act == VY_ACT_GELU_ERF) v = vy_act_fwd_fast<VY_ACT_GELU_ERF>(v);
      else if (a.act == VY_ACT_GELU_TANH) v = vy_act_fwd_fast<VY_ACT_GELU_TANH>(v);
      else if (a.act == VY_ACT_RELU2) v = vy_act_fwd<VY_ACT_RELU2>(v);
      else if (a.act == VY_ACT_SOFTCAP) v = vy_act_fwd<VY_ACT_SOFTCAP>(v, a.act_arg);
      if (real) a.y[em * a.ldy + n] = (bf16)(v + res);
    } else if constexpr (EPI == GATED) {
      const float g = vy_round_bf16(own), up = vy_round_bf16(other);   // (lanes of row 0: own is the gate's)
      if (real && er == 0) a.y[em * a.ldy + u] = (bf16)((a.act == VY_ACT_SILU ? vy_silu(g) : vy_gelu_tanh(g)) * up);
    } else {
      float v = own + bias;
      if (a.cos_tab && n < a.nq + a.nkv) {
        const float c = vy_round_bf16(cs), s = vy_round_bf16(sn);
        const float t = vy_round_bf16(vy_round_bf16(other + other_bias) * s), m0 = vy_round_bf16(vy_round_bf16(v) * c);
        v = er ? m0 + t : m0 - t;
      }
      if (real) {
        const int hd = n >> 6, d = n & 63, hq = a.nq >> 6, hkv = a.nkv >> 6;
        bf16* dst;
        if (hd < hq) dst = a.q + (int64_t)em * a.nq + n;
        else if (hd < hq + hkv) dst = a.k + em * a.c_sb + (hd - hq) * a.c_sh + (int64_t)pos * a.c_sl + d;
        else dst = a.v + em * a.c_sb + (hd - hq - hkv) * a.c_sh + (int64_t)pos * a.c_sl + d;
        *dst = (bf16)v;
      }
    }
  }
}

template <int EPI, int PRO, int KC, int NW>
void go_waves(const Args& a, int units, hipStream_t st) {
  // every workgroup redoes the operand rows, so there are no more of them than fit on the chip at once (by registers): the waves of
  // wide products loop, with the next rows' weights requested ahead
  const int most = (PRO != STREAM ? 2048 : KC <= 4 ? 1024 : 512) * 4 / NW, wgs = (units + NW - 1) / NW;
  const int grid = (wgs < most ? wgs : most) + (PRO == RMS && a.cache ? 1 : 0);
  if (a.M == 1) hipLaunchKernelGGL((few_kernel<EPI, PRO, 1, KC, NW>), dim3(grid), dim3(64 * NW), 0, st, a);
  else if (a.M == 2) hipLaunchKernelGGL((few_kernel<EPI, PRO, 2, KC, NW>), dim3(grid), dim3(64 * NW), 0, st, a);
  else hipLaunchKernelGGL((few_kernel<EPI, PRO, 4, KC, NW>), dim3(grid), dim3(64 * NW), 0, st, a);
}
template <int EPI, int PRO, int KC>
void go_rows(const Args& a, hipStream_t st) {
  constexpr int R = (EPI != STORE || KC % 2) ? 2 : 1;
  const int units = EPI == STORE ? (a.N + R - 1) / R : EPI == QKV ? a.N / 2 : a.N;
  // Operand rows that are made are made once a workgroup, so it has as many waves as leave no CU without one: what a CU takes in for them
  // (the shares, or the stream, the sublayer and two weight rows, out of L2 behind the weights) falls with the workgroups on it.  Up to
  // 1024 waves in all, which are a workgroup of four per CU at most: 4 (1152 columns of QKV, K = 768, 3.39 us, in workgroups of eight 3.46).
  // One / four rows on four, eight and sixteen waves: PARTS, 3072 x 768, 5.0, 4.6, 4.9 / 7.9, 6.4, 6.9, 4096 x 1024 7.3, 6.0, 5.4 / 17.2,
  // 13.3, 9.7; STREAM, 1792 x 1024, 4.1, 3.9, 4.0 / 5.3, 4.6, 4.9, 4096 x 1024 5.1, 4.9, 4.7 / 7.5, 6.3, 5.7; gated, 4096 x 1024, 6.4, 6.3,
  // 6.2 / 9.0, 8.0, 7.5.  Sixteen waves of K = 2048 do not fit the registers (3584 rows 6.8, 6.5, 9.2).
  if constexpr (KC <= 4 && (PRO == STREAM || PRO == PARTS)) {
    if (units > 3072) return go_waves<EPI, PRO, KC, 16>(a, units, st);
  }
  if constexpr (PRO != PLAIN) {
    if (units > 1024) return go_waves<EPI, PRO, KC, 8>(a, units, st);
  }
  go_waves<EPI, PRO, KC, 4>(a, units, st);
}

}  // namespace

bool few_k(int epi, int pro, int64_t K) {
  if (K % 256) return false;
  const int kc = (int)(K / 256);
  if (pro == PLAIN) return epi == QKV ? kc >= 2 && kc <= 4 : epi == STORE && (kc == 2 || kc == 3 || kc == 4 || kc == 8 || kc == 12 || kc == 16);
  if (pro == LAYER) return epi != GATED && kc >= 2 && kc <= 4;
  if (pro == RMS) return epi == STORE && (kc == 2 || kc == 4);   // (an even kc: a lane's quads pair up to 16-byte chunks; the query latents of bench.py's models)
  if (pro == PARTS) return epi == STORE && kc >= 2 && kc <= 4;
  return epi != QKV && (kc == 4 || kc == 8);
}

int few_go(int epi, int pro, const Args& a, int64_t K, hipStream_t st) {
  if (!few_k(epi, pro, K) || a.M < 1 || a.M > 4 || a.N < 1) return VY_ERR_UNSUPPORTED;
  const int kc = (int)(K / 256);
#define FEW(E, P, KC_) case KC_: go_rows<E, P, KC_>(a, st); break
  if (pro == PLAIN && epi == QKV) switch (kc) { FEW(QKV, PLAIN, 2); FEW(QKV, PLAIN, 3); FEW(QKV, PLAIN, 4); }
  else if (pro == PLAIN) switch (kc) { FEW(STORE, PLAIN, 2); FEW(STORE, PLAIN, 3); FEW(STORE, PLAIN, 4); FEW(STORE, PLAIN, 8); FEW(STORE, PLAIN, 12); FEW(STORE, PLAIN, 16); }
  else if (pro == LAYER && epi == QKV) switch (kc) { FEW(QKV, LAYER, 2); FEW(QKV, LAYER, 3); FEW(QKV, LAYER, 4); }
  else if (pro == RMS) switch (kc) { FEW(STORE, RMS, 2); FEW(STORE, RMS, 4); }
  else if (pro == PARTS) switch (kc) { FEW(STORE, PARTS, 2); FEW(STORE, PARTS, 3); FEW(STORE, PARTS, 4); }
  else if (pro == LAYER) switch (kc) { FEW(STORE, LAYER, 2); FEW(STORE, LAYER, 3); FEW(STORE, LAYER, 4); }
  else if (epi == STORE) switch (kc) { FEW(STORE, STREAM, 4); FEW(STORE, STREAM, 8); }
  else switch (kc) { FEW(GATED, STREAM, 4); FEW(GATED, STREAM, 8); }
#undef FEW
  VY_CHECK_LAUNCH("few_kernel");
  return VY_OK;
}

}  // namespace vy_few

// test aid, not part of include/vyom_hip.h: one product by itself on contiguous rows.  a, b: gamma and beta of LAYER and PARTS (bf16), w_post and
// w_pre of STREAM (fp32); PARTS: n shares s_in [n][M][K] and their bias `residual`; RMS: weights sin_tab; y: QKV's queries [M][nq], k and v [M][nkv]
extern "C" int vy_debug_few(int epi, int pro, const void* x, const void* a, const void* b, const float* s_in, float* s_out, void* h, int n,
                            int rms, float eps, const void* w, const void* bias, int act, float act_arg, const void* residual, void* y,
                            int64_t ldy, void* k, void* v, int nq, int nkv, const float* cos_tab, const float* sin_tab, int pos, int M,
                            int N, int64_t K, void* stream) {
  vy_few::Args f{};
  f.x = (const bf16*)x; f.ldx = K;
  if (pro == vy_few::PARTS) {
    f.parts = s_in; f.n_parts = n; f.x_bias = (const bf16*)residual;
    residual = nullptr;
  }
  if (pro == vy_few::RMS) {
    if (k) {   // rows v [M][K] of nkv columns, weights b, into row cos_tab[slot] (integers; below nq, of a ring of -nq) of k [slot][2][nkv]; slots h
      f.kv = (const bf16*)v; f.w_kv = (const float*)b; f.n_kv = f.np_kv = nkv; f.cache = (bf16*)k; f.k_ss = 2 * (int64_t)nkv; f.k_st = nkv;
      f.cap = nq < 0 ? -nq : nq; f.ring = nq < 0; f.start = (const int*)cos_tab; f.slots = (const int*)h;
    }
    b = sin_tab; h = nullptr;
  }
  if (pro == vy_few::LAYER || pro == vy_few::PARTS) { f.ln_g = (const bf16*)a; f.ln_b = (const bf16*)b; }
  else { f.w_post = (const float*)a; f.w_pre = (const float*)b; }
  f.s_in = s_in; f.s_out = s_out; f.lds = K; f.n = n; f.rms = rms; f.eps = eps; f.h = (bf16*)h; f.ldh = K;
  f.w = (const bf16*)w; f.N = N; f.M = M; f.bias = (const bf16*)bias; f.act = act; f.act_arg = act_arg;
  f.residual = (const bf16*)residual; f.ldr = N; f.y = (bf16*)y; f.ldy = ldy;
  if (epi == vy_few::QKV) {   // (one cache row a sequence: `pos` turns, the rows lie at 0)
    f.q = (bf16*)y; f.k = (bf16*)k - (int64_t)pos * nkv; f.v = (bf16*)v - (int64_t)pos * nkv; f.c_sb = nkv; f.c_sh = 64; f.c_sl = nkv;
    f.cos_tab = cos_tab; f.sin_tab = sin_tab; f.pos = pos; f.nq = nq; f.nkv = nkv;
  }
  return vy_few::few_go(epi, pro, f, K, (hipStream_t)stream);
}
