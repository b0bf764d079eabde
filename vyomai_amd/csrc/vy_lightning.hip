// Linear attention with a per-head decay:
//   S_t = decay S_(t-1) + k_t v_t^T ,  o_t = S_t^T q_t
// with q, k, v = silu of the projections (lightning attention), or q and k rotated by their position and k scaled (retention).
//
// Two forms of the same sums:
//   * decay_recurrent_kernel: token by token, the state in registers (fp32).  Decode steps, fp32 models, and head widths
//     the chunked form does not cover.
//   * chunked (bf16 prefill), C = VY_DECAY_CHUNK tokens at a time on MFMA, three launches:
//       chunk_kv_kernel    U_c = sum_j decay^(m-1-j) k_j v_j^T over the m tokens of chunk c         (all chunks at once)
//       chunk_scan_kernel  S_(c+1) = decay^m S_c + U_c, elementwise along the chunks; leaves S_c where U_c was
//       chunk_out_kernel   O = [lower(Q K^T) * decay^(i-j)] V + decay^(i+1) Q S_c                    (all chunks at once)
//
// 32-bit throughout where it enters the recurrence: decays are fp32 tables made in double precision on the host, the state
// is fp32, and every MFMA operand that carries a decay or a state (decayed keys, decayed scores, S_c) is fed as TWO bf16
// numbers hi + lo (~16 bits of mantissa); only q, k, v themselves -- projections -- are plain bf16.  Rotated q and k (ROT) are no
// projections any more: they are made in fp32 on the way in and go on as hi + lo as well.
#include "vy_decay.h"

namespace {

using namespace vy_decay;

// ---- chunked form ----------------------------------------------------------------------------
// Both kernels of a chunk request everything they read before they use any of it, and take `span` value columns, 64 at a time, so
// that keys, queries and scores are made once for all of them and the next tile is on its way while one is multiplied.  Bound by
// memory then (the states and q, k, v once are 54 us of chunk_out at 8 x 1024 tokens and 16 heads of 128 x 128, 40 us of chunk_kv):
// 135 -> 68 and 79 -> 50 us against a workgroup per 64 columns that loaded piece after piece.
__device__ __forceinline__ bf16x8 raw8(const bf16* p, bool ok) { return ok ? *reinterpret_cast<const bf16x8*>(p) : bf16x8{}; }
__device__ __forceinline__ bf16x8 act8(bf16x8 r, int silu) {   // (zero stays zero)
  if (silu) {
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (bf16)vy_silu((float)r[e]);
  }
  return r;
}
// eight key columns d .. of a chunk's token: rotated and scaled (ROT), else as loaded
template <bool ROT>
__device__ __forceinline__ void key8(const DecayArgs& a, bf16x8 raw, int pos, int d, float (&v)[8]) {
  const bf16x8 k8 = act8(raw, a.silu);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (float)k8[e];
  if constexpr (ROT) {
    if (a.half) rotate(trig_row(a, pos), a.half, d, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= a.k_scale;
  }
}

// grid (chunks, value columns / span, B * h)
template <int DKP, bool ROT>
__global__ __launch_bounds__(256) void chunk_kv_kernel(DecayArgs a, int span) {
  constexpr int KP = (DKP + 8) * 2, VP = (64 + 8) * 2, KN = C * (DKP / 8) / 256;
  static_assert(C * 8 == 512 && KN * 256 == C * (DKP / 8), "whole pieces per thread");
  __shared__ __attribute__((aligned(16))) char smem[C * (2 * KP + VP)];
  char* kh = smem;
  char* kl = smem + C * KP;
  char* vt = smem + 2 * C * KP;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int ch = blockIdx.x, bh = blockIdx.z, b = bh / a.h, head = bh - b * a.h;
  const int first_v = (int)blockIdx.y * span, end_v = min(a.dv, first_v + span);
  const int n = a.count ? min(a.count[b], a.L) : a.L;
  const int m = max(0, min(C, n - ch * C));            // tokens of this chunk
  const int first = ROT ? a.start[a.slots ? a.slots[b] : b] + ch * C : 0;
  const float* pw = a.pow + (int64_t)head * (C + 1);
  const bf16* P = (const bf16*)a.p + ((int64_t)b * a.L + ch * C) * a.ldp;
  bf16x8 k8[KN], v8[2];
  float w[KN];
  auto fetch = [&](int v0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = threadIdx.x + 256 * i, t = x >> 3, d = v0 + (x & 7) * 8;
      v8[i] = raw8(P + (int64_t)t * a.ldp + a.ov + head * a.dv + d, t < m && d < a.dv);
    }
  };
#pragma unroll
  for (int i = 0; i < KN; ++i) {
    const int x = threadIdx.x + 256 * i, t = x / (DKP / 8), d = (x % (DKP / 8)) * 8;
    k8[i] = raw8(P + (int64_t)t * a.ldp + a.ok + head * a.dk + d, t < m && d < a.dk);
    w[i] = t < m ? pw[m - 1 - t] : 0.f;
  }
  fetch(first_v);
#pragma unroll
  for (int i = 0; i < KN; ++i) {
    const int x = threadIdx.x + 256 * i, t = x / (DKP / 8), d = (x % (DKP / 8)) * 8;
    float v[8];
    key8<ROT>(a, k8[i], first + t, d, v);
    bf16x8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; ++e) { bf16 p, q; split_bf16(v[e] * w[i], p, q); hi[e] = p; lo[e] = q; }
    *reinterpret_cast<bf16x8*>(kh + t * KP + d * 2) = hi;
    *reinterpret_cast<bf16x8*>(kl + t * KP + d * 2) = lo;
  }
  float* U = a.U + ((int64_t)bh * a.nc + ch) * a.dk * a.dv;
  const int lr = 4 * kq + (r16 >> 2), lc = (4 * (r16 & 3)) * 2;
  const unsigned khb = vy_lds_addr(kh) + lr * KP + lc, klb = vy_lds_addr(kl) + lr * KP + lc, vb = vy_lds_addr(vt) + lr * VP + lc;
  for (int v0 = first_v; v0 < end_v; v0 += 64) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = threadIdx.x + 256 * i;
      *reinterpret_cast<bf16x8*>(vt + (x >> 3) * VP + (x & 7) * 16) = act8(v8[i], a.silu);
    }
    __syncthreads();
    if (v0 + 64 < end_v) fetch(v0 + 64);
    for (int blk = wave; blk < DKP / 16; blk += 4) {      // 16 key rows of the state
      if (blk * 16 >= a.dk) break;
      f32x4 acc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int tt = 0; tt < C / 32; ++tt) {
        bf16x8 fh = tr_frag<0>(khb + tt * 32 * KP + blk * 32, KP), fl = tr_frag<0>(klb + tt * 32 * KP + blk * 32, KP);
        bf16x8 fv[4];
        vy_static_for<4>([&](auto i_c) {
          constexpr int i = decltype(i_c)::value;
          fv[i] = tr_frag<i * 32>(vb + tt * 32 * VP, VP);
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        vy_tie(fh);
        vy_tie(fl);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          vy_tie(fv[i]);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl, fv[i], acc[i], 0, 0, 0);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fh, fv[i], acc[i], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = blk * 16 + 4 * kq + e, c = v0 + 16 * i + r16;
          if (r < a.dk && c < a.dv) U[(int64_t)r * a.dv + c] = acc[i][e];
        }
    }
    __syncthreads();   // the tile has been read
  }
}

// grid (chunks, value columns / span, B * h): wave w computes rows 16 w .. + 15 of the chunk (C = 64)
template <int DKP, bool ROT>
__global__ __launch_bounds__(256, 2) void chunk_out_kernel(DecayArgs a, int span) {
  static_assert(C == 64, "one 16-row block per wave");
  constexpr int KP = (DKP + 8) * 2, VP = (64 + 8) * 2, KN = C * (DKP / 8) / 256, SN = DKP * 16 / 256;
  constexpr int KS = DKP / 32, KB = ROT ? 2 : 1;        // key images: hi, lo
  __shared__ __attribute__((aligned(16))) char smem[C * (KB * KP + VP) + 2 * DKP * VP + (C + 1) * 4];
  char* kt = smem;
  char* vt = smem + KB * C * KP;
  char* sh = vt + C * VP;
  char* sl = sh + DKP * VP;
  float* pw = reinterpret_cast<float*>(sl + DKP * VP);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int ch = blockIdx.x, bh = blockIdx.z, b = bh / a.h, head = bh - b * a.h;
  const int first_v = (int)blockIdx.y * span, end_v = min(a.dv, first_v + span);
  const int rows = min(C, a.L - ch * C);
  const bf16* P = (const bf16*)a.p + ((int64_t)b * a.L + ch * C) * a.ldp;
  const float* Sg = a.U + ((int64_t)bh * a.nc + ch) * a.dk * a.dv;
  const int first = ROT ? a.start[a.slots ? a.slots[b] : b] + ch * C : 0;
  // the wave's query rows, in the k order of the transposed state fragments (4 kq .. and 16 + 4 kq ..)
  const int qi = 16 * wave + r16;
  bf16x8 k8[KN], v8[2];
  bf16x4 q4[KS][2];
  f32x4 s4[SN];
  auto fetch = [&](int v0) {
#pragma unroll
    for (int i = 0; i < SN; ++i) {
      const int x = threadIdx.x + 256 * i, r = x >> 4, c = v0 + (x & 15) * 4;
      s4[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (r < a.dk && c < a.dv) s4[i] = *reinterpret_cast<const f32x4*>(Sg + (int64_t)r * a.dv + c);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = threadIdx.x + 256 * i, t = x >> 3, d = v0 + (x & 7) * 8;
      v8[i] = raw8(P + (int64_t)t * a.ldp + a.ov + head * a.dv + d, t < rows && d < a.dv);
    }
  };
  auto put = [&]() {   // what fetch has brought
#pragma unroll
    for (int i = 0; i < SN; ++i) {
      const int x = threadIdx.x + 256 * i, at = (x >> 4) * VP + (x & 15) * 8;
      union { struct { bf16x4 hi, lo; } h; f32x4 f; } w;
      w.f = s4[i];
      *reinterpret_cast<bf16x4*>(sh + at) = w.h.hi;
      *reinterpret_cast<bf16x4*>(sl + at) = w.h.lo;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int x = threadIdx.x + 256 * i;
      *reinterpret_cast<bf16x8*>(vt + (x >> 3) * VP + (x & 7) * 16) = act8(v8[i], a.silu);
    }
  };
#pragma unroll
  for (int i = 0; i < KN; ++i) {
    const int x = threadIdx.x + 256 * i, t = x / (DKP / 8), d = (x % (DKP / 8)) * 8;
    k8[i] = raw8(P + (int64_t)t * a.ldp + a.ok + head * a.dk + d, t < rows && d < a.dk);
  }
  {
    const bf16* Q = P + (int64_t)min(qi, rows - 1) * a.ldp + a.oq + head * a.dk;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const int d = 32 * ks + 16 * hf + 4 * kq;
        q4[ks][hf] = d < a.dk ? *reinterpret_cast<const bf16x4*>(Q + d) : bf16x4{};
      }
  }
  fetch(first_v);
  if (threadIdx.x <= C) pw[threadIdx.x] = a.pow[(int64_t)head * (C + 1) + threadIdx.x];
#pragma unroll
  for (int i = 0; i < KN; ++i) {
    const int x = threadIdx.x + 256 * i, t = x / (DKP / 8), d = (x % (DKP / 8)) * 8;
    if constexpr (ROT) {
      float v[8];
      key8<true>(a, k8[i], first + t, d, v);
      bf16x8 hi, lo;
#pragma unroll
      for (int e = 0; e < 8; ++e) { bf16 p, q; split_bf16(v[e], p, q); hi[e] = p; lo[e] = q; }
      *reinterpret_cast<bf16x8*>(kt + t * KP + d * 2) = hi;
      *reinterpret_cast<bf16x8*>(kt + C * KP + t * KP + d * 2) = lo;
    } else {
      *reinterpret_cast<bf16x8*>(kt + t * KP + d * 2) = act8(k8[i], a.silu);
    }
  }
  bf16x8 qf[KS], ql[ROT ? KS : 1];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int d = 32 * ks + 16 * hf + 4 * kq;
      if constexpr (ROT) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = activate((float)q4[ks][hf][e], a.silu);
        if (a.half) rotate(trig_row(a, first + qi), a.half, d, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) { bf16 x, y; split_bf16(v[e], x, y); qf[ks][4 * hf + e] = x; ql[ks][4 * hf + e] = y; }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) qf[ks][4 * hf + e] = (bf16)activate((float)q4[ks][hf][e], a.silu);
      }
    }
  put();
  __syncthreads();
  // decayed scores, transposed, 32 keys at a time
  bf16x8 ph[C / 32], pl[C / 32];
#pragma unroll
  for (int tt = 0; tt < C / 32; ++tt) {
    if (32 * tt > 16 * wave + 15) break;
    f32x4 sc[2];
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      sc[blk] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        union { struct { bf16x4 a, b; } h; bf16x8 v; } kf;
        const char* kr = kt + (32 * tt + 16 * blk + r16) * KP + (32 * ks + 4 * kq) * 2;
        kf.h.a = *reinterpret_cast<const bf16x4*>(kr);
        kf.h.b = *reinterpret_cast<const bf16x4*>(kr + 32);
        if constexpr (ROT) {
          union { struct { bf16x4 a, b; } h; bf16x8 v; } kl;
          kl.h.a = *reinterpret_cast<const bf16x4*>(kr + C * KP);
          kl.h.b = *reinterpret_cast<const bf16x4*>(kr + C * KP + 32);
          sc[blk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kl.v, qf[ks], sc[blk], 0, 0, 0);
          sc[blk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.v, ql[ks], sc[blk], 0, 0, 0);
        }
        sc[blk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.v, qf[ks], sc[blk], 0, 0, 0);
      }
    }
#pragma unroll
    for (int blk = 0; blk < 2; ++blk)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kj = 32 * tt + 16 * blk + 4 * kq + r;
        const float s = kj <= qi ? sc[blk][r] * pw[qi - kj] : 0.f;
        bf16 x, y;
        split_bf16(s, x, y);
        ph[tt][4 * blk + r] = x;
        pl[tt][4 * blk + r] = y;
      }
  }
  const float dq = pw[qi + 1];
  const int lr = 4 * kq + (r16 >> 2), lc = (4 * (r16 & 3)) * 2;
  const unsigned shb = vy_lds_addr(sh) + lr * VP + lc, slb = vy_lds_addr(sl) + lr * VP + lc, vb = vy_lds_addr(vt) + lr * VP + lc;
  for (int v0 = first_v; v0 < end_v; v0 += 64) {
    const bool more = v0 + 64 < end_v;
    if (more) fetch(v0 + 64);
    f32x4 o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    // O^T += S^T Q^T
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      bf16x8 fh[4], fl[4];
      vy_static_for<4>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        fh[i] = tr_frag<i * 32>(shb + ks * 32 * VP, VP);
        fl[i] = tr_frag<i * 32>(slb + ks * 32 * VP, VP);
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        vy_tie(fh[i]);
        vy_tie(fl[i]);
        o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[i], qf[ks], o[i], 0, 0, 0);
        if constexpr (ROT) o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fh[i], ql[ks], o[i], 0, 0, 0);
        o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fh[i], qf[ks], o[i], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[i][e] *= dq;
    // O^T += V^T (decayed scores)^T
#pragma unroll
    for (int tt = 0; tt < C / 32; ++tt) {
      if (32 * tt > 16 * wave + 15) break;
      bf16x8 fv[4];
      vy_static_for<4>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        fv[i] = tr_frag<i * 32>(vb + tt * 32 * VP, VP);
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        vy_tie(fv[i]);
        o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fv[i], pl[tt], o[i], 0, 0, 0);
        o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fv[i], ph[tt], o[i], 0, 0, 0);
      }
    }
    if (qi < rows) {
      bf16* O = (bf16*)a.out + ((int64_t)b * a.L + ch * C + qi) * a.ldo + head * a.dv + v0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 16 * i + 4 * kq;
        if (v0 + c < a.dv) {
          bf16x4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = (bf16)o[i][e];
          *reinterpret_cast<bf16x4*>(O + c) = w;
        }
      }
    }
    if (more) {
      __syncthreads();   // the tiles have been read
      put();
      __syncthreads();
    }
  }
}

}  // namespace

extern "C" int64_t vy_decay_attn_ws_bytes(int64_t B, int64_t L, int32_t h, int32_t dk, int32_t dv, int dtype) {
  return chunked(L, dk, dtype) ? B * h * vy_cdiv(L, C) * dk * dv * 4 : 0;
}

extern "C" int vy_decay_attn(const void* p, int64_t ldp, int64_t oq, int64_t ok, int64_t ov, float* state,
                             const float* decay_pow, const int32_t* slots, const int32_t* start, const int32_t* count,
                             void* out, int64_t ldo, int64_t B, int64_t L, int32_t h, int32_t dk, int32_t dv, int silu,
                             const float* rope, int32_t rope_dims, int32_t rope_len, float k_scale, void* ws, int64_t ws_bytes,
                             int dtype, void* stream) {
  const char* who = "vy_decay_attn";
  if (!p || !state || !decay_pow || !start || !out) VY_FAIL(VY_ERR_ARG, "%s: null pointer", who);
  if (B <= 0 || L <= 0 || h <= 0 || dk <= 0 || dv <= 0 || L > INT32_MAX) VY_FAIL(VY_ERR_ARG, "%s: empty problem", who);
  if (dk % 8 || dv % 8 || ldp % 8 || ldo % 8 || oq % 8 || ok % 8 || ov % 8) VY_FAIL(VY_ERR_ARG, "%s: widths, strides and offsets must be multiples of 8", who);
  if (dtype != VY_BF16 && dtype != VY_F32) VY_FAIL(VY_ERR_ARG, "%s: bad dtype %d", who, dtype);
  if (B * h > 65535) VY_FAIL(VY_ERR_UNSUPPORTED, "%s: %ld (sequence, head) pairs", who, (long)(B * h));
  if (rope_dims < 0 || rope_dims % 2 || rope_dims > dk || (rope_dims && (!rope || rope_len < 1)))
    VY_FAIL(VY_ERR_ARG, "%s: rotary table of %d columns, %d positions for heads of %d", who, rope_dims, rope_len, dk);
  hipStream_t st = (hipStream_t)stream;
  DecayArgs a{p, ldp, oq, ok, ov, state, decay_pow, slots, start, count, out, ldo, (int)B, (int)L, h, dk, dv, silu,
              (int)vy_cdiv(L, C), (float*)ws, (const float2*)rope, rope_dims / 2, rope_len > 0 ? rope_len : 1, k_scale, nullptr, nullptr, nullptr};
  if (chunked(L, dk, dtype)) {
    if (!ws || ws_bytes < vy_decay_attn_ws_bytes(B, L, h, dk, dv, dtype)) VY_FAIL(VY_ERR_ARG, "%s: workspace too small", who);
    // all value columns in one workgroup where every CU gets one (heads of 128 x 128, chunk_out: 2048 workgroups 68 us, 4096 of 64
    // columns 89; 256 and 512: 14.0 and 14.8; 88 and 176: 12.5 and 10.0)
    const int span = B * h * a.nc >= 256 ? (int)vy_cdiv(dv, 64) * 64 : 64;
    const dim3 grid(a.nc, (unsigned)vy_cdiv(dv, span), (unsigned)(B * h)), block(256);
    const dim3 sgrid((unsigned)vy_cdiv((int64_t)dk * dv, 1024), (unsigned)(B * h));
#define CH_GO(D, ROT)                                                           \
  do {                                                                          \
    hipLaunchKernelGGL((chunk_kv_kernel<D, ROT>), grid, block, 0, st, a, span); \
    hipLaunchKernelGGL(chunk_scan_kernel<false>, sgrid, block, 0, st, a);              \
    hipLaunchKernelGGL((chunk_out_kernel<D, ROT>), grid, block, 0, st, a, span); \
  } while (0)
    const bool rot = a.half || k_scale != 1.f;
    if (dk <= 32) { if (rot) CH_GO(32, true); else CH_GO(32, false); }
    else if (dk <= 64) { if (rot) CH_GO(64, true); else CH_GO(64, false); }
    else { if (rot) CH_GO(128, true); else CH_GO(128, false); }
#undef CH_GO
  } else if (dtype == VY_BF16 ? recurrent_go<bf16, false>(a, st) : recurrent_go<float, false>(a, st)) {
    VY_FAIL(VY_ERR_UNSUPPORTED, "%s: key width %d > 512", who, dk);
  }
  VY_CHECK_LAUNCH(who);
  return VY_OK;
}
