// Native decode driver (host code) of decoders that mix layer kinds: one call runs a whole single-token step of a batch of
// sequences of different lengths -- embedding, every layer (latent attention over its latent cache or ring, decayed or gated
// linear attention over its fp32 state, or windowed or differential attention over its ring), dense or routed feed-forward behind
// or beside the mixer, final norm and vocabulary product.  See include/vyom_hip.h (vy_hybrid_decoder_step).
#include "vy_common.h"
#include "vy_few.h"
#include <utility>

int vy_residual_norm_ex(float* x, int64_t ldx, const void* y, int64_t ldy, const void* table, int64_t ldt, const int64_t* ids,
                        int64_t V, int32_t* err, float table_scale, const vy_routed_rows* routed, const float* w_post,
                        float eps_post, const float* w_pre, float eps_pre, void* h, int64_t ldh, int64_t M, int64_t N, int64_t NP,
                        int rms, int* advance, const int* slots, int n_adv, int dtype, void* stream);
int vy_residual_route(float* x, int64_t ldx, const void* y, int64_t ldy, const float* w_post, const float* w_pre, float eps, void* h,
                      int64_t ldh, int64_t M, int64_t N, int64_t NP, int rms, const vy_moe* d, int32_t* ids, float* weight, int dtype,
                      void* stream);
int vy_moe_few(const vy_moe* d, const void* h, int64_t ldh, int64_t M, const int32_t* ids, void* rows, int64_t ldr, void* ws,
               int64_t ws_bytes, int dtype, void* stream);
int vy_parallel_decode(const vy_hybrid_plan* p, const vy_hybrid_layer* L, const void* h, void* in, void* ao, void* y, void* erows,
                       int32_t* eids, float* ew, void* moe_ws, int64_t moe_ws_bytes, const int32_t* slots, const int32_t* lengths,
                       int64_t max_keys, void* mix_ws, int64_t mix_ws_bytes, void* stream);
int vy_dec_gemv1_act(const void* x, const void* w, const void* bias, int act, float act_arg, void* y, int N, int K, hipStream_t st);
int vy_rows_linear(const void* x, const void* w, const void* bias, int act, float act_arg, void* y, int64_t ldy, int64_t M, int64_t N,
                   int64_t K, hipStream_t st);
int vy_rows_parts(const void* x, const void* w, float* parts, int64_t M, int64_t N, int64_t K, hipStream_t st);
int vy_residual_norm_parts(float* x, int64_t ldx, const float* parts, int slices, const float* w_post, const float* w_pre, float eps,
                           void* h, int64_t ldh, int64_t M, int64_t N, int64_t NP, int rms, int* advance, const int* slots, int n_adv,
                           hipStream_t st);
int vy_dec_gemv1_gated(const void* x, const void* wgu, void* y, int I, int K, int act, int prescaled, float eps, hipStream_t st);
int vy_gemv_gated(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* norm_w, float eps, void* y, int64_t ldy,
                  int64_t M, int64_t I, int64_t K, int act, void* stream);

namespace {

int64_t up(int64_t x) { return (x + 255) / 256 * 256; }

struct Sizes { int64_t in, q, cq, ao, o, gu, ff, mix_ws, top, moe_ws, values; };   // widest of each over the layers

Sizes sizes_of(const vy_hybrid_plan* p) {
  Sizes s{};
  auto mx = [](int64_t& a, int64_t b) { if (b > a) a = b; };
  for (int l = 0; l < p->num_layers; ++l) {
    const vy_hybrid_layer& L = p->layers[l];
    mx(s.in, L.n_in);
    const bool parallel = L.form == VY_FORM_PARALLEL;
    mx(s.ao, (int64_t)L.heads * L.vdim + (parallel ? L.ff : 0));
    if (L.mixer == VY_MIX_LATENT) {
      if (L.w_uq) mx(s.q, (int64_t)L.heads * L.dim);
      if (L.w_uq) mx(s.cq, L.q_rank_p);
      mx(s.mix_ws, vy_latent_decode_ws_bytes(p->B, L.heads, L.kv_rank_p));
    } else if (L.mixer == VY_MIX_WINDOW) {
      mx(s.mix_ws, vy_window_decode_ws_bytes(p->B, L.heads, L.kv_heads, L.vdim, L.cap, L.diff != nullptr));
      if (L.values != VY_VALUES_OWN) mx(s.values, (int64_t)L.kv_heads * L.vdim);
    } else {
      mx(s.o, (int64_t)L.heads * L.vdim);
    }
    if (!parallel) {
      mx(s.gu, 2 * (int64_t)L.ff);
      mx(s.ff, L.ff);
    }
    if (L.moe) {
      mx(s.top, L.moe->top);
      mx(s.moe_ws, vy_moe_ws_bytes(L.moe, p->B, p->dtype));
    }
  }
  return s;
}

// y[B, N] = act(x[B, K] W^T + bias); cap: of VY_ACT_SOFTCAP
int product(const vy_hybrid_plan* p, const void* x, const void* w, void* y, int64_t ldy, int64_t N, int64_t K, void* stream,
            const void* bias = nullptr, int act = VY_ACT_NONE, float cap = 0.f) {
  if (p->dtype == VY_BF16 && p->B == 1 && N <= INT32_MAX) {
    const int rc = vy_dec_gemv1_act(x, w, bias, act, cap, y, (int)N, (int)K, (hipStream_t)stream);
    if (rc != VY_ERR_UNSUPPORTED) return rc;
  }
  if (p->dtype == VY_BF16 && p->B <= 4 && N <= INT32_MAX / 2 && vy_few::few_k(vy_few::STORE, vy_few::PLAIN, K) &&
      (act == VY_ACT_NONE || act == VY_ACT_RELU2 || act == VY_ACT_SOFTCAP) && w && (uintptr_t)w % 16 == 0 && ldy >= N) {
    vy_few::Args a{};
    a.M = (int)p->B; a.x = (const bf16*)x; a.ldx = K; a.w = (const bf16*)w; a.N = (int)N; a.bias = (const bf16*)bias; a.act = act;
    a.act_arg = cap; a.y = (bf16*)y; a.ldy = ldy;
    return vy_few::few_go(vy_few::STORE, vy_few::PLAIN, a, K, (hipStream_t)stream);
  }
  if (p->dtype == VY_BF16) {
    const int rc = vy_rows_linear(x, w, bias, act, cap, y, ldy, p->B, N, K, (hipStream_t)stream);
    if (rc != VY_ERR_UNSUPPORTED) return rc;
  }
  if (act == VY_ACT_SOFTCAP) return vy_linear_softcap_fwd(x, K, w, K, y, ldy, p->B, N, K, cap, p->dtype, stream);
  return vy_linear_fwd(x, K, w, K, bias, nullptr, 0, y, ldy, nullptr, p->B, N, K, act, p->dtype, stream);
}

constexpr int MOST_PARTS = 8;   // of vy_rows_parts
int64_t parts_bytes(const vy_hybrid_plan* p) { return p->dtype == VY_BF16 && p->B >= 5 && p->B <= 32 ? MOST_PARTS * (int64_t)p->B * p->dp * 4 : 0; }

// packed [gate | up] rows -> activation rows
int activation(const vy_hybrid_plan* p, const vy_hybrid_layer& L, const void* gu, int64_t ldg, void* act, int64_t lda, void* stream) {
  if (L.clamped) return vy_clamped_act_fwd(gu, ldg, act, lda, p->B, L.ff, L.limit, L.alpha, p->dtype, stream);
  return vy_gated_act_fwd(gu, ldg, act, lda, p->B, L.ff, p->act, p->dtype, stream);
}

int gated(const vy_hybrid_plan* p, const vy_hybrid_layer& L, const void* x, void* gu, void* act, void* stream) {
  if (!L.clamped && p->dtype == VY_BF16 && p->B == 1) {
    const int rc = vy_dec_gemv1_gated(x, L.w_gu, act, L.ff, p->dp, p->act, 0, 0.f, (hipStream_t)stream);
    if (rc != VY_ERR_UNSUPPORTED) return rc;
  }
  if (!L.clamped && p->dtype == VY_BF16 && p->B <= 4)
    return vy_gemv_gated(x, p->dp, L.w_gu, p->dp, nullptr, 0.f, act, L.ff, p->B, L.ff, p->dp, p->act, stream);
  const int rc = product(p, x, L.w_gu, gu, 2 * (int64_t)L.ff, 2 * (int64_t)L.ff, p->dp, stream);
  return rc ? rc : activation(p, L, gu, 2 * (int64_t)L.ff, act, L.ff, stream);
}

}  // namespace

extern "C" int64_t vy_hybrid_ws_bytes(const vy_hybrid_plan* p) {
  if (!p || !p->layers) return -1;
  const Sizes s = sizes_of(p);
  const int64_t e = p->dtype == VY_BF16 ? 2 : 4, B = p->B;
  return 2 * up(B * p->dp * 4) + 2 * up(B * p->dp * e) + up(B * s.in * e) + up(B * s.q * e) + up(B * s.cq * e) +
         up(B * s.ao * e) + up(B * s.o * e) + up(B * s.gu * e) + up(B * s.ff * e) + up(s.mix_ws) + up(B * s.top * p->dp * e) +
         3 * up(B * s.top * 4) + up(s.moe_ws) + up(B * s.values * e) + up(parts_bytes(p));
}

extern "C" int vy_hybrid_decoder_step(const vy_hybrid_plan* p, const int64_t* ids, const int32_t* slots, int32_t* lengths,
                                      int64_t max_keys, void* logits, int64_t ldv, void* stream) {
  const char* who = "vy_hybrid_decoder_step";
  if (!p || !p->layers || !p->ws || !ids || !lengths || !logits) VY_FAIL(VY_ERR_ARG, "%s: null plan/input/workspace/output", who);
  if (p->ws_bytes < vy_hybrid_ws_bytes(p)) VY_FAIL(VY_ERR_ARG, "%s: workspace too small", who);
  if (max_keys < 1) VY_FAIL(VY_ERR_ARG, "%s: max_keys %ld", who, (long)max_keys);
  const Sizes s = sizes_of(p);
  const int64_t e = p->dtype == VY_BF16 ? 2 : 4, B = p->B, dp = p->dp;
  char* w = (char*)p->ws;
  auto take = [&](int64_t bytes) { char* r = w; w += up(bytes); return r; };
  float* x = (float*)take(B * dp * 4);
  float* x2 = (float*)take(B * dp * 4);   // the stream behind a norm that a product has made (workgroups that read x may still run)
  void* h = take(B * dp * e);
  void* y = take(B * dp * e);
  void* in = take(B * s.in * e);
  void* q = take(B * s.q * e);
  void* cq = take(B * s.cq * e);
  void* ao = take(B * s.ao * e);
  void* o = take(B * s.o * e);
  void* gu = take(B * s.gu * e);
  void* act = take(B * s.ff * e);
  void* mws = take(s.mix_ws);
  void* erows = take(B * s.top * dp * e);
  int32_t* eids = (int32_t*)take(B * s.top * 4);
  int32_t* epos = (int32_t*)take(B * s.top * 4);
  float* ew = (float*)take(B * s.top * 4);
  void* ews = take(s.moe_ws);
  void* values = take(B * s.values * e);
  float* parts = (float*)take(parts_bytes(p));
  const vy_hybrid_layer* values_of = nullptr;   // the layer that filled them
  int rc;
  auto norm = [&](const void* yy, const vy_routed_rows* routed, const float* post, const float* pre, bool last) {
    return vy_residual_norm_ex(x, dp, yy, dp, p->embed, dp, yy || routed ? nullptr : ids, p->vocab, p->err, p->embed_scale, routed,
                               post, p->eps, pre, p->eps, h, dp, B, p->d, dp, p->rms, last ? lengths : nullptr, slots,
                               last ? (int)B : 0, p->dtype, stream);
  };
  // 1 to 4 rows: the norm in front of a product is the product's own (STREAM of vy_few.hip)
  struct { const float *post, *pre; bool last, due; } later{};
  auto settle = [&]() {
    if (!later.due) return (int)VY_OK;
    later.due = false;
    return norm(y, nullptr, later.post, later.pre, later.last);
  };
  // out = epilogue(h W^T + bias) behind whatever norm is due
  auto from_stream = [&](int epi, const void* weight, const void* bias, int act, float cap, void* out, int64_t ldo, int64_t N) {
    if (!later.due) return (int)VY_ERR_UNSUPPORTED;
    const bool known = epi == vy_few::GATED ? act == VY_ACT_SILU || act == VY_ACT_GELU_TANH
                                            : act == VY_ACT_NONE || act == VY_ACT_RELU2 || act == VY_ACT_SOFTCAP;
    if (!known || !vy_few::few_k(epi, vy_few::STREAM, dp) || N > INT32_MAX / 2 || ldo < N || !weight || (uintptr_t)weight % 16 ||
        (uintptr_t)later.post % 16 || (uintptr_t)later.pre % 16) {
      const int bad = settle();
      return bad ? bad : (int)VY_ERR_UNSUPPORTED;
    }
    vy_few::Args a{};
    a.M = (int)B; a.x = (const bf16*)y; a.ldx = dp; a.s_in = x; a.s_out = x2; a.lds = dp;
    a.w_post = later.post; a.w_pre = later.pre; a.n = p->d; a.rms = p->rms; a.eps = p->eps;
    if (later.last) { a.advance = lengths; a.slots = slots; a.n_adv = (int)B; }
    a.w = (const bf16*)weight; a.N = (int)N; a.bias = (const bf16*)bias; a.act = act; a.act_arg = cap; a.y = (bf16*)out; a.ldy = ldo;
    later.due = false;
    const int bad = vy_few::few_go(epi, vy_few::STREAM, a, dp, (hipStream_t)stream);
    std::swap(x, x2);
    return bad;
  };
  // the stream += norm(in W^T), then its next norm: with few rows the product leaves slices that the norm adds up, or the norm waits
  // for the product that reads it (`own`: such a product is the next launch)
  auto into_stream = [&](const void* xin, const void* weight, int64_t K, const float* post, const float* pre, bool last, bool own) {
    if (own && p->dtype == VY_BF16 && B <= 4) {
      const int bad = product(p, xin, weight, y, dp, dp, K, stream);
      later = {post, pre, last, true};
      return bad;
    }
    const int n = parts_bytes(p) ? vy_rows_parts(xin, weight, parts, B, dp, K, (hipStream_t)stream) : 0;
    if (n)
      return vy_residual_norm_parts(x, dp, parts, n, post, pre, p->eps, h, dp, B, p->d, dp, p->rms, last ? lengths : nullptr, slots,
                                    last ? (int)B : 0, (hipStream_t)stream);
    const int bad = product(p, xin, weight, y, dp, dp, K, stream);
    return bad ? bad : norm(y, nullptr, post, pre, last);
  };
  if ((rc = norm(nullptr, nullptr, nullptr, p->layers[0].norm1, false))) return rc;
  for (int l = 0; l < p->num_layers; ++l) {
    const vy_hybrid_layer& L = p->layers[l];
    const bool last = l + 1 == p->num_layers, parallel = L.form == VY_FORM_PARALLEL;
    const float* next = last ? p->final_norm : p->layers[l + 1].norm1;
    const bool own = last || p->layers[l + 1].form != VY_FORM_PARALLEL;
    const int64_t nv = (int64_t)L.heads * L.vdim, nk = (int64_t)L.heads * L.dim, na = nv + (parallel ? L.ff : 0);
    if (parallel) {   // windowed attention beside clamped feed-forwards: the pieces of the layer share launches
      rc = vy_parallel_decode(p, &L, h, in, ao, y, erows, eids, ew, ews, s.moe_ws, slots, lengths, max_keys, mws, s.mix_ws, stream);
      if (rc == VY_OK) {
        const vy_routed_rows rows{erows, dp, nullptr, ew, L.moe ? L.moe->top : 0};
        if ((rc = norm(y, L.moe ? &rows : nullptr, L.norm1b, next, last))) return rc;
        continue;
      }
      if (rc != VY_ERR_UNSUPPORTED) return rc;
    }
    rc = from_stream(vy_few::STORE, L.w_in, L.b_in, VY_ACT_NONE, 0.f, in, L.n_in, L.n_in);
    if (rc == VY_ERR_UNSUPPORTED) rc = product(p, h, L.w_in, in, L.n_in, L.n_in, dp, stream, L.b_in);
    if (rc) return rc;
    if (L.mixer == VY_MIX_LATENT) {
      if (!L.ring && max_keys > L.cap) VY_FAIL(VY_ERR_ARG, "%s: %ld keys exceed the cache capacity %d", who, (long)max_keys, L.cap);
      const int64_t nq = L.w_uq ? L.q_rank_p : nk;   // columns ahead of the key/value latent: the queries' latent, or the queries
      // 1 to 4 rows: the queries' product norms its latent itself, beside the new tokens' cache rows (2.4 + 3.0 us of a layer -> 3.3; the
      // gated norm in front of an output projection, done the same way, gave nothing: 2.1 + 2.6 -> 4.3)
      const bool own_norm = L.w_uq && p->dtype == VY_BF16 && B <= 4 && vy_few::few_k(vy_few::STORE, vy_few::RMS, L.q_rank_p) && L.q_norm && L.c_norm &&
                            L.cache && L.cap > 0 && L.kv_rank > 0 && L.kv_rank_p >= L.kv_rank && L.kv_rank_p <= 1024 && L.q_rank > 0 && L.q_rank <= L.q_rank_p &&
                            (L.kv_rank_p | L.n_in | L.c_ss | L.c_st) % 8 == 0 && nk <= INT32_MAX &&
                            ((uintptr_t)L.w_uq | (uintptr_t)L.q_norm | (uintptr_t)L.cache) % 16 == 0;
      if (own_norm) {
        vy_few::Args a{};
        a.M = (int)B; a.x = (const bf16*)in; a.ldx = L.n_in; a.w_pre = L.q_norm; a.n = L.q_rank; a.eps = p->eps;
        a.kv = (const bf16*)in + nq; a.w_kv = L.c_norm; a.n_kv = L.kv_rank; a.np_kv = L.kv_rank_p; a.cache = (bf16*)L.cache;
        a.k_ss = L.c_ss; a.k_st = L.c_st; a.cap = L.cap; a.ring = L.ring; a.start = lengths; a.slots = slots;
        a.w = (const bf16*)L.w_uq; a.N = (int)nk; a.y = (bf16*)q; a.ldy = nk;
        if ((rc = vy_few::few_go(vy_few::STORE, vy_few::RMS, a, L.q_rank_p, (hipStream_t)stream))) return rc;
      } else {
        if ((rc = vy_latent_norm(in, L.n_in, L.w_uq ? L.q_norm : nullptr, cq, L.q_rank_p, L.q_rank, (int)nq, L.c_norm, nullptr, 0, L.kv_rank,
                                 L.kv_rank_p, L.cache, L.c_ss, L.c_st, L.cap, L.ring, slots, lengths, nullptr, B, 1, p->eps, p->dtype,
                                 stream))) return rc;
        if (L.w_uq && (rc = product(p, cq, L.w_uq, q, nk, nk, L.q_rank_p, stream))) return rc;
      }
      const char* gate = L.gate ? (const char*)in + (nq + L.kv_rank_p) * e : nullptr;
      if ((rc = vy_latent_decode(L.w_uq ? q : in, L.w_uq ? nk : L.n_in, L.w_ukt, L.w_uv, L.cache, L.c_ss, L.c_st, slots, lengths, max_keys, ao,
                                 na, gate, L.n_in, L.gate_heads, L.ring ? L.cap : 0, (int)B, L.heads, L.dim, L.vdim, L.kv_rank_p,
                                 L.scale, mws, s.mix_ws, p->dtype, stream)))
        return rc;
    } else if (L.mixer == VY_MIX_WINDOW) {
      const int64_t gk = (int64_t)L.kv_heads * L.dim, gv = (int64_t)L.kv_heads * L.vdim;
      vy_qkv_prep prep{};
      if (L.prep) prep = *L.prep;
      if (L.values == VY_VALUES_FIRST) {
        prep.v_out = values;
        prep.ldo = gv;
        values_of = &L;
      } else if (L.values == VY_VALUES_MIX) {
        const vy_hybrid_layer* F = values_of;
        if (!F || !F->prep || F->kv_heads * F->prep->n_v != L.kv_heads * prep.n_v)
          VY_FAIL(VY_ERR_ARG, "%s: layer %d has no values to mix in", who, l);
        prep.v_mix = values;
        prep.ldm = (int64_t)F->kv_heads * F->vdim;
        prep.m_v = F->prep->n_v;
        prep.m_vp = F->vdim;
      }
      if ((rc = vy_window_decode(in, L.n_in, 0, nk, nk + gk, L.gate ? nk + gk + gv : -1, L.cache, L.c_ss, L.c_sh, L.cap, L.keep, L.rope,
                                 L.rope_dims, L.rope_len, L.prep || L.values != VY_VALUES_OWN ? &prep : nullptr, L.diff, slots, lengths, max_keys, ao, na, B, L.heads, L.kv_heads, L.dim, L.vdim, L.scale,
                                 L.sink, mws, s.mix_ws, p->dtype, stream))) return rc;
    } else if (L.mixer == VY_MIX_GATED) {
      if ((rc = vy_gated_attn(in, L.n_in, 0, nk, 2 * nk, L.state, L.f_bias, L.f_lower, slots, lengths, nullptr, o, nv, B, 1, L.heads, L.dim,
                              L.vdim, L.silu, nullptr, 0, p->dtype, stream))) return rc;
      if ((rc = vy_head_norm_gate(o, nv, L.mix_norm, nullptr, 0, ao, na, B, L.heads, L.mix_n, L.vdim, p->eps, p->dtype, stream))) return rc;
    } else {
      if ((rc = vy_decay_attn(in, L.n_in, 0, nk, 2 * nk, L.state, L.decay_pow, slots, lengths, nullptr, o, nv, B, 1, L.heads, L.dim,
                              L.vdim, L.silu, L.rope, L.rope_dims, L.rope_len, L.k_scale, nullptr, 0, p->dtype, stream))) return rc;
      const char* gate = (const char*)in + (2 * nk + nv) * e;
      if (!L.mix_norm) {
        if ((rc = vy_head_norm_gate(o, nv, nullptr, gate, L.n_in, ao, na, B, L.heads, L.mix_n, L.vdim, p->eps, p->dtype, stream))) return rc;
      } else if ((rc = vy_rmsnorm_gate(o, nv, L.mix_norm, gate, L.n_in, ao, na, B, L.mix_n, nv, p->eps, p->dtype, stream))) return rc;
    }
    vy_routed_rows rows{erows, dp, epos, ew, L.moe ? L.moe->top : 0};
    const vy_routed_rows* routed = L.moe ? &rows : nullptr;
    auto experts = [&]() {
      return L.moe ? vy_moe_fwd(L.moe, h, dp, B, nullptr, 1, erows, dp, eids, epos, ew, ews, s.moe_ws, p->dtype, stream) : VY_OK;
    };
    if (parallel) {
      if (L.ff && (rc = activation(p, L, (const char*)in + (L.n_in - 2 * (int64_t)L.ff) * e, L.n_in, (char*)ao + nv * e, na, stream)))
        return rc;
      if ((rc = experts())) return rc;
      if ((rc = product(p, ao, L.w_o, y, dp, dp, na, stream))) return rc;
      if ((rc = norm(y, routed, L.norm1b, next, last))) return rc;
      continue;
    }
    if (!L.ff && !L.moe) {
      if ((rc = into_stream(ao, L.w_o, nv, L.norm1b, next, last, own))) return rc;
      continue;
    }
    // few tokens: the choice of experts comes with the residual sum
    bool chosen = false;
    if (L.moe) {
      if ((rc = product(p, ao, L.w_o, y, dp, dp, nv, stream))) return rc;
      rc = vy_moe_few(L.moe, nullptr, 0, B, nullptr, nullptr, 0, nullptr, 0, p->dtype, stream);
      if (rc == VY_OK)
        rc = vy_residual_route(x, dp, y, dp, L.norm1b, L.norm2, p->eps, h, dp, B, p->d, dp, p->rms, L.moe, eids, ew, p->dtype, stream);
      if (rc && rc != VY_ERR_UNSUPPORTED) return rc;
      chosen = rc == VY_OK;
      if (!chosen && (rc = norm(y, nullptr, L.norm1b, L.norm2, false))) return rc;
    } else if ((rc = into_stream(ao, L.w_o, nv, L.norm1b, L.norm2, false, true))) {
      return rc;
    }
    if (L.ff) {
      if (L.w_up) {
        rc = from_stream(vy_few::STORE, L.w_up, nullptr, p->act, 0.f, act, L.ff, L.ff);
        if (rc == VY_ERR_UNSUPPORTED) rc = product(p, h, L.w_up, act, L.ff, L.ff, dp, stream, nullptr, p->act);
      } else {
        rc = from_stream(vy_few::GATED, L.w_gu, nullptr, L.clamped ? VY_ACT_NONE : p->act, 0.f, act, L.ff, L.ff);
        if (rc == VY_ERR_UNSUPPORTED) rc = gated(p, L, h, gu, act, stream);
      }
      if (rc) return rc;
      if (!L.moe) {
        if ((rc = into_stream(act, L.w_down, L.ff, L.norm2b, next, last, own))) return rc;
        continue;
      }
      if ((rc = product(p, act, L.w_down, y, dp, dp, L.ff, stream))) return rc;
    }
    if (chosen) {
      rows.pos = nullptr;
      rc = vy_moe_few(L.moe, h, dp, B, eids, erows, dp, ews, s.moe_ws, p->dtype, stream);
    } else {
      rc = experts();
    }
    if (rc) return rc;
    if ((rc = norm(L.ff ? y : nullptr, routed, L.norm2b, next, last))) return rc;
  }
  const int cap = p->softcap > 0.f ? VY_ACT_SOFTCAP : VY_ACT_NONE;
  rc = from_stream(vy_few::STORE, p->head, nullptr, cap, p->softcap, logits, ldv, p->vocab);
  return rc == VY_ERR_UNSUPPORTED ? product(p, h, p->head, logits, ldv, p->vocab, dp, stream, nullptr, cap, p->softcap) : rc;
}
