// Native decode driver (host code): chains the kernel launchers for one single-token step so the
// Python side makes ONE call per generated token.  See include/vyom_hip.h (vy_decoder_step).
#include "vy_common.h"
#include "vy_few.h"
#include <stdlib.h>
#include <initializer_list>

int vy_qkv_rope_fwd_ex(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias,
                       const float* cos_tab, const float* sin_tab, int64_t pos0, const int* pos_dev, void* q,
                       int64_t q_sb, int64_t q_sh, int64_t q_sl, void* k, int64_t k_sb, int64_t k_sh, int64_t k_sl,
                       void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl, int64_t B, int64_t L, int64_t K, int h,
                       int hk, int dh, int dtype, void* stream);
int vy_attn_decode_ex(const void* q, int64_t q_sb, int64_t q_sh, const void* k, int64_t k_sb, int64_t k_sh,
                      int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl, void* out,
                      int64_t o_sb, int64_t B, int h, int hk, int64_t S, const int* pos_dev, int dh, float scale,
                      int dtype, void* stream);

int vy_gemv_norm(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* norm_w, float eps,
                 const void* residual, int64_t ldr, void* y, int64_t ldy, int64_t M, int64_t N, int64_t K, void* stream);
int vy_gemv_qkv_norm(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* norm_w, float eps,
                     void* q, int64_t q_sb, int64_t q_sh, void* k, int64_t k_sb, int64_t k_sh, int64_t k_sl, void* v,
                     int64_t v_sb, int64_t v_sh, int64_t v_sl, int64_t B, int64_t K, int h, int hk, int dh,
                     const float* cos_tab, const float* sin_tab, int64_t pos, void* stream);
#define VY_NORM_PRESCALED ((const void*)(intptr_t)-1)
int vy_gemv_gated(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* norm_w, float eps, void* y, int64_t ldy,
                  int64_t M, int64_t I, int64_t K, int act, void* stream);
int vy_rope_qk(void* q, int64_t q_sb, int64_t q_sh, int64_t q_sl, int hq, void* k, int64_t k_sb, int64_t k_sh,
               int64_t k_sl, int hk, const float* cos_tab, const float* sin_tab, int64_t pos0, int64_t B, int64_t L, int dh,
               int dtype, hipStream_t st);
int64_t vy_splitk_ws_floats(int64_t N);
int vy_linear_res_ln_skinny(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias,
                            const void* residual, int64_t ldr, const void* gamma, const void* beta, float eps,
                            void* y, int64_t ldy, float* part, int64_t M, int64_t N, int64_t K, void* stream);

// lean decode kernels (vy_decode.hip)
bool vy_dec_supported(int B, int d, int h, int hk, int dh, int ffn, int dtype);
int vy_dec_qkv(const void* x, const void* w, const void* bias, const float* cos_tab, const float* sin_tab, int64_t pos0,
               const int* pos_dev, void* q, void* k, void* v, int64_t c_sb, int64_t c_sh, int64_t c_sl, int B, int d, int h,
               int hk, hipStream_t st);
int vy_dec_linear_ex(const void* x, int ldx, const void* w, const void* bias, const void* residual, int ldr, const void* ln_g,
                     const void* ln_b, float ln_eps, void* y, int ldy, int B, int N, int K, int act, hipStream_t st);
int vy_dec_attn_out(const void* q, const void* k, const void* v, int64_t c_sb, int64_t c_sh, int64_t c_sl, const void* wo, float* part,
                    int64_t room, int B, int h, int hk, int64_t S, int64_t smax, const int* pos_dev, float scale, hipStream_t st);
int vy_dec_linear(const void* x, int ldx, const void* w, const void* bias, void* y, int ldy, int B, int N, int K, int act,
                  hipStream_t st);
int vy_dec_linear_res_ln(const void* x, int ldx, const void* w, const void* bias, const void* residual, int ldr,
                         const void* gamma, const void* beta, float eps, void* y, int ldy, float* part, int B, int N, int K,
                         int act, hipStream_t st);

static int g_decode_lean = -1;
static int g_gemma_lean = -1;
extern "C" int vy_debug_set_gemma_lean(int v) { g_gemma_lean = v; return 0; }   // test aid: 0 = general kernels for B = 1 too
// measurement / test aid, not part of include/vyom_hip.h: 0 = general launchers, 1 = the decode-only kernels
extern "C" int vy_debug_set_decode_lean(int v) { g_decode_lean = v; return 0; }

int vy_dec_gemv1(const void* x, const void* w, const void* bias, const void* residual, void* y, int N, int K, int prescaled,
                 float eps, hipStream_t st);
int vy_dec_gemv1_gated(const void* x, const void* wgu, void* y, int I, int K, int act, int prescaled, float eps, hipStream_t st);
int vy_dec_gemv1_qkv(const void* x, const void* w, const void* bias, void* q, void* k, void* v, int64_t c_sh, int h, int hk,
                     int dh, const float* cos_tab, const float* sin_tab, int64_t pos, int K, int prescaled, float eps,
                     hipStream_t st);

namespace {
inline int64_t esize(int dtype) { return dtype == VY_BF16 ? 2 : 4; }
inline int64_t up(int64_t x) { return (x + 255) / 256 * 256; }
}  // namespace

extern "C" int64_t vy_decode_ws_bytes(int32_t B, int32_t d, int32_t h, int32_t hk, int32_t dh, int32_t ffn,
                                      int32_t dtype) {
  const int64_t e = esize(dtype);
  // q, attn out, s (pre-LN), a (post-LN1), mid (ffn), two ping-pong hidden buffers, split-K partials
  return up(B * (int64_t)h * dh * e) + 5 * up(B * (int64_t)d * e) + up(B * (int64_t)ffn * e) +
         up((vy_splitk_ws_floats(d) > 24 * 32 * (int64_t)d ? vy_splitk_ws_floats(d) : 24 * 32 * (int64_t)d) * 4) + 4096;
}

// Do the kernels of vy_few.hip take the step's sizes and operands?  (whole 256-column pieces, weights and the hidden rows on 16 bytes,
// norms on 8; a null weight or norm is the general launchers' to refuse or to leave out)
static bool few_operands(const vy_decode_plan* p, const void* x, const void* hidden_out, const void* logits) {
  using namespace vy_few;
  if (!few_k(QKV, PLAIN, p->d) || !few_k(QKV, LAYER, p->d) || !few_k(STORE, PLAIN, p->d) || !few_k(STORE, LAYER, p->d) ||
      !few_k(STORE, PLAIN, p->ffn) || p->dh != 64 || p->h * 64 != p->d ||
      (p->act != VY_ACT_NONE && p->act != VY_ACT_GELU_ERF && p->act != VY_ACT_GELU_TANH))
    return false;
  uintptr_t all = (uintptr_t)hidden_out;   // the low bits of every address
  bool given = true;
  auto need = [&](std::initializer_list<const void*> weights, std::initializer_list<const void*> norms) {
    for (const void* w : weights) { all |= (uintptr_t)w; given = given && w; }
    for (const void* n : norms) { all |= (uintptr_t)n << 1; given = given && n; }
  };
  need({x}, {});
  for (int l = 0; l < p->num_layers; ++l) {
    const vy_decode_layer& L = p->layers[l];
    need({L.wqkv, L.wo, L.w1, L.w2}, {L.ln1_w, L.ln1_b, L.ln2_w, L.ln2_b});
  }
  if (logits) need({p->head_wd, p->head_wv}, {p->head_ln_w, p->head_ln_b});
  return given && all % 16 == 0 && (!logits || p->vocab > 0);
}

// Does the output projection go into the attention (vy_dec_attn_out)?  That saves a launch, 1.2 us of a layer, but every workgroup of the
// feed-forward's first product then adds up the heads' fp32 shares -- h B d of them, out of L2 -- and query heads that share a key head are
// attended to by one workgroup, which three and four of them only repay where their keys are streamed otherwise (kv_bytes: one layer's keys
// and values, against the 1 MB above which vy_dec_attn streams them).  A step with the projection inside / by itself, 12 layers, us:
//   one sequence: 512 columns 168 / 184 behind 60 tokens, 768 191 / 206, behind 500 209 / 241; 1024 244 / 239, but 264 / 275 behind 640 where
//   two heads share streamed keys
//   two: 512 columns 176 / 193, 768 217 / 221 and 235 / 256, 1024 291 / 255;   four: 512 204 / 207, 768 260 / 243, 1024 401 / 292
//   two heads a key head, 768 columns: three sequences 233 / 235 and 259 / 272, four 239 / 237 and 265 / 275
//   three: two sequences 215 / 217 behind 60, 245 / 236 behind 500, three 240 / 232 and 271 / 286, four 244 / 237 and 277 / 290
//   four: two sequences 226 / 217, behind 500 262 / 236, three behind 500 288 / 302
//   six: two sequences 212 / 217, three 247 / 234, behind 700 tokens 273 / 296
bool vy_dec_shares_pay(int B, int h, int hk, int64_t kv_bytes) {
  const int d = 64 * h, rep = hk > 0 ? h / hk : 1, units = rep >= 2 && rep <= 4 ? hk : h;
  const bool streamed = kv_bytes > (1 << 20);
  if (B == 1) return d <= 768 || (rep > 1 && streamed);
  if (d > 768) return false;   // (the product's sums of two and more rows of 1024 columns: registers)
  if (rep == 3 || rep == 4) return streamed;
  return units * B * d * 4 <= (72 << 10) || (rep > 4 && streamed);
}

// The step of 1 to 4 sequences on the kernels of vy_few.hip: four launches per layer -- LayerNorms inside the products behind them, the
// output projection inside the attention -- or five, the projection by itself (vy_dec_shares_pay; longer contexts).
static int few_decoder_step(const vy_decode_plan* p, const void* x, int64_t pos, const int32_t* pos_dev, void* hidden_out, void* logits,
                            int64_t ldv, hipStream_t st) {
  using namespace vy_few;
  const int64_t e = 2;
  const int B = p->B, d = p->d, h = p->h, hk = p->hk;
  char* w = (char*)p->ws;
  auto take = [&](int64_t n) { char* r = w; w += up(n * e); return (bf16*)r; };
  bf16 *q = take(B * (int64_t)d), *ao = take(B * (int64_t)d), *s1 = take(B * (int64_t)d), *s2 = take(B * (int64_t)d);
  bf16* hb[2] = {take(B * (int64_t)d), take(B * (int64_t)d)};
  bf16* mid = take(B * (int64_t)p->ffn);
  float* part = (float*)w;            // the attention heads' shares of the output projection
  const int64_t part_bytes = 24 * 32 * (int64_t)d * 4;   // (vy_decode_ws_bytes)
  const bf16* cur = (const bf16*)x;   // the layer's input rows: of the first layer x, of the others LN2 of the layer before
  const vy_decode_layer* before = nullptr;
  int rc;
  for (int l = 0; l < p->num_layers; ++l) {
    const vy_decode_layer& L = p->layers[l];
    Args a{};
    a.M = B; a.w = (const bf16*)L.wqkv; a.bias = (const bf16*)L.bqkv; a.N = (h + 2 * hk) * 64;
    a.q = q; a.k = (bf16*)L.kcache; a.v = (bf16*)L.vcache; a.c_sb = L.c_sb; a.c_sh = L.c_sh; a.c_sl = L.c_sl;
    a.cos_tab = p->cos_tab; a.sin_tab = p->sin_tab; a.pos_dev = pos_dev; a.pos = (int)pos; a.nq = h * 64; a.nkv = hk * 64;
    if (before) {
      a.x = s2; a.ldx = d; a.ln_g = (const bf16*)before->ln2_w; a.ln_b = (const bf16*)before->ln2_b; a.eps = p->eps_ffn;
      a.h = hb[l & 1]; a.ldh = d;
      cur = hb[l & 1];
    } else {
      a.x = cur; a.ldx = d;
    }
    if ((rc = few_go(QKV, before ? LAYER : PLAIN, a, d, st))) return rc;
    Args f{};
    f.M = B; f.ln_g = (const bf16*)L.ln1_w; f.ln_b = (const bf16*)L.ln1_b; f.eps = p->eps_attn;
    f.w = (const bf16*)L.w1; f.bias = (const bf16*)L.b1; f.N = p->ffn; f.act = p->act; f.y = mid; f.ldy = p->ffn;
    const int64_t smax = L.c_sh / (L.c_sl ? L.c_sl : 1), kv_bytes = 2ll * B * hk * (pos_dev ? smax : pos + 1) * 64 * 2;
    const int shares = few_k(STORE, PARTS, d) && (uintptr_t)L.bo % 8 == 0 && vy_dec_shares_pay(B, h, hk, kv_bytes)
                           ? vy_dec_attn_out(q, L.kcache, L.vcache, L.c_sb, L.c_sh, L.c_sl, L.wo, part, part_bytes, B, h, hk, pos + 1, smax,
                                             pos_dev, 0.125f, st)
                           : 0;
    if (shares < 0) return shares;
    if (shares) {
      f.parts = part; f.n_parts = shares; f.x_bias = (const bf16*)L.bo; f.x = cur; f.ldx = d;
      if ((rc = few_go(STORE, PARTS, f, d, st))) return rc;
    } else {
      if ((rc = vy_attn_decode_ex(q, d, 64, L.kcache, L.c_sb, L.c_sh, L.c_sl, L.vcache, L.c_sb, L.c_sh, L.c_sl, ao, d, B, h, hk, pos + 1,
                                  pos_dev, 64, 0.125f, VY_BF16, st))) return rc;
      Args o{};
      o.M = B; o.x = ao; o.ldx = d; o.w = (const bf16*)L.wo; o.bias = (const bf16*)L.bo; o.N = d; o.residual = cur; o.ldr = d;
      o.y = s1; o.ldy = d;
      if ((rc = few_go(STORE, PLAIN, o, d, st))) return rc;
      f.x = s1; f.ldx = d;
      if ((rc = few_go(STORE, LAYER, f, d, st))) return rc;
    }
    Args g{};
    g.M = B; g.x = mid; g.ldx = p->ffn; g.w = (const bf16*)L.w2; g.bias = (const bf16*)L.b2; g.N = d; g.residual = cur; g.ldr = d;
    g.y = s2; g.ldy = d;
    if ((rc = few_go(STORE, PLAIN, g, p->ffn, st))) return rc;
    before = &L;
  }
  if (!logits)
    return hidden_out ? vy_layernorm_fwd(s2, d, before->ln2_w, before->ln2_b, hidden_out, d, nullptr, nullptr, B, d, p->eps_ffn, VY_BF16, st)
                      : VY_OK;
  Args a{};
  a.M = B; a.x = s2; a.ldx = d; a.ln_g = (const bf16*)before->ln2_w; a.ln_b = (const bf16*)before->ln2_b; a.eps = p->eps_ffn;
  a.h = (bf16*)hidden_out; a.ldh = d; a.w = (const bf16*)p->head_wd; a.bias = (const bf16*)p->head_bd; a.N = d; a.act = VY_ACT_GELU_ERF;
  a.y = s1; a.ldy = d;
  if ((rc = few_go(STORE, LAYER, a, d, st))) return rc;
  Args v{};
  v.M = B; v.x = s1; v.ldx = d; v.ln_g = (const bf16*)p->head_ln_w; v.ln_b = (const bf16*)p->head_ln_b; v.eps = p->eps_head;
  v.w = (const bf16*)p->head_wv; v.once = 1; v.bias = (const bf16*)p->head_bias; v.N = p->vocab; v.y = (bf16*)logits; v.ldy = ldv;
  return few_go(STORE, LAYER, v, d, st);
}

extern "C" int vy_decoder_step(const vy_decode_plan* p, const void* x, int64_t pos, const int32_t* pos_dev,
                               void* hidden_out, void* logits, int64_t ldv, void* stream) {
  const char* who = "vy_decoder_step";
  if (!p || !x || !p->layers || !p->ws) VY_FAIL(VY_ERR_ARG, "%s: null plan/input/workspace", who);
  if (p->ws_bytes < vy_decode_ws_bytes(p->B, p->d, p->h, p->hk, p->dh, p->ffn, p->dtype))
    VY_FAIL(VY_ERR_ARG, "%s: workspace too small", who);
  if (logits && ldv < p->vocab) VY_FAIL(VY_ERR_ARG, "%s: logits rows of %ld for a vocabulary of %d", who, (long)ldv, p->vocab);
  const int64_t e = esize(p->dtype);
  const int B = p->B, d = p->d, h = p->h, hk = p->hk, dh = p->dh;
  char* w = (char*)p->ws;
  void* q = w; w += up(B * (int64_t)h * dh * e);
  void* ao = w; w += up(B * (int64_t)d * e);
  void* s = w; w += up(B * (int64_t)d * e);
  void* a = w; w += up(B * (int64_t)d * e);
  void* hb[2];
  hb[0] = w; w += up(B * (int64_t)d * e);
  hb[1] = w; w += up(B * (int64_t)d * e);
  void* mid = w; w += up(B * (int64_t)p->ffn * e);
  float* part = (float*)w;
  // M <= 32 rows in bf16: the two N = d projections (24 workgroups as plain skinny GEMMs) run split-K
  // over ~all CUs, their bias + residual + LayerNorm fused into the kernel that adds the partials
  const bool splitk = p->dtype == VY_BF16 && B <= 32 && d % 32 == 0 && d <= 8192 && p->ffn % 16 == 0;
  const float scale = 1.0f / sqrtf((float)dh);
  // the decode-only kernels of vy_decode.hip (short dependent chains): bf16, 64-wide heads, K of every projection a
  // chunk size they exist for (VY_DECODE_LEAN=0: the general launchers, for A/B runs and the equality test)
  if (g_decode_lean < 0) { const char* e = getenv("VY_DECODE_LEAN"); g_decode_lean = e ? atoi(e) : 1; }
  const bool lean = g_decode_lean && vy_dec_supported(B, d, h, hk, dh, p->ffn, p->dtype);
  hipStream_t hst = (hipStream_t)stream;
  if (lean && B <= 4 && p->num_layers > 0 && (pos_dev || pos >= 0) && few_operands(p, x, hidden_out, logits))
    return few_decoder_step(p, x, pos, pos_dev, hidden_out, logits, ldv, hst);
  const void* cur = x;
  for (int l = 0; l < p->num_layers; ++l) {
    const vy_decode_layer& L = p->layers[l];
    if (!pos_dev && pos < 0) VY_FAIL(VY_ERR_ARG, "%s: negative position", who);
    // K/V of this token go straight into the cache at index pos (host offset, or the kernel adds
    // *pos_dev itself when the step is being captured into a graph)
    const int64_t hpos = pos_dev ? 0 : pos;
    void* kdst = (char*)L.kcache + hpos * L.c_sl * e;
    void* vdst = (char*)L.vcache + hpos * L.c_sl * e;
    if (lean) {
      int rc = vy_dec_qkv(cur, L.wqkv, L.bqkv, p->cos_tab, p->sin_tab, pos, pos_dev, q, kdst, vdst, L.c_sb, L.c_sh, L.c_sl, B,
                          d, h, hk, hst);
      if (rc) return rc;
      rc = vy_attn_decode_ex(q, (int64_t)h * dh, dh, L.kcache, L.c_sb, L.c_sh, L.c_sl, L.vcache, L.c_sb, L.c_sh,
                             L.c_sl, ao, d, B, h, hk, pos + 1, pos_dev, dh, scale, p->dtype, stream);
      if (rc) return rc;
      // LN1's output feeds FFN1 only (the FFN residual is the layer input): the out-projection keeps whole rows per
      // workgroup (K = d is one chunk: 16-column workgroups, bias + residual in the epilogue) and FFN1 normalises its
      // input rows on the way in -- no split-K partials, no finish + LayerNorm launch: 6 links per layer instead of 7
      static const int lnfold = [] { const char* e = getenv("VY_DEC_LNFOLD"); return e ? atoi(e) : 1; }();
      if (lnfold) {
        rc = vy_dec_linear_ex(ao, d, L.wo, L.bo, cur, d, nullptr, nullptr, 0.f, s, d, B, d, d, VY_ACT_NONE, hst);
        if (rc) return rc;
        rc = vy_dec_linear_ex(s, d, L.w1, L.b1, nullptr, 0, L.ln1_w, L.ln1_b, p->eps_attn, mid, p->ffn, B, p->ffn, d, p->act, hst);
        if (rc) return rc;
      } else {
        rc = vy_dec_linear_res_ln(ao, d, L.wo, L.bo, cur, d, L.ln1_w, L.ln1_b, p->eps_attn, a, d, part, B, d, d, VY_ACT_NONE, hst);
        if (rc) return rc;
        rc = vy_dec_linear(a, d, L.w1, L.b1, mid, p->ffn, B, p->ffn, d, p->act, hst);
        if (rc) return rc;
      }
      void* nxt_l = hb[l & 1];   // FFN residual = the LAYER INPUT (reference models/decoder.py:241-250)
      rc = vy_dec_linear_res_ln(mid, p->ffn, L.w2, L.b2, cur, d, L.ln2_w, L.ln2_b, p->eps_ffn, nxt_l, d, part, B, d, p->ffn,
                                VY_ACT_NONE, hst);
      if (rc) return rc;
      cur = nxt_l;
      continue;
    }
    int rc = vy_qkv_rope_fwd_ex(cur, d, L.wqkv, d, L.bqkv, p->cos_tab, p->sin_tab, pos, pos_dev, q, (int64_t)h * dh,
                                dh, dh, kdst, L.c_sb, L.c_sh, L.c_sl, vdst, L.c_sb, L.c_sh, L.c_sl, B, 1, d, h, hk,
                                dh, p->dtype, stream);
    if (rc) return rc;
    rc = vy_attn_decode_ex(q, (int64_t)h * dh, dh, L.kcache, L.c_sb, L.c_sh, L.c_sl, L.vcache, L.c_sb, L.c_sh,
                           L.c_sl, ao, d, B, h, hk, pos + 1, pos_dev, dh, scale, p->dtype, stream);
    if (rc) return rc;
    if (splitk) {
      rc = vy_linear_res_ln_skinny(ao, d, L.wo, d, L.bo, cur, d, L.ln1_w, L.ln1_b, p->eps_attn, a, d, part, B, d, d, stream);
      if (rc) return rc;
    } else {
      rc = vy_linear_fwd(ao, d, L.wo, d, L.bo, cur, d, s, d, nullptr, B, d, d, VY_ACT_NONE, p->dtype, stream);
      if (rc) return rc;
      rc = vy_layernorm_fwd(s, d, L.ln1_w, L.ln1_b, a, d, nullptr, nullptr, B, d, p->eps_attn, p->dtype, stream);
      if (rc) return rc;
    }
    rc = vy_linear_fwd(a, d, L.w1, d, L.b1, nullptr, 0, mid, p->ffn, nullptr, B, p->ffn, d, p->act, p->dtype, stream);
    if (rc) return rc;
    // FFN residual = the LAYER INPUT (reference models/decoder.py:241-250)
    void* nxt = hb[l & 1];
    if (splitk) {
      rc = vy_linear_res_ln_skinny(mid, p->ffn, L.w2, p->ffn, L.b2, cur, d, L.ln2_w, L.ln2_b, p->eps_ffn, nxt, d, part, B,
                                   d, p->ffn, stream);
      if (rc) return rc;
    } else {
      rc = vy_linear_fwd(mid, p->ffn, L.w2, p->ffn, L.b2, cur, d, s, d, nullptr, B, d, p->ffn, VY_ACT_NONE, p->dtype, stream);
      if (rc) return rc;
      rc = vy_layernorm_fwd(s, d, L.ln2_w, L.ln2_b, nxt, d, nullptr, nullptr, B, d, p->eps_ffn, p->dtype, stream);
      if (rc) return rc;
    }
    cur = nxt;
  }
  if (hidden_out && hidden_out != cur) {
    if (hipMemcpyAsync(hidden_out, cur, B * (int64_t)d * e, hipMemcpyDeviceToDevice, (hipStream_t)stream) != hipSuccess)
      VY_FAIL(VY_ERR_LAUNCH, "%s: copy of the hidden state failed", who);
  }
  if (logits) {
    int rc;
    if (lean) {   // LayerNorm(gelu(dense)) of the LM head: partial tile + finish
      rc = vy_dec_linear_res_ln(cur, d, p->head_wd, p->head_bd, nullptr, 0, p->head_ln_w, p->head_ln_b, p->eps_head, a, d,
                                part, B, d, d, VY_ACT_GELU_ERF, hst);
      if (rc) return rc;
    } else {
      rc = vy_linear_fwd(cur, d, p->head_wd, d, p->head_bd, nullptr, 0, s, d, nullptr, B, d, d, VY_ACT_GELU_ERF,
                         p->dtype, stream);
      if (rc) return rc;
      rc = vy_layernorm_fwd(s, d, p->head_ln_w, p->head_ln_b, a, d, nullptr, nullptr, B, d, p->eps_head, p->dtype, stream);
      if (rc) return rc;
    }
    rc = vy_linear_fwd(a, d, p->head_wv, d, p->head_bias, nullptr, 0, logits, ldv, nullptr, B, p->vocab, d,
                       VY_ACT_NONE, p->dtype, stream);
    if (rc) return rc;
  }
  return VY_OK;
}

extern "C" int64_t vy_gemma_ws_bytes(int32_t B, int32_t d, int32_t h, int32_t dh, int32_t ffn, int32_t dtype) {
  const int64_t e = esize(dtype);
  // normed input, q, attention output, two hidden buffers (x after attention / layer output), [gate|up], act
  return 4 * up(B * (int64_t)d * e) + 2 * up(B * (int64_t)h * dh * e) + up(2 * B * (int64_t)ffn * e) +
         up(B * (int64_t)ffn * e) + 4096;
}

extern "C" int vy_gemma_decoder_step(const vy_gemma_plan* p, const void* x, int64_t pos, void* logits, int64_t ldv,
                                     void* stream) {
  const char* who = "vy_gemma_decoder_step";
  if (!p || !x || !p->layers || !p->ws || !logits) VY_FAIL(VY_ERR_ARG, "%s: null plan/input/workspace/output", who);
  if (pos < 0) VY_FAIL(VY_ERR_ARG, "%s: negative position", who);
  if (p->ws_bytes < vy_gemma_ws_bytes(p->B, p->d, p->h, p->dh, p->ffn, p->dtype)) VY_FAIL(VY_ERR_ARG, "%s: workspace too small", who);
  const int64_t e = esize(p->dtype);
  const int B = p->B, d = p->d, h = p->h, hk = p->hk, dh = p->dh, ffn = p->ffn;
  char* w = (char*)p->ws;
  void* n = w; w += up(B * (int64_t)d * e);
  void* q = w; w += up(B * (int64_t)h * dh * e);
  void* ao = w; w += up(B * (int64_t)h * dh * e);
  void* x1 = w; w += up(B * (int64_t)d * e);
  void* hb[2];
  hb[0] = w; w += up(B * (int64_t)d * e);
  hb[1] = w; w += up(B * (int64_t)d * e);
  void* gu = w; w += up(2 * B * (int64_t)ffn * e);
  void* act = w;
  const float scale = 1.0f / sqrtf((float)dh);
  const void* cur = x;
  int rc;
  // Single-sequence bf16 decode (B <= 4) is a chain of matrix-vector products: the RMSNorm of each projection's
  // input is folded into the product (every wave redoes the row statistics from the chunks it reads anyway) and
  // the GeGLU into the gate/up product -- 6 launches per layer instead of 9 (VY_GEMMA_FUSED=0: the unfused chain).
  static const int fused_env = [] { const char* e = getenv("VY_GEMMA_FUSED"); return e ? atoi(e) : 1; }();
  const bool fused = fused_env && p->dtype == VY_BF16 && B <= 4 && d % 8 == 0 && ffn % 8 == 0 && ((int64_t)h * dh) % 8 == 0;
  // (folding the RMSNorm into the products as well -- VY_GEMMA_FUSED=2 -- measured SLOWER, 2.05 vs 1.76 ms per token:
  // every one of the N waves of a product redoes the row statistics and the normalisation of its input)
  const bool fold_norm = fused_env >= 2;
  // a plan whose weights already carry the norms' (1 + w) can only run on the chain that skips the RMSNorm launches: on
  // any other chain the factor would be applied twice and the tokens would be wrong without a word
  if ((p->flags & VY_GEMMA_PRESCALED) && !fused)
    VY_FAIL(VY_ERR_ARG, "%s: the plan's weights are pre-scaled by the RMSNorm weights, which needs the fused matrix-vector "
            "chain (bf16, B <= 4, d / ffn / h*dh multiples of 8, VY_GEMMA_FUSED != 0)", who);
  const bool prescaled = fused && (p->flags & VY_GEMMA_PRESCALED);
  static const int rope_env = [] { const char* e = getenv("VY_GEMMA_ROPE_FUSED"); return e ? atoi(e) : 1; }();
  const bool rope_fused = fused && rope_env && p->cos_tab && dh % 4 == 0 && (dh & (dh - 1)) == 0;
  if (g_gemma_lean < 0) { const char* e = getenv("VY_GEMMA_LEAN"); g_gemma_lean = e ? atoi(e) : 1; }
  const bool lean1 = g_gemma_lean && B == 1 && !fold_norm;
  for (int l = 0; l < p->num_layers; ++l) {
    const vy_gemma_layer& L = p->layers[l];
    void* kdst = (char*)L.kcache + pos * L.c_sl * e;
    void* vdst = (char*)L.vcache + pos * L.c_sl * e;
    void* nxt = hb[l & 1];
    if (fused && lean1) {
      // one sequence: the straight-line matrix-vector kernels of vy_decode.hip (norms folded when the plan's weights
      // are pre-scaled, rotary pairs swapped inside the QKV product); any unsupported shape -> the general chain below
      hipStream_t hs = (hipStream_t)stream;
      const void* qin = cur;
      if (!prescaled) {
        if ((rc = vy_rmsnorm_fwd(cur, d, L.ln_in, n, d, B, d, p->eps, 1.0f, p->dtype, stream))) return rc;
        qin = n;
      }
      rc = vy_dec_gemv1_qkv(qin, L.wqkv, L.bqkv, q, kdst, vdst, L.c_sh, h, hk, dh, rope_fused ? p->cos_tab : nullptr, p->sin_tab,
                            pos, d, prescaled, p->eps, hs);
      if (rc != VY_OK && rc != VY_ERR_UNSUPPORTED) return rc;   // only an unsupported shape falls through to the general chain
      if (rc == VY_OK) {
        if (p->cos_tab && !rope_fused &&
            (rc = vy_rope_qk(q, (int64_t)h * dh, dh, dh, h, kdst, L.c_sb, L.c_sh, L.c_sl, hk, p->cos_tab, p->sin_tab,
                             pos, B, 1, dh, p->dtype, hs))) return rc;
        if ((rc = vy_attn_decode_ex(q, (int64_t)h * dh, dh, L.kcache, L.c_sb, L.c_sh, L.c_sl, L.vcache, L.c_sb, L.c_sh, L.c_sl,
                                    ao, (int64_t)h * dh, B, h, hk, pos + 1, nullptr, dh, scale, p->dtype, stream))) return rc;
        if ((rc = vy_dec_gemv1(ao, L.wo, L.bo, cur, x1, d, h * dh, 0, 0.f, hs))) {
          if (rc != VY_ERR_UNSUPPORTED) return rc;
          if ((rc = vy_gemv_norm(ao, (int64_t)h * dh, L.wo, (int64_t)h * dh, L.bo, nullptr, 0.f, cur, d, x1, d, B, d,
                                 (int64_t)h * dh, stream))) return rc;
        }
        const void* gin = x1;
        if (!prescaled) {
          if ((rc = vy_rmsnorm_fwd(x1, d, L.ln_post, n, d, B, d, p->eps, 1.0f, p->dtype, stream))) return rc;
          gin = n;
        }
        if ((rc = vy_dec_gemv1_gated(gin, L.wgu, act, ffn, d, VY_ACT_GELU_TANH, prescaled, p->eps, hs))) {
          if (rc != VY_ERR_UNSUPPORTED) return rc;
          if ((rc = vy_gemv_gated(gin, d, L.wgu, d, prescaled ? VY_NORM_PRESCALED : nullptr, p->eps, act, ffn, B, ffn, d,
                                  VY_ACT_GELU_TANH, stream))) return rc;
        }
        if ((rc = vy_dec_gemv1(act, L.wdown, nullptr, x1, nxt, d, ffn, 0, 0.f, hs))) {
          if (rc != VY_ERR_UNSUPPORTED) return rc;
          if ((rc = vy_gemv_norm(act, ffn, L.wdown, ffn, nullptr, nullptr, 0.f, x1, d, nxt, d, B, d, ffn, stream))) return rc;
        }
        cur = nxt;
        continue;
      }
    }
    if (fused) {
      // prescaled: the weights carry the norms' (1 + w), the products scale themselves by the row's rsqrt(mean x^2):
      // no RMSNorm launch; rope_fused: rotary pairs swapped inside the QKV product's workgroups: no RoPE launch
      const void* qin = cur;
      const void* qnorm = prescaled ? VY_NORM_PRESCALED : (fold_norm ? L.ln_in : nullptr);
      if (!fold_norm && !prescaled) {
        if ((rc = vy_rmsnorm_fwd(cur, d, L.ln_in, n, d, B, d, p->eps, 1.0f, p->dtype, stream))) return rc;
        qin = n;
      }
      if ((rc = vy_gemv_qkv_norm(qin, d, L.wqkv, d, L.bqkv, qnorm, p->eps, q, (int64_t)h * dh, dh, kdst, L.c_sb, L.c_sh,
                                 L.c_sl, vdst, L.c_sb, L.c_sh, L.c_sl, B, d, h, hk, dh, rope_fused ? p->cos_tab : nullptr,
                                 p->sin_tab, pos, stream))) return rc;
      if (p->cos_tab && !rope_fused &&
          (rc = vy_rope_qk(q, (int64_t)h * dh, dh, dh, h, kdst, L.c_sb, L.c_sh, L.c_sl, hk, p->cos_tab, p->sin_tab,
                           pos, B, 1, dh, p->dtype, (hipStream_t)stream))) return rc;
      if ((rc = vy_attn_decode_ex(q, (int64_t)h * dh, dh, L.kcache, L.c_sb, L.c_sh, L.c_sl, L.vcache, L.c_sb, L.c_sh, L.c_sl,
                                  ao, (int64_t)h * dh, B, h, hk, pos + 1, nullptr, dh, scale, p->dtype, stream))) return rc;
      if ((rc = vy_gemv_norm(ao, (int64_t)h * dh, L.wo, (int64_t)h * dh, L.bo, nullptr, 0.f, cur, d, x1, d, B, d,
                             (int64_t)h * dh, stream))) return rc;
      const void* gin = x1;
      const void* gnorm = prescaled ? VY_NORM_PRESCALED : (fold_norm ? L.ln_post : nullptr);
      if (!fold_norm && !prescaled) {
        if ((rc = vy_rmsnorm_fwd(x1, d, L.ln_post, n, d, B, d, p->eps, 1.0f, p->dtype, stream))) return rc;
        gin = n;
      }
      if ((rc = vy_gemv_gated(gin, d, L.wgu, d, gnorm, p->eps, act, ffn, B, ffn, d, VY_ACT_GELU_TANH, stream))) return rc;
      if ((rc = vy_gemv_norm(act, ffn, L.wdown, ffn, nullptr, nullptr, 0.f, x1, d, nxt, d, B, d, ffn, stream))) return rc;
      cur = nxt;
      continue;
    }
    if ((rc = vy_rmsnorm_fwd(cur, d, L.ln_in, n, d, B, d, p->eps, 1.0f, p->dtype, stream))) return rc;
    if ((rc = vy_qkv_rope_fwd_ex(n, d, L.wqkv, d, L.bqkv, p->cos_tab, p->sin_tab, pos, nullptr, q, (int64_t)h * dh, dh, dh,
                                 kdst, L.c_sb, L.c_sh, L.c_sl, vdst, L.c_sb, L.c_sh, L.c_sl, B, 1, d, h, hk, dh, p->dtype,
                                 stream))) return rc;
    if ((rc = vy_attn_decode_ex(q, (int64_t)h * dh, dh, L.kcache, L.c_sb, L.c_sh, L.c_sl, L.vcache, L.c_sb, L.c_sh, L.c_sl,
                                ao, (int64_t)h * dh, B, h, hk, pos + 1, nullptr, dh, scale, p->dtype, stream))) return rc;
    if ((rc = vy_linear_fwd(ao, (int64_t)h * dh, L.wo, (int64_t)h * dh, L.bo, cur, d, x1, d, nullptr, B, d, (int64_t)h * dh,
                            VY_ACT_NONE, p->dtype, stream))) return rc;
    if ((rc = vy_rmsnorm_fwd(x1, d, L.ln_post, n, d, B, d, p->eps, 1.0f, p->dtype, stream))) return rc;
    if ((rc = vy_linear_fwd(n, d, L.wgu, d, nullptr, nullptr, 0, gu, 2 * (int64_t)ffn, nullptr, B, 2 * (int64_t)ffn, d,
                            VY_ACT_NONE, p->dtype, stream))) return rc;
    if ((rc = vy_gated_act_fwd(gu, 2 * (int64_t)ffn, act, ffn, B, ffn, VY_ACT_GELU_TANH, p->dtype, stream))) return rc;
    if ((rc = vy_linear_fwd(act, ffn, L.wdown, ffn, nullptr, x1, d, nxt, d, nullptr, B, d, ffn, VY_ACT_NONE, p->dtype,
                            stream))) return rc;
    cur = nxt;
  }
  if (fused && fold_norm)   // final norm folded into the vocabulary product
    return vy_gemv_norm(cur, d, p->head_w, d, nullptr, p->norm_w, p->eps, nullptr, 0, logits, ldv, B, p->vocab, d, stream);
  if ((rc = vy_rmsnorm_fwd(cur, d, p->norm_w, n, d, B, d, p->eps, 1.0f, p->dtype, stream))) return rc;
  return vy_linear_fwd(n, d, p->head_w, d, nullptr, nullptr, 0, logits, ldv, nullptr, B, p->vocab, d, VY_ACT_NONE,
                       p->dtype, stream);
}
