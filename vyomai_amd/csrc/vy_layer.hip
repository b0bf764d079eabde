// One post-LN layer of the text and vision models without gradients (host code): the seven launches of vy_text_layer_fwd behind one
// call.  A few short texts keep the GPU busy for about 50 us per layer, and enqueueing the launches one by one from Python took four
// times that.
#include "vy_common.h"

extern "C" int64_t vy_text_layer_ws_bytes(int64_t B, int64_t L, int32_t h, int32_t dh, int32_t ffn, int dtype) {
  const int64_t d = (int64_t)h * dh, wide = ffn > 2 * d ? ffn : 2 * d;   // [q | heads] and, once they are used up, the inner rows
  return B * L * (wide + 2 * d) * (dtype == VY_BF16 ? 2 : 4);
}

extern "C" int vy_text_layer_fwd(const vy_text_layer* l, const void* x, void* y, int64_t B, int64_t L, void* ws, int64_t ws_bytes,
                                 void* stream) {
  const char* who = "vy_text_layer_fwd";
  if (!l || !x || !y || !ws || B <= 0 || L <= 0) VY_FAIL(VY_ERR_ARG, "%s: null operand or empty batch", who);
  if (l->dtype != VY_BF16 && l->dtype != VY_F32) VY_FAIL(VY_ERR_ARG, "%s: bad dtype %d", who, l->dtype);
  if (l->h <= 0 || l->hk <= 0 || l->dh <= 0 || l->ffn <= 0 || (l->mask_kind & VY_MASK_ADDITIVE))
    VY_FAIL(VY_ERR_ARG, "%s: bad sizes or mask", who);
  if (ws_bytes < vy_text_layer_ws_bytes(B, L, l->h, l->dh, l->ffn, l->dtype)) VY_FAIL(VY_ERR_ARG, "%s: workspace too small", who);
  const int64_t d = (int64_t)l->h * l->dh, M = B * L, e = l->dtype == VY_BF16 ? 2 : 4, wide = l->ffn > 2 * d ? l->ffn : 2 * d;
  char* q = (char*)ws;
  char* o = q + M * d * e;
  char* inner = q;                       // over q and the heads
  char* sum = q + M * wide * e;          // ahead of both norms
  char* a = sum + M * d * e;
  const float scale = (float)(1.0 / sqrt((double)l->dh));
  int rc;
  if ((rc = vy_qkv_rope_fwd(x, d, l->wqkv, d, l->bqkv, l->cos_tab, l->sin_tab, l->pos0, q, L * d, L * l->dh, l->dh, l->k_new, l->kn_sb,
                            l->kn_sh, l->kn_sl, l->v_new, l->vn_sb, l->vn_sh, l->vn_sl, B, L, d, l->h, l->hk, l->dh, l->dtype, stream)))
    return rc;
  if (L == 1 && l->mask_kind == VY_MASK_NONE)
    rc = vy_attn_decode(q, d, l->dh, l->k, l->k_sb, l->k_sh, l->k_sl, l->v, l->v_sb, l->v_sh, l->v_sl, o, d, B, l->h, l->hk, l->S, l->dh,
                        scale, l->dtype, stream);
  else
    rc = vy_attn_fwd(q, L * d, L * l->dh, l->dh, l->k, l->k_sb, l->k_sh, l->k_sl, l->v, l->v_sb, l->v_sh, l->v_sl, o, L * d, d, nullptr,
                     l->mask_kind, l->start_pos, l->keypad, l->kp_sb, nullptr, 0, 0, B, l->h, l->hk, L, l->S, l->dh, scale, l->dtype,
                     stream);
  if (rc) return rc;
  if ((rc = vy_linear_fwd(o, d, l->wo, d, l->bo, x, d, sum, d, nullptr, M, d, d, VY_ACT_NONE, l->dtype, stream))) return rc;
  if ((rc = vy_layernorm_fwd(sum, d, l->ln1_w, l->ln1_b, a, d, nullptr, nullptr, M, d, l->eps1, l->dtype, stream))) return rc;
  if ((rc = vy_linear_fwd(a, d, l->w1, d, l->b1, nullptr, 0, inner, l->ffn, nullptr, M, l->ffn, d, l->act, l->dtype, stream))) return rc;
  if ((rc = vy_linear_fwd(inner, l->ffn, l->w2, l->ffn, l->b2, x, d, sum, d, nullptr, M, d, l->ffn, VY_ACT_NONE, l->dtype, stream))) return rc;
  return vy_layernorm_fwd(sum, d, l->ln2_w, l->ln2_b, y, d, nullptr, nullptr, M, d, l->eps2, l->dtype, stream);
}
