// One post-LN layer of the text and vision models (host code): the seven launches of vy_text_layer_fwd, and the seven and nine of a
// layer in training, behind one call each.  A few short texts keep the GPU busy for about 50 us per layer, and enqueueing the launches one
// by one from Python took four times that; a training step of 5 x 333 tokens, 12 layers, is 4.5 ms of kernels, and its layers one operation at
// a time took the host 6.5 and more.
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

static int kept_layer(const char* who, const vy_text_layer* l, const vy_text_layer_kept* t, int64_t B, int64_t L) {
  if (!l || !t || B <= 0 || L <= 0) VY_FAIL(VY_ERR_ARG, "%s: null operand or empty batch", who);
  if (l->dtype != VY_BF16 && l->dtype != VY_F32) VY_FAIL(VY_ERR_ARG, "%s: bad dtype %d", who, l->dtype);
  if (l->h <= 0 || l->hk <= 0 || l->dh <= 0 || l->ffn <= 0 || (l->mask_kind & VY_MASK_ADDITIVE)) VY_FAIL(VY_ERR_ARG, "%s: bad sizes or mask", who);
  if (l->k != l->k_new || l->v != l->v_new || l->S != L) VY_FAIL(VY_ERR_ARG, "%s: keys and values of this call alone", who);
  if (!t->q || !t->o || !t->s1 || !t->a || !t->deriv || !t->inner || !t->s2 || !t->lse || !t->mean1 || !t->rstd1 || !t->mean2 || !t->rstd2)
    VY_FAIL(VY_ERR_ARG, "%s: null tensor", who);
  return VY_OK;
}

extern "C" int vy_text_layer_train_fwd(const vy_text_layer* l, const vy_text_layer_kept* t, const void* x, void* y, int64_t B, int64_t L,
                                       void* stream) {
  const char* who = "vy_text_layer_train_fwd";
  if (int rc = kept_layer(who, l, t, B, L)) return rc;
  if (!x || !y) VY_FAIL(VY_ERR_ARG, "%s: null operand", who);
  const int64_t d = (int64_t)l->h * l->dh, M = B * L;
  const float scale = (float)(1.0 / sqrt((double)l->dh));
  int rc;
  if ((rc = vy_qkv_rope_fwd(x, d, l->wqkv, d, l->bqkv, l->cos_tab, l->sin_tab, l->pos0, t->q, L * d, L * l->dh, l->dh, l->k_new, l->kn_sb,
                            l->kn_sh, l->kn_sl, l->v_new, l->vn_sb, l->vn_sh, l->vn_sl, B, L, d, l->h, l->hk, l->dh, l->dtype, stream)))
    return rc;
  if ((rc = vy_attn_fwd(t->q, L * d, L * l->dh, l->dh, l->k, l->k_sb, l->k_sh, l->k_sl, l->v, l->v_sb, l->v_sh, l->v_sl, t->o, L * d, d,
                        t->lse, l->mask_kind, l->start_pos, l->keypad, l->kp_sb, nullptr, 0, 0, B, l->h, l->hk, L, l->S, l->dh, scale,
                        l->dtype, stream)))
    return rc;
  if ((rc = vy_linear_fwd(t->o, d, l->wo, d, l->bo, x, d, t->s1, d, nullptr, M, d, d, VY_ACT_NONE, l->dtype, stream))) return rc;
  if ((rc = vy_layernorm_fwd(t->s1, d, l->ln1_w, l->ln1_b, t->a, d, t->mean1, t->rstd1, M, d, l->eps1, l->dtype, stream))) return rc;
  // (the derivative is kept, not the pre-activation: the backward product's epilogue multiplies by it)
  if ((rc = vy_linear_fwd(t->a, d, l->w1, d, l->b1, nullptr, 0, t->inner, l->ffn, t->deriv, M, l->ffn, d, l->act | VY_ACT_SAVE_DERIV,
                          l->dtype, stream)))
    return rc;
  if ((rc = vy_linear_fwd(t->inner, l->ffn, l->w2, l->ffn, l->b2, x, d, t->s2, d, nullptr, M, d, l->ffn, VY_ACT_NONE, l->dtype, stream))) return rc;
  return vy_layernorm_fwd(t->s2, d, l->ln2_w, l->ln2_b, y, d, t->mean2, t->rstd2, M, d, l->eps2, l->dtype, stream);
}

extern "C" int vy_text_layer_bwd(const vy_text_layer* l, const vy_text_layer_kept* t, const vy_text_layer_grads* g, const void* dy, void* dx,
                                 int64_t B, int64_t L, void* stream) {
  const char* who = "vy_text_layer_bwd";
  if (int rc = kept_layer(who, l, t, B, L)) return rc;
  if (!g || !dy || !dx || !g->wt_qkv || !g->wt_o || !g->wt_1 || !g->wt_2 || (!g->ln_ws1 && (!g->dln1_w || !g->dln1_b || !g->dln2_w || !g->dln2_b)) ||
      !g->ds2 || !g->dpre || !g->da || !g->ds1 || !g->dheads || !g->dqkv || !g->ln_ws || !g->delta)
    VY_FAIL(VY_ERR_ARG, "%s: null tensor", who);
  const int64_t d = (int64_t)l->h * l->dh, kv = (int64_t)l->hk * l->dh, W = d + 2 * kv, M = B * L, e = l->dtype == VY_BF16 ? 2 : 4, dh = l->dh;
  const float scale = (float)(1.0 / sqrt((double)l->dh));
  char *dq = (char*)g->dqkv, *dk = dq + d * e, *dv = dk + kv * e;
  const bool later = g->ln_ws1 != nullptr;   // the norms' column sums, with other layers'
  float *ln1_w = later ? nullptr : g->dln1_w, *ln1_b = later ? nullptr : g->dln1_b, *ln2_w = later ? nullptr : g->dln2_w, *ln2_b = later ? nullptr : g->dln2_b;
  int rc;
  if ((rc = vy_layernorm_bwd(dy, d, t->s2, d, l->ln2_w, t->mean2, t->rstd2, g->ds2, d, ln2_w, ln2_b, 1.f, g->ln_ws, M, d, l->dtype, stream))) return rc;
  if ((rc = vy_linear_dgrad(g->ds2, d, g->wt_2, g->ld_2, t->deriv, l->ffn, l->act | VY_ACT_SAVE_DERIV, nullptr, 0, nullptr, 0, g->dpre, l->ffn, M, d,
                            l->ffn, l->dtype, stream)))
    return rc;
  if ((rc = vy_linear_dgrad(g->dpre, l->ffn, g->wt_1, g->ld_1, nullptr, 0, VY_ACT_NONE, nullptr, 0, nullptr, 0, g->da, d, M, l->ffn, d, l->dtype, stream)))
    return rc;
  if ((rc = vy_layernorm_bwd(g->da, d, t->s1, d, l->ln1_w, t->mean1, t->rstd1, g->ds1, d, ln1_w, ln1_b, 1.f, later ? g->ln_ws1 : g->ln_ws, M, d, l->dtype, stream)))
    return rc;
  if ((rc = vy_linear_dgrad(g->ds1, d, g->wt_o, g->ld_o, nullptr, 0, VY_ACT_NONE, nullptr, 0, nullptr, 0, g->dheads, d, M, d, d, l->dtype, stream))) return rc;
  if ((rc = vy_attn_bwd(t->q, L * d, L * dh, dh, l->k, l->k_sb, l->k_sh, l->k_sl, l->v, l->v_sb, l->v_sh, l->v_sl, t->o, g->dheads, L * d, d, t->lse,
                        g->delta, dq, L * W, dh, W, dk, L * W, dh, W, dv, L * W, dh, W, l->mask_kind, l->start_pos, l->keypad, l->kp_sb, l->cos_tab,
                        l->sin_tab, l->pos0, B, l->h, l->hk, L, l->S, l->dh, scale, l->dtype, stream)))
    return rc;
  // the layer input's other two gradients, of the residual paths, are added in this product's epilogue
  return vy_linear_dgrad(g->dqkv, W, g->wt_qkv, g->ld_qkv, nullptr, 0, VY_ACT_NONE, g->ds2, d, g->ds1, d, dx, d, M, W, d, l->dtype, stream);
}
