"""The three fused groups of a VyomAI layer, forward and backward, on the HIP kernels:

  self_attention_block      QKV+RoPE -> flash attention -> out-proj + residual -> LayerNorm
  linear_residual_layernorm AttentionSelfOutput on its own
  ffn_block                 GEMM+GELU -> GEMM + residual -> LayerNorm

The grouping follows the reference author's own fused ops (Examples/vyom-ai-decoder-fused.ipynb
cells 2-7: LinearRms, FFNGeLU, ScaledDotProductAttention, RotaryEmbeddingFunction).  Inference
calls go straight to the forward kernels; when gradients are required the same kernels run inside
torch.autograd.Function wrappers whose backward is the vy_*_bwd / dgrad / wgrad entry points.
PyTorch autograd is only the tape; no PyTorch math runs in either direction.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import _lib, ops
from ._lib import VyomHipError
from .layers.attention import AttentionSelfOutput, _param, _shadow as _param_shadow
from .layers.ffn import FeedForward
from .layers.mask import AttnMask
from .layers.positional_embeddings import resolve_freqs


_shadow = _param_shadow


def _wants_grad(*ts) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in ts)


# ------------------------------------------------------------------------------------------
# forward-only (inference) paths
# ------------------------------------------------------------------------------------------


def _drop_args(p_drop: float, training: bool):
    """(p, seed, offset) of one dropout call when the module is in train() with p > 0 (nn.Dropout's
    condition in the reference: layers/attention.py:70, layers/ffn.py:38), else None."""
    if not training or p_drop <= 0.0:
        return None
    from .rng import next_dropout
    return next_dropout(p_drop)


def linear_residual_layernorm(x, residual, w, b, ln_w, ln_b, eps, p_drop: float = 0.0, training: bool = False):
    """LN(dropout(x W^T + b) + residual): AttentionSelfOutput (reference layers/attention.py:69-72)."""
    drop = _drop_args(p_drop, training)
    if _wants_grad(x, residual, w, b, ln_w, ln_b):
        from .autograd_train import LinearResidualLayerNormFn
        return LinearResidualLayerNormFn.apply(x, residual, w, b, ln_w, ln_b, eps, drop)
    dt = x.dtype
    s = ops.linear(x, _shadow(w, dt), _shadow(b, dt), residual=residual, dropout=drop)
    y, _, _ = ops.layernorm(s, _shadow(ln_w, dt), _shadow(ln_b, dt), eps)
    return y


def ffn_block(x, residual, w1, b1, w2, b2, ln_w, ln_b, eps, act, p_drop: float = 0.0, training: bool = False):
    """LN(dropout(act(x W1^T + b1) W2^T + b2) + residual): FeedForward (reference layers/ffn.py:32-40)."""
    drop = _drop_args(p_drop, training)
    if _wants_grad(x, residual, w1, b1, w2, b2, ln_w, ln_b):
        from .autograd_train import FfnBlockFn
        return FfnBlockFn.apply(x, residual, w1, b1, w2, b2, ln_w, ln_b, eps, act, drop)
    dt = x.dtype
    hmid = ops.linear(x, _shadow(w1, dt), _shadow(b1, dt), act=act)
    s = ops.linear(hmid, _shadow(w2, dt), _shadow(b2, dt), residual=residual, dropout=drop)
    y, _, _ = ops.layernorm(s, _shadow(ln_w, dt), _shadow(ln_b, dt), eps)
    return y


def _mask_args(mask, B, L, S, device):
    """-> dict(causal, start_pos, keypad, addmask) for ops.attention."""
    if mask is None:
        return dict(causal=False, start_pos=0, keypad=None, addmask=None)
    if isinstance(mask, AttnMask):
        kp = mask.keypad
        if kp is not None:
            if kp.shape[-1] < S:
                raise ValueError(f"attention mask covers {kp.shape[-1]} keys, attention sees {S}")
            kp = kp[:, :S]
            if kp.device != device:
                kp = kp.to(device)
            if not kp.is_contiguous() and kp.stride(1) != 1:
                kp = kp.contiguous()
        return dict(causal=mask.causal, start_pos=mask.start_pos, keypad=kp, addmask=None)
    # dense additive float mask, the reference's interface: (B|1, 1, L|1, S)
    if mask.dim() != 4 or mask.shape[-1] != S:
        raise ValueError(f"additive attention_mask must be (B,1,L,S) with S={S}, got {tuple(mask.shape)}")
    am = mask.to(device=device, dtype=torch.float32)
    if am.stride(3) != 1:
        am = am.contiguous()
    return dict(causal=False, start_pos=0, keypad=None, addmask=am)


def self_attention_block(mod, x, attention_mask, freqs, cache, cache_index, start_pos):
    """mod: a vyomai_amd.layers.attention._SelfAttentionBase.  Returns LN(out(attn(x)) + x)."""
    B, L, _ = x.shape
    h, hk, dh = mod.num_attention_heads, mod.num_key_value_heads, mod.head_dim
    dt, dev = x.dtype, x.device
    w, b = mod._packed()
    aso = mod.out
    train = _wants_grad(x, w, b, aso.dense.weight)
    if train:
        if cache is not None:
            raise VyomHipError("KV caching is an inference feature; call under torch.no_grad()")
        from .autograd_train import SelfAttentionFn
        o = SelfAttentionFn.apply(x, mod, attention_mask, freqs, start_pos, *mod._params())
        return linear_residual_layernorm(o, x, aso.dense.weight, aso.dense.bias, aso.layernorm.weight,
                                         aso.layernorm.bias, aso.layernorm.eps, aso.dropout.p, aso.training)
    cos, sin, pos0 = resolve_freqs(freqs, dev)
    q = torch.empty((B, h, L, dh), dtype=dt, device=dev)
    if cache is not None:
        if cache_index is None:
            kw, vw = cache.reserve(B, hk, L, dh, start_pos, dt, dev)
        else:
            kw, vw = cache.reserve(cache_index, B, hk, L, dh, start_pos, dt, dev)
    else:
        kw = torch.empty((B, hk, L, dh), dtype=dt, device=dev)
        vw = torch.empty_like(kw)
    sw, sb = mod._packed_shadow(dt, (w, b))
    ops.qkv_rope(x, sw, sb, h, hk, dh, cos, sin, pos0, q, kw, vw)
    if cache is not None:
        k_all, v_all = cache.commit() if cache_index is None else cache.commit(cache_index)
    else:
        k_all, v_all = kw, vw
    S = k_all.shape[2]
    if L == 1 and attention_mask is None:
        o = ops.attention_decode(q, k_all, v_all, S)
    else:
        o = ops.attention(q, k_all, v_all, **_mask_args(attention_mask, B, L, S, dev))
    return linear_residual_layernorm(o, x, aso.dense.weight, aso.dense.bias, aso.layernorm.weight,
                                     aso.layernorm.bias, aso.layernorm.eps, aso.dropout.p, aso.training)


_GLOBAL_HOOKS = (torch.nn.modules.module._global_forward_hooks, torch.nn.modules.module._global_forward_pre_hooks)
_GLOBAL_BACKWARD_HOOKS = (torch.nn.modules.module._global_backward_hooks, torch.nn.modules.module._global_backward_pre_hooks)


def _plain_layer(att, ff, x, mask) -> bool:
    """May a post-LN layer be one native call?  Not with a module of another class, with a hook or with a forward of its own, active dropout,
    a dense mask, rows that are not contiguous: the modules are then to be called one by one."""
    if type(ff) is not FeedForward or "_whole_layer" not in type(att).__dict__ or not (mask is None or isinstance(mask, AttnMask)):
        return False
    aso = att._modules.get("out")
    if type(aso) is not AttentionSelfOutput or _GLOBAL_HOOKS[0] or _GLOBAL_HOOKS[1]:
        return False
    for d in (att.__dict__, aso.__dict__, ff.__dict__):
        if d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d:
            return False
    if type(x) is not torch.Tensor or not x.is_cuda or x.dim() != 3 or not x.is_contiguous() or ops._Lanes.active:
        return False
    if (aso.training and aso._modules["dropout"].p > 0.0) or (ff.training and ff._modules["dropout"].p > 0.0):
        return False
    return (x.dtype is torch.bfloat16 or x.dtype is torch.float32) and x.shape[2] == att.num_attention_heads * att.head_dim and 0 not in x.shape


def _layer_params(att, ff):
    """Weights and biases of the output projection, its norm, the two projections of the feed-forward and its norm."""
    aso, f = att._modules["out"]._modules, ff._modules
    return [_param(m, n) for m in (aso["dense"], aso["layernorm"], f["intermediate"], f["out"], f["layernorm"]) for n in ("weight", "bias")]


def _fits(keep, x, att, inner) -> bool:
    """keep: [Wqkv, bqkv, *_layer_params] in the compute type."""
    dev, d = x.device, x.shape[2]
    for t in keep:
        if t is not None and (t.device != dev or not t.is_contiguous()):
            return False
    return keep[0].shape == (d + 2 * att.num_key_value_heads * att.head_dim, d) and keep[2].shape == (d, d) and keep[6].shape == (inner, d) \
        and keep[8].shape == (d, inner)


def layer_forward(att, ff, x, mask, freqs, cache=None, start_pos: int = 0):
    """ff(att(x), x) of one post-LN layer without gradients as ONE native call (vy_text_layer_fwd), the same launches in the same order:
    a layer of a few short texts is 50 us of GPU work, and four times that in Python.  None: the modules are to be called one by one
    (_plain_layer)."""
    if torch.is_grad_enabled() or not _plain_layer(att, ff, x, mask):
        return None
    dt, dev = x.dtype, x.device
    B, L, d = x.shape
    h, hk, dh = att.num_attention_heads, att.num_key_value_heads, att.head_dim
    keep = [*att._packed_shadow(dt, None, att._params()), *[_shadow(p, dt) for p in _layer_params(att, ff)]]
    inner = keep[6].shape[0]
    if not _fits(keep, x, att, inner):
        return None
    cos, sin, pos0 = resolve_freqs(freqs, dev)
    kv = None
    if cache is None:
        kv = torch.empty((2, B, hk, L, dh), dtype=dt, device=dev)
        k = kv.data_ptr()
        v, S = k + kv.stride(0) * kv.element_size(), L
        k_new, v_new, strides = k, v, (hk * L * dh, L * dh, dh) * 4
    else:
        kn, vn = cache.reserve(att.layer_idx, B, hk, L, dh, start_pos, dt, dev)
        kc, vc = cache.commit(att.layer_idx)
        assert kn.stride(3) == 1 and vn.stride(3) == 1
        k_new, v_new, k, v, S = kn.data_ptr(), vn.data_ptr(), kc.data_ptr(), vc.data_ptr(), kc.shape[2]
        strides = (*kn.stride()[:3], *vn.stride()[:3], *kc.stride()[:3], *vc.stride()[:3])
    m = _mask_args(mask, B, L, S, dev)
    kp = m["keypad"]
    kind = (_lib.MASK_CAUSAL if m["causal"] else 0) | (_lib.MASK_KEYPAD if kp is not None else 0)
    if kp is not None:
        assert kp.dtype == torch.uint8 and kp.shape == (B, S) and kp.stride(1) == 1
    desc = _lib.VyTextLayer(h, hk, dh, inner, ff.act, kind, _lib.dtype_code(dt), att._modules["out"]._modules["layernorm"].eps,
                            ff._modules["layernorm"].eps, *(None if t is None else t.data_ptr() for t in keep), ops._ptr(cos), ops._ptr(sin),
                            pos0, k_new, v_new, *strides[:6], k, v, *strides[6:], S, m["start_pos"], ops._ptr(kp),
                            kp.stride(0) if kp is not None else 0)
    return ops.text_layer(desc, x)


def _backward_hooks(att, ff) -> bool:
    """Is there a hook on the gradients of the two modules' outputs or inputs?"""
    if _GLOBAL_BACKWARD_HOOKS[0] or _GLOBAL_BACKWARD_HOOKS[1]:
        return True
    return any(d["_backward_hooks"] or d["_backward_pre_hooks"] for d in (att.__dict__, ff.__dict__))


def layer_train(att, ff, x, mask, freqs):
    """The same with gradients: one autograd function, whose forward and backward are a native call each (vy_text_layer_train_fwd,
    vy_text_layer_bwd), where every gradient goes straight into the trainer's arena.  None: as above, and with a backward hook, which only
    a call of its module sees."""
    if not torch.is_grad_enabled() or not _plain_layer(att, ff, x, mask) or _backward_hooks(att, ff):
        return None
    from .autograd_train import TextLayerFn
    members = att._params()
    params = _layer_params(att, ff) + members
    for p in params:
        if p is not None and not (getattr(p, "_vy_direct", False) and p.requires_grad and p.grad is not None):
            return None
    if params[1] is None or params[3] is None or params[7] is None or params[9] is None:   # (biases of norms and projections)
        return None
    B, L, _ = x.shape
    causal, kp, start = False, None, 0
    if mask is not None:
        causal, kp, start = mask.causal, mask.keypad, mask.start_pos
        if kp is not None:
            if not kp.is_cuda or kp.dtype is not torch.uint8 or kp.dim() != 2 or kp.shape[0] != B or kp.shape[1] < L:
                return None
            kp = kp[:, :L].contiguous() if kp.shape[1] != L else kp
            if kp.stride(1) != 1:
                return None
    dt = x.dtype
    keep = [*att._packed_shadow(dt, None, members), *[_shadow(p, dt) for p in params[:10]]]
    if not _fits(keep, x, att, keep[6].shape[0]):
        return None
    return TextLayerFn.apply(x, kp, att, ff, keep, causal, start, resolve_freqs(freqs, x.device), *params)


def _split(x2: torch.Tensor, heads: int, dh: int) -> torch.Tensor:
    """(B, L, heads*dh) projection output -> (B, heads, L, dh) strided view (no copy)."""
    B, L, _ = x2.shape
    return x2.view(B, L, heads, dh).permute(0, 2, 1, 3)


def cross_attention_block(mod, x, enc, enc_mask, use_cache: bool):
    """mod: layers.attention._CrossAttentionBase.  Returns LN(out(attn(q(x), k(enc), v(enc))) + x).
    Reference layers/attention.py:410-474 / 512-573."""
    B, L, _ = x.shape
    h, hk, dh = mod.num_attention_heads, mod.num_key_value_heads, mod.head_dim
    dt, dev = x.dtype, x.device
    aso = mod.out
    wq, bq = mod.query.weight, mod.query.bias
    wk, bk = mod.key.weight, mod.key.bias
    wv, bv = mod.value.weight, mod.value.bias
    if _wants_grad(x, enc, wq, wk, wv, aso.dense.weight):
        if use_cache:
            raise VyomHipError("KV caching is an inference feature; call under torch.no_grad()")
        from .autograd_train import CrossAttentionFn
        o = CrossAttentionFn.apply(x, enc, mod, enc_mask, wq, bq, wk, bk, wv, bv)
        return linear_residual_layernorm(o, x, aso.dense.weight, aso.dense.bias, aso.layernorm.weight,
                                         aso.layernorm.bias, aso.layernorm.eps, aso.dropout.p, aso.training)

    def project():
        k2 = ops.linear(enc, _shadow(wk, dt), _shadow(bk, dt))
        v2 = ops.linear(enc, _shadow(wv, dt), _shadow(bv, dt))
        return _split(k2, hk, dh), _split(v2, hk, dh)

    q = _split(ops.linear(x, _shadow(wq, dt), _shadow(bq, dt)), h, dh)
    if use_cache:
        cache = getattr(mod, "cache", None)
        if cache is None:
            raise ValueError("use_cache is True please enable model._setup_cache() to use kv-cache")
        if len(cache) == 0:   # first step: the encoder states are the same for the whole generation
            k, v = cache.update(*project())
        else:
            k, v = cache.get()
    else:
        k, v = project()
    S = k.shape[2]
    o = ops.attention(q, k, v, **_mask_args(enc_mask, B, L, S, dev))
    return linear_residual_layernorm(o, x, aso.dense.weight, aso.dense.bias, aso.layernorm.weight,
                                     aso.layernorm.bias, aso.layernorm.eps, aso.dropout.p, aso.training)

