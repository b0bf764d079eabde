"""Case definitions shared by the golden generator (reference side) and the tests
(oracle / HIP side): configs, masks and sub-sampling.  numpy only."""
from __future__ import annotations

import copy
from dataclasses import dataclass
from typing import Optional, Tuple

import numpy as np

FMIN = float(np.finfo(np.float32).min)

# (batch, seq) per module-level tag; 'wide' uses L=17 (not a tile multiple, as in the
# reference tests' 17-token rows)
MODULE_BL = {"micro": (2, 16), "wide": (2, 17)}


@dataclass
class TextCfg:
    hidden_size: int = 768
    num_attention_heads: int = 12
    max_position_embeddings: int = 514
    num_hidden_layers: int = 4
    vocab_size: int = 50265
    hidden_dropout_prob: float = 0.1
    initializer_range: float = 0.02
    intermediate_size: int = 3072
    layer_norm_eps: float = 1e-05
    hidden_act: str = "gelu"


@dataclass
class GqaCfg(TextCfg):
    num_key_value_heads: int = 4


from vyomai_amd.shapes import VitCfg  # noqa: E402


def test_cfg() -> TextCfg:
    """The Config of the reference's tests (tests/test_decoder.py:12-23)."""
    return TextCfg()


test_cfg.__test__ = False  # not a pytest test


def micro_cfg() -> GqaCfg:
    return GqaCfg(hidden_size=64, num_attention_heads=4, max_position_embeddings=64,
                  num_hidden_layers=1, vocab_size=97, num_key_value_heads=2)


def wide_cfg() -> GqaCfg:
    return GqaCfg(num_hidden_layers=1, num_key_value_heads=4)


def vit_cfg() -> VitCfg:
    return VitCfg()


def with_kv(cfg, attn_type: Optional[str]):
    """Config for a vanilla / gqa model.  The reference's StaticCacheOne reads
    config.num_key_value_heads even for vanilla attention (layers/kv_cache.py:275-282), so
    vanilla configs must not carry the attribute."""
    base = {k: getattr(cfg, k) for k in TextCfg.__dataclass_fields__ if hasattr(cfg, k)}
    if attn_type == "gqa":
        return GqaCfg(**base, num_key_value_heads=getattr(cfg, "num_key_value_heads", 4))
    return TextCfg(**base)


def one_layer(cfg, gqa: bool):
    c = with_kv(cfg, "gqa" if gqa else None)
    c.num_hidden_layers = 1
    return c


def keypad(batch: int, seq: int) -> np.ndarray:
    """(B, L) int64 0/1 right-padding mask; row b keeps seq - (3*b + 2) % (seq//2) tokens, row 0 full."""
    m = np.ones((batch, seq), dtype=np.int64)
    for b in range(1, batch):
        keep = seq - ((3 * b + 2) % max(seq // 2, 1)) - 1
        m[b, keep:] = 0
    return m


def causal_additive(batch: int, seq: int, start_pos: int, keypad_full: Optional[np.ndarray]) -> np.ndarray:
    """Dense (B,1,L,start+L) additive fp32 mask as DecoderModel builds it
    (reference models/decoder.py:360-362, 376-419), restated in numpy."""
    total = seq + start_pos
    am = np.ones((batch, total), dtype=np.float32) if keypad_full is None else keypad_full.astype(np.float32)
    i = np.arange(seq)[:, None]
    j = np.arange(total)[None, :]
    causal = (j <= i + start_pos).astype(np.float32)
    ext = causal[None, None] * am[:, None, None, :]
    return ((1.0 - ext) * FMIN).astype(np.float32)


def reference_test_inputs():
    """Token rows / masks hard-coded in the reference tests (tests/test_decoder.py:28-46)."""
    ids = np.array([
        [0, 2387, 766, 16, 181, 967, 46035, 2, 1, 1, 1, 1, 1, 1, 1, 1, 1],
        [0, 12196, 16, 110, 766, 2, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1],
        [0, 37111, 1137, 162, 110, 766, 2, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1]], dtype=np.int64)
    am = np.array([
        [1, 1, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0, 0, 0, 0, 0],
        [1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0],
        [1, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0]], dtype=np.int64)
    return ids, am


def sub(y):
    """Sub-sample a (B, L, D) activation: every 8th position (offset 1) x every 4th feature."""
    return y[:, 1::8, ::4]


def sub2(g):
    """Sub-sample a 2-D gradient: rows ::7, cols ::5."""
    return g[::7, ::5]


from vyomai_amd.shapes import (attn_shapes, aso_shapes, ffn_shapes, layer_shapes, lm_head_shapes,  # noqa: E402,F401
                               text_model_shapes, s2s_layer_shapes, s2s_model_shapes, vit_shapes, SIGLIP, GEMMA,
                               siglip_layer_shapes, gemma_layer_shapes)


# reduced vocabulary of the PaliGemma model golden (true widths, 2 + 2 layers); the image placeholder id
PG_SMALL_VOCAB, PG_IMAGE_TOKEN = 4099, 4000


# ---- sampling processors / speculative decoding ----------------------------------

def sampling_logits() -> np.ndarray:
    """(3, 1531) fp32 logits: row 0 flat-ish, row 1 peaked, row 2 wide."""
    from vyomai_amd import recipe
    x = recipe.uniform("samp.logits", (3, 1531))
    return (x * np.array([[1.5], [9.0], [4.0]], dtype=np.float32)).astype(np.float32)


# name -> (reference class, constructor args)
PROCESSORS = {
    "greedy": ("GreedyProcessor", (1,)),
    "multinomial_t07": ("MultinomialProcessor", (0.7,)),
    "topk50_t08": ("TopKProcessor", (0.8, 50)),
    "topk_all": ("TopKProcessor", (1.0, 5000)),
    "nucleus09_t02": ("NucleusProcessor", (0.2, 0.9)),
    "nucleus05_t1": ("NucleusProcessor", (1.0, 0.5)),
    "topk40_nucleus08_t09": ("TopKNucleusProcessor", (0.9, 40, 0.8)),
}


def speculative_draws() -> np.ndarray:
    """The uniform [0,1) numbers the acceptance test consumes, in order."""
    from vyomai_amd import recipe
    return (recipe.uniform("spec.rand", (512,)) * 0.5 + 0.5).astype(np.float32)


SPECULATIVE = {
    # a small drafter against a deeper target: accepts and rejects mixed
    "mixed": dict(target_layers=3, drafter_layers=1, drafter_prefix="spec.drafter.", prompt_len=6, gamma=4,
                  max_gen_len=18, eos=2, skip=False, first_target=True, processor=("GreedyProcessor", (1,))),
    # the drafter IS the target (same weights): every draft is accepted
    "same": dict(target_layers=2, drafter_layers=2, drafter_prefix="spec.target.", prompt_len=5, gamma=3,
                 max_gen_len=11, eos=2, skip=False, first_target=True, processor=("GreedyProcessor", (1,))),
    # no target prefill, no sample adjustment, temperature != 1, two stop tokens
    "plain": dict(target_layers=2, drafter_layers=1, drafter_prefix="spec.drafter.", prompt_len=7, gamma=5,
                  max_gen_len=14, eos=[2, 7], skip=True, first_target=False, processor=("GreedyProcessor", (0.7,))),
}
