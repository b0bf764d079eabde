"""Decode steps of 1 to 4 sequences, whose products make their operand rows themselves (vyomai_amd/csrc/vy_few.hip): every number of
rows, the widths that have kernels, padded widths, odd vocabularies and layers without a feed-forward, against steps that run the
norms and products one by one."""
import pytest
import torch

from tests.test_decode_lean_gpu import _plan, _step

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


def decoder(width, pos_kind, kv_heads, dtype, layers=2):
    import vyomai_amd as V
    from vyomai_amd import recipe
    cfg = V.EncoderConfig(hidden_size=width, num_attention_heads=width // 64, num_hidden_layers=layers, max_position_embeddings=256,
                          intermediate_size=4 * width, hidden_dropout_prob=0.0, vocab_size=1003)
    if kv_heads:
        cfg.num_key_value_heads = kv_heads
    m = V.DecoderModel(cfg, pos_kind, "gqa" if kv_heads else None)
    recipe.load_recipe_(m)
    return cfg, m.to(DEV).to(dtype).eval()


@pytest.mark.parametrize("B", [1, 2, 3, 4])
@pytest.mark.parametrize("width,pos_kind,kv_heads", [(512, "rope", None), (768, "rope", 4), (768, "absolute", None), (1024, "rope", 2)])
def test_decoder_step(B, width, pos_kind, kv_heads):
    """Against the fp32 step on the same weights.  A layer rounds seven rows to bf16 (operand, q / k / v, attention, both sums, the
    normalised sum, the feed-forward's middle), the head three; each adds at most 2^-8 relative to what comes out of a norm."""
    g = torch.Generator().manual_seed(width + B)
    cfg, m = decoder(width, pos_kind, kv_heads, BF)
    x = (torch.randn(B, width, generator=g) * 0.5).to(BF).to(DEV)
    plan, cache = _plan(cfg, m, B, BF)
    got = _step(plan, cache, x, 37, 1)
    for lean in (0, 1):   # the general launchers; the same kernels again, from the state that the first call left
        other, its = _plan(cfg, m, B, BF)
        same = _step(other, its, x, 37, lean)
        for (k, v), (ok, ov) in zip(got[2], same[2]):
            assert (k - ok).norm() <= 14 * 2.0 ** -8 * ok.norm() and (v - ov).norm() <= 14 * 2.0 ** -8 * ov.norm()
    assert torch.equal(got[0], same[0]) and torch.equal(got[1], same[1])
    cfg32, m32 = decoder(width, pos_kind, kv_heads, torch.float32)
    plan32, cache32 = _plan(cfg32, m32, B, torch.float32)
    want = _step(plan32, cache32, x.float(), 37, 1)
    # (this plan's cache holds the unrounded rows: one more rounding)
    for a, b, n in ((got[1], want[1], 15), (got[0], want[0], 18)):
        assert torch.isfinite(a).all() and (a - b).norm() <= n * 2.0 ** -8 * b.norm(), float((a - b).norm() / b.norm())


def gisitar(width):
    from vyomai_amd import GisitarConfig, GisitarModel
    lig = {"type": "lightning", "mixer": {"heads": 8, "dim": 64, "vdim": 64, "decay": [0.9] * 8}}
    lat = {"type": "latent_attention", "mixer": {"heads": 4, "dim": 64, "vdim": 64, "q_rank": 256, "kv_rank": 128, "scale": 0.125}}
    ff = {"kind": "dense", "ff": 1496}
    return GisitarModel(GisitarConfig(vocab=1003, width=width, layers=[{**lig, "mlp": None}, {**lat, "mlp": ff}, {**lig, "mlp": ff},
                                                                       {**lat, "mlp": None}]))


def biruvik(width):
    from tests import biruvik_cases as K
    from vyomai_amd import BiruvikConfig, BiruvikModel
    return BiruvikModel(BiruvikConfig.from_dict(K.config([K.hgrn2(4, 64, 64, mlp=K.dense(1500)), K.latent(4, 64, 64, 128, 64),
                                                          K.attention(4, 2, 64, 128, mlp=K.dense(768))], width=width, vocab=1003)))


@pytest.mark.parametrize("B", [1, 2, 3, 4])
@pytest.mark.parametrize("make,width", [(gisitar, 1024), (gisitar, 1020), (gisitar, 2048), (gisitar, 1032), (biruvik, 1024),
                                        (biruvik, 2044)])
def test_hybrid_step(make, width, B):
    """A next token through the step and through the prompt path (other product and norm kernels): the logits agree within bf16
    roundings of the sublayers' inputs, 2^-9 relative each, at most eight per layer and a vocabulary product."""
    torch.manual_seed(width)
    with torch.device(DEV):
        torch.set_default_dtype(BF)
        try:
            m = make(width).eval()
        finally:
            torch.set_default_dtype(torch.float32)
    ids = torch.randint(0, 1003, (B, 6), device=DEV, generator=torch.Generator(device=DEV).manual_seed(B))
    cache = m.new_cache(B + 2, 8)
    cache.allocate(2)   # (slots that are not the rows numbers)
    slots = cache.allocate(B)
    m.prefill(ids[:, :2].contiguous(), [2] * B, cache, slots)
    for t in range(2, 6):
        got = m.decode(ids[:, t].contiguous(), cache, slots).double()
        other = m.new_cache(B, 8)
        s = other.allocate(B)
        want = m.logits(m.prefill(ids[:, :t + 1].contiguous(), [t + 1] * B, other, s)[:, -1]).double()
        assert torch.isfinite(got).all()
        assert (got - want).norm() <= 8 * len(m.layers) * 2.0 ** -9 * want.norm(), float((got - want).norm() / want.norm())


@pytest.mark.parametrize("B", [1, 2, 3, 4])
@pytest.mark.parametrize("q_rank,kv_rank,window", [(512, 128, None), (512, 250, 5), (508, 128, 5), (1024, 512, None), (1020, 1000, 3), (1024, 64, 8)])
def test_hybrid_step_with_wide_query_latents(q_rank, kv_rank, window, B):
    """Query latents of 512 and 1024 columns (padded to them), which the queries' product norms itself: in slots that are not the rows'
    numbers, with every earlier token in the cache and with rings that turn (the windows are shorter than the 12 tokens).  Bound: as above."""
    from vyomai_amd import GisitarConfig, GisitarModel
    from vyomai_amd.layers.latent_attention import LatentAttention
    torch.manual_seed(q_rank + kv_rank)
    mixer = {"heads": 4, "dim": 64, "vdim": 64, "q_rank": q_rank, "kv_rank": kv_rank, "scale": 0.125}
    with torch.device(DEV):
        torch.set_default_dtype(BF)
        try:
            m = GisitarModel(GisitarConfig(vocab=1003, width=1024, layers=[{"type": "latent_attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": 1496}},
                                                                           {"type": "latent_attention", "mixer": mixer, "mlp": None}]))
            if window:
                for layer in m.layers:
                    layer.mixer = LatentAttention(1024, 4, 64, 64, q_rank, kv_rank, 0.125, 1e-5, window=window)
        finally:
            torch.set_default_dtype(torch.float32)
    m = m.eval()
    assert m.layers[0].mixer.packed().q_norm.numel() in (512, 1024)
    ids = torch.randint(0, 1003, (B, 12), device=DEV, generator=torch.Generator(device=DEV).manual_seed(B))
    cache = m.new_cache(B + 2, 16)
    cache.allocate(2)
    slots = cache.allocate(B)[::-1]
    m.prefill(ids[:, :2].contiguous(), [2] * B, cache, slots)
    for t in range(2, 12):
        got = m.decode(ids[:, t].contiguous(), cache, slots).double()
        other = m.new_cache(B, 16)
        s = other.allocate(B)
        want = m.logits(m.prefill(ids[:, :t + 1].contiguous(), [t + 1] * B, other, s)[:, -1]).double()
        assert torch.isfinite(got).all()
        assert (got - want).norm() <= 8 * len(m.layers) * 2.0 ** -9 * want.norm(), float((got - want).norm() / want.norm())


@pytest.mark.parametrize("B", [1, 2, 4])
def test_what_a_step_refuses(B):
    """Vocabulary weights that are not there and logits rows narrower than the vocabulary: errors, as from the general launchers, and the
    plan works again afterwards."""
    from vyomai_amd._lib import VyomHipError
    cfg, m = decoder(512, "rope", None, BF, layers=1)
    x = torch.randn(B, 512, device=DEV, generator=torch.Generator(device=DEV).manual_seed(B)).to(BF)
    plan, cache = _plan(cfg, m, B, BF)
    want = _step(plan, cache, x, 5, 1)[0]
    keep, ldv = plan.plan.head_wv, plan.ldv
    plan.plan.head_wv = None
    with pytest.raises(VyomHipError, match="null operand"):
        plan.step(x, 6)
    plan.plan.head_wv, plan.ldv = keep, 1000
    with pytest.raises(VyomHipError, match="1000"):
        plan.step(x, 6)
    plan.ldv = ldv
    assert torch.equal(_step(plan, cache, x, 5, 1)[0], want)


@pytest.mark.parametrize("B", [2, 4])
def test_what_a_hybrid_step_refuses(B):
    from vyomai_amd import _lib, decode_plan
    torch.manual_seed(3)
    with torch.device(DEV):
        torch.set_default_dtype(BF)
        try:
            m = gisitar(1024).eval()
        finally:
            torch.set_default_dtype(torch.float32)
    ids = torch.randint(0, 1003, (B, 3), device=DEV)
    cache = m.new_cache(B, 8)
    slots = cache.allocate(B)
    m.prefill(ids[:, :2].contiguous(), [2] * B, cache, slots)
    plans, real = [], decode_plan.HybridDecodePlan.step

    def seen(self, *a):
        plans.append((self, a))
        return real(self, *a)
    decode_plan.HybridDecodePlan.step = seen
    try:
        m.decode(ids[:, 2].contiguous(), cache, slots)
    finally:
        decode_plan.HybridDecodePlan.step = real
    plan, args = plans[0]
    head, ldv = plan.plan.head, plan.ldv
    plan.plan.head = None
    with pytest.raises(_lib.VyomHipError, match="null operand"):
        real(plan, *args)
    plan.plan.head, plan.ldv = head, 1000
    with pytest.raises(_lib.VyomHipError, match="ldy < N"):
        real(plan, *args)
    plan.plan.head, plan.ldv = head, ldv


def test_hidden_rows_at_any_address():
    """vy_decoder_step leaves the hidden state wherever it is asked to: two bytes off a 16-byte line the general launchers take the step."""
    import ctypes as C
    from vyomai_amd import _lib, ops
    cfg, m = decoder(768, "rope", 4, BF)
    x = torch.randn(2, 768, device=DEV, generator=torch.Generator(device=DEV).manual_seed(9)).to(BF)
    plan, cache = _plan(cfg, m, 2, BF)
    logits, want = plan.step(x, 5, want_hidden=True)
    want = want.clone()
    for off in (0, 1, 4):
        room = torch.zeros(2 * 768 + 16, dtype=BF, device=DEV)
        for logits_ptr in (logits.data_ptr(), None):
            _lib.call("vy_decoder_step", C.byref(plan.plan), x.data_ptr(), 5, None, room.data_ptr() + 2 * off, logits_ptr, plan.ldv,
                      ops._raw_stream())
            got = room[off:off + 2 * 768].view(2, 768).float()
            assert (got - want.float()).norm() <= 18 * 2.0 ** -8 * want.float().norm() and room[:off].eq(0).all() and room[off + 1536:].eq(0).all()


def test_what_four_sequences_cost():
    """Width 1024: a step of four takes 1.2 times what a step of one takes; with the output projection inside the attention, whose sixteen
    heads' shares every workgroup of the next product adds up, 1.65 times."""
    from tests.test_decode_products_gpu import microseconds
    us = {}
    for B in (1, 4):
        cfg, m = decoder(1024, "rope", None, BF, layers=6)
        plan, cache = _plan(cfg, m, B, BF)
        x, hidden = torch.randn(B, 1024, device=DEV).to(BF), torch.empty(B, 1024, dtype=BF, device=DEV)
        us[B] = microseconds(lambda: plan._launch(x.data_ptr(), 60, None, hidden.data_ptr(), None), 4)
    assert us[4] <= 1.4 * us[1], us
