"""A layer as one native call against the same layer module by module (a forward hook on a module asks for that): equal bit by bit over
what the call takes -- layer classes, masks, caches, single tokens, both data types, fp32 weights under bf16 rows -- and refused to
the general path where it does not."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


def config(**kw):
    import vyomai_amd as V
    cfg = V.EncoderConfig(num_hidden_layers=2, hidden_size=kw.pop("d", 128), num_attention_heads=kw.pop("h", 2), vocab_size=97,
                          max_position_embeddings=64, hidden_dropout_prob=kw.pop("p", 0.0))
    for k, v in kw.items():
        setattr(cfg, k, v)
    return cfg


def both(model, layers, call):
    """call() with the native layers and with a hook on every feed-forward; how often the native call ran in each."""
    from vyomai_amd import ops
    runs, inner = [0], ops.text_layer

    def counted(*a):
        runs[0] += 1
        return inner(*a)
    ops.text_layer = counted
    try:
        a, n = call(), runs[0]
        handles = [l.feed_forward.register_forward_hook(lambda *a: None) for l in layers]
        b, m = call(), runs[0] - n
        for h in handles:
            h.remove()
    finally:
        ops.text_layer = inner
    return a, b, n, m


@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("attention", [None, "gqa"])
@pytest.mark.parametrize("B,L,padded", [(1, 1, False), (3, 17, True), (2, 64, False), (5, 33, True)])
def test_encoder_layers(dtype, attention, B, L, padded):
    import vyomai_amd as V
    torch.manual_seed(B + L)
    m = V.EncoderModel(config(h=4, d=256, num_key_value_heads=2), "rope", attention).to(DEV, dtype).eval()
    ids = torch.randint(3, 97, (B, L), device=DEV)
    keep = torch.ones(B, L, dtype=torch.long, device=DEV)
    if padded:
        keep[0, L // 2:] = 0
    with torch.no_grad():
        a, b, n, k = both(m, m.all_layer, lambda: m(ids, keep).logits)
    assert n == 2 and k == 0 and torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("cache", ["none", "static", "dynamic"])
@pytest.mark.parametrize("pos", ["rope", "absolute"])
def test_decoder_layers_and_their_caches(dtype, cache, pos):
    import vyomai_amd as V
    torch.manual_seed(7)
    cfg = config(d=128, h=2)
    m = V.DecoderModel(cfg, pos, None).to(DEV, dtype).eval()
    ids = torch.randint(3, 97, (3, 21), device=DEV)

    def go():
        kw = {}
        if cache != "none":
            kv = V.StaticCacheOne(cfg, max_cache_len=32, batch_size=3, dtype=dtype) if cache == "static" else V.DynamicCacheOne(cfg)
            kw = dict(use_cache=True, kv_cache=kv)
        first = m(ids[:, :12], **kw).logits
        if cache == "none":
            return first
        portion = m(ids[:, 12:20], start_pos=12, **kw).logits
        one = m(ids[:, 20:], start_pos=20, **kw).logits
        return torch.cat([first, portion, one], 1)
    with torch.no_grad():
        a, b, n, k = both(m, m.all_layer, go)
    assert n == (2 if cache == "none" else 6) and k == 0 and torch.equal(a, b)


def test_odd_head_widths_and_inner_sizes():
    import vyomai_amd as V
    torch.manual_seed(3)
    m = V.EncoderModel(config(d=144, h=2), "absolute", None).to(DEV, BF).eval()       # heads of 72
    ids = torch.randint(3, 97, (2, 19), device=DEV)
    with torch.no_grad():
        a, b, n, k = both(m, m.all_layer, lambda: m(ids, torch.ones_like(ids)).logits)
    assert n == 2 and k == 0 and torch.equal(a, b)


def test_what_the_native_layer_does_not_take():
    import vyomai_amd as V
    from vyomai_amd.autograd import layer_forward
    torch.manual_seed(5)
    cfg = config(p=0.5)
    m = V.DecoderModel(cfg, "rope", None).to(DEV, BF).eval()
    l, x = m.all_layer[0], torch.randn(2, 8, 128, device=DEV, dtype=BF)
    with torch.no_grad():
        assert layer_forward(l.attention, l.feed_forward, x, None, None) is not None
        assert layer_forward(l.attention, l.feed_forward, x.transpose(0, 1), None, None) is None          # rows not contiguous
        assert layer_forward(l.attention, l.feed_forward, x, torch.zeros(2, 1, 8, 8, device=DEV), None) is None   # dense mask
        l.train()
        assert layer_forward(l.attention, l.feed_forward, x, None, None) is None                          # dropout
        l.eval()

        class Mine(type(l.attention)):
            def forward(self, *a, **k):
                return super().forward(*a, **k)
        l.attention.__class__ = Mine
        assert layer_forward(l.attention, l.feed_forward, x, None, None) is None                          # another forward
    l.attention.__class__ = Mine.__mro__[1]
    assert layer_forward(l.attention, l.feed_forward, x, None, None) is None                              # gradients wanted


@pytest.mark.parametrize("which", ["attention", "feed_forward"])
def test_a_forward_set_on_a_module_is_called(which):
    """As profilers and quantisers wrap modules: layer.feed_forward.forward = wrapped."""
    import vyomai_amd as V
    torch.manual_seed(6)
    m = V.EncoderModel(config(), "rope", None).to(DEV, BF).eval()
    ids = torch.randint(3, 97, (2, 9), device=DEV)
    keep = torch.ones_like(ids)
    with torch.no_grad():
        want = m(ids, keep).logits
        module, calls = getattr(m.all_layer[1], which), []
        inner = module.forward

        def wrapped(*a, **k):
            calls.append(1)
            return inner(*a, **k) * 2
        module.forward = wrapped
        twice = m(ids, keep).logits
        assert len(calls) == 1 and not torch.equal(twice, want)
        del module.forward
        assert torch.equal(m(ids, keep).logits, want) and len(calls) == 1


def test_an_attention_of_the_users_own():
    """A layer calls whatever module stands in its place, without asking it for a layer number."""
    import vyomai_amd as V
    torch.manual_seed(8)
    cfg = config()
    l = V.DecoderModel(cfg, "rope", None).to(DEV, BF).eval().all_layer[0]

    class Halves(torch.nn.Module):
        def forward(self, hidden_state, attention_mask, freqs=None, use_cache=False, kv_cache=None, start_pos=0):
            return hidden_state / 2, kv_cache
    l.attention = Halves()
    x = torch.randn(2, 8, 128, device=DEV, generator=torch.Generator(device=DEV).manual_seed(8)).to(BF)
    cache = V.DynamicCacheOne(cfg)
    with torch.no_grad():
        for kw in ({}, dict(use_cache=True, kv_cache=cache, start_pos=3)):
            y, kept = l(x, None, None, **kw)
            assert torch.equal(y, l.feed_forward(x / 2, x)) and kept is kw.get("kv_cache")
