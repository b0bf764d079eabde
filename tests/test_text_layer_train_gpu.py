"""A post-LN layer in training as one native call each way (vy_text_layer_train_fwd, vy_text_layer_bwd) against the modules one by one, whose
launches it makes in their order: the same bits.  What keeps the modules: hooks, dropout, parameters that are not the trainer's."""
import copy

import pytest
import torch

from tests.golden import cases

pytestmark = pytest.mark.gpu
DEV = "cuda"


def model(kind, width, heads, kv=None, layers=2, dropout=0.0):
    import vyomai_amd as V
    cfg = cases.with_kv(cases.test_cfg(), kv)
    cfg.num_hidden_layers, cfg.hidden_size, cfg.num_attention_heads, cfg.intermediate_size = layers, width, heads, 4 * width
    cfg.hidden_dropout_prob, cfg.vocab_size, cfg.max_position_embeddings = dropout, 500, 512
    torch.manual_seed(width + heads)
    m = (V.EncoderModel if kind == "encoder" else V.DecoderModel)(cfg, "rope", "gqa" if kv else None)
    return m.to(DEV).train()


def step(m, ids, mask, dtype=torch.bfloat16, one_by_one=False):
    """-> (states, gradients by name, native calls) of one backward pass of a fixed loss."""
    from vyomai_amd import _lib, autograd
    from vyomai_amd.models import decoder, encoder
    from vyomai_amd.training import FlatTrainer
    tr = FlatTrainer(m, lr=0.0, compute_dtype=dtype)
    seen, real = [], _lib.call
    _lib.call = lambda name, *a: (seen.append(name), real(name, *a))[1]
    if one_by_one:
        encoder.layer_train = decoder.layer_train = lambda *a: None
    try:
        tr.zero_grad()
        out = m.forward_hidden(ids, mask)[0] if hasattr(m, "lm_head") else m(ids, mask).logits
        w = torch.linspace(-1, 1, out.numel(), device=DEV).view(out.shape)
        tr.backward((out.float() * w).mean())
        torch.cuda.synchronize()
    finally:
        _lib.call = real
        encoder.layer_train = decoder.layer_train = autograd.layer_train
    return out.detach().clone(), {n: p.grad.clone() for n, p in m.named_parameters() if "all_layer" in n}, [n for n in seen if n.startswith("vy_text_layer")]


def inputs(B, L, padded):
    g = torch.Generator(device=DEV).manual_seed(B * L)
    ids = torch.randint(3, 500, (B, L), generator=g, device=DEV)
    mask = None
    if padded:
        mask = (torch.arange(L, device=DEV)[None] < torch.randint(1, L + 1, (B, 1), generator=g, device=DEV)).long()
    return ids, mask


@pytest.mark.parametrize("kind,width,heads,kv,B,L,padded,dtype", [
    ("decoder", 512, 8, None, 3, 65, False, torch.bfloat16), ("decoder", 768, 12, 4, 5, 33, True, torch.bfloat16),
    ("encoder", 512, 8, 4, 2, 128, True, torch.bfloat16), ("decoder", 512, 8, None, 1, 1, False, torch.bfloat16),
    ("decoder", 256, 2, None, 2, 40, False, torch.bfloat16), ("encoder", 256, 4, None, 2, 19, True, torch.float32)])
def test_bits_of_the_modules_one_by_one(kind, width, heads, kv, B, L, padded, dtype):
    ids, mask = inputs(B, L, padded)
    if kind == "encoder" and mask is None:
        mask = torch.ones_like(ids)
    a = model(kind, width, heads, kv)
    b = copy.deepcopy(a)
    y, grads, calls = step(a, ids, mask, dtype)
    y2, grads2, calls2 = step(b, ids, mask, dtype, one_by_one=True)
    assert calls == ["vy_text_layer_train_fwd"] * 2 + ["vy_text_layer_bwd"] * 2 and not calls2
    assert torch.equal(y, y2)
    for n in grads:
        # (weight gradients of products smaller than 512 x 512, and all in fp32, are sums in atomics: any order)
        close = (grads[n] - grads2[n]).abs().max() <= 2.0 ** -16 * grads2[n].abs().max() + 1e-12
        assert torch.equal(grads[n], grads2[n]) or close, n
        assert grads2[n].abs().max() > 0 or L == 1, n


def vision_step(one_by_one):
    """One backward pass of the captioning loss, both towers -> (loss, gradients of their layers, native calls)"""
    import vyomai_amd as V
    from vyomai_amd import _lib, autograd
    from vyomai_amd.models import multimodel, vision_encoder
    from vyomai_amd.training import FlatTrainer
    vcfg, cfg = cases.vit_cfg(), cases.with_kv(cases.test_cfg(), 4)
    vcfg.num_hidden_layers, vcfg.hidden_dropout_prob = 2, 0.0
    cfg.num_hidden_layers, cfg.hidden_dropout_prob, cfg.vocab_size = 2, 0.0, 500
    torch.manual_seed(5)
    vlm = V.VisionLanguageModel(cfg, V.Vit(vcfg), "rope", "gqa").to(DEV).train()
    tr = FlatTrainer(vlm, lr=0.0)
    ids = torch.randint(3, 500, (3, 12), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    img = torch.rand(3, 3, 224, 224, generator=torch.Generator(device=DEV).manual_seed(2), device=DEV).to(torch.bfloat16)
    mask = torch.ones_like(ids)
    mask[1, 8:] = 0
    seen, real = [], _lib.call
    _lib.call = lambda name, *a: (seen.append(name), real(name, *a))[1]
    if one_by_one:
        multimodel.layer_train = vision_encoder.layer_train = lambda *a: None
    try:
        tr.zero_grad()
        loss = vlm.caption_loss(img, ids, mask)
        tr.backward(loss)
        torch.cuda.synchronize()
    finally:
        _lib.call = real
        multimodel.layer_train = vision_encoder.layer_train = autograd.layer_train
    return loss.detach().clone(), {n: p.grad.clone() for n, p in vlm.named_parameters() if "all_layer" in n}, [n for n in seen if n.startswith("vy_text_layer")]


def test_vision_and_captioning_layers():
    """A packed projection with one bias, rows without a mask, and keys of an image ahead of padded ones."""
    (y, grads, calls), (y2, grads2, calls2) = vision_step(False), vision_step(True)
    assert calls == ["vy_text_layer_train_fwd"] * 4 + ["vy_text_layer_bwd"] * 4 and not calls2
    assert (y - y2).abs() <= 36 * 2.0 ** -24 * y2 and any("qkv" in n for n in grads)      # (a sum over 36 tokens in atomics)
    for n in grads:
        assert grads2[n].abs().max() > 0 and (grads[n] - grads2[n]).abs().max() <= 2.0 ** -16 * grads2[n].abs().max(), n      # (sums in atomics)


@pytest.mark.parametrize("causal", [False, True])
def test_mask_of_more_keys_than_rows(causal):
    """A layer by itself whose mask covers more keys than there are rows: the first ones count."""
    from vyomai_amd import autograd
    from vyomai_amd.layers.mask import AttnMask
    from vyomai_amd.training import FlatTrainer
    B, L, d = 3, 21, 512
    g = torch.Generator(device=DEV).manual_seed(4)
    x0, w = (torch.randn(B, L, d, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    keep = (torch.rand(B, L + 9, generator=g, device=DEV) < 0.6).to(torch.uint8)
    keep[:, 0] = 1
    results = []
    for one_by_one in (False, True):
        m = model("decoder", d, 8, layers=1)
        tr = FlatTrainer(m, lr=0.0)
        tr.zero_grad()
        layer, x = m.all_layer[0], x0.clone().requires_grad_()
        mask = AttnMask(causal=causal, start_pos=0, keypad=keep)
        if one_by_one:
            y = layer.feed_forward(layer.attention(hidden_state=x, attention_mask=mask, freqs=None)[0], x)
        else:
            y = autograd.layer_train(layer.attention, layer.feed_forward, x, mask, None)
            assert y is not None
        (y.float() * w.float()).sum().backward()
        torch.cuda.synchronize()
        results.append((y.detach(), x.grad, {n: p.grad.clone() for n, p in layer.named_parameters()}))
    (y, dx, grads), (y2, dx2, grads2) = results
    assert torch.equal(y, y2)
    # (one by one, autograd adds the input's three gradients in bf16 where no layer asked for them to be deferred: a rounding of each sum)
    assert ((dx.float() - dx2.float()).abs() <= 2.0 ** -6 * dx2.float().abs() + 2.0 ** -7 * dx2.float().abs().mean()).all()
    for n in grads:
        assert (grads[n] - grads2[n]).abs().max() <= 2.0 ** -16 * grads2[n].abs().max() + 1e-12, n


def test_what_keeps_the_modules():
    ids, mask = inputs(2, 20, False)
    m = model("decoder", 512, 8)
    ran = []
    handle = m.all_layer[0].feed_forward.register_forward_hook(lambda *a: ran.append(1))
    calls = step(m, ids, mask)[2]
    handle.remove()
    assert ran == [1] and calls == ["vy_text_layer_train_fwd", "vy_text_layer_bwd"]      # (the other layer's)
    assert not step(model("decoder", 512, 8, dropout=0.1), ids, mask)[2]
    m = model("decoder", 512, 8)
    m.all_layer[1].attention.out.dense.weight.requires_grad_(False)
    assert step(m, ids, mask)[2] == ["vy_text_layer_train_fwd", "vy_text_layer_bwd"]
    m = model("decoder", 512, 8).to(torch.bfloat16)      # (no trainer: gradients are returned)
    m.forward_hidden(ids, None)[0].float().square().mean().backward()
    assert all(p.grad is not None for n, p in m.named_parameters() if "all_layer" in n)


def test_saved_tensors_go_through_their_hooks():
    ids, mask = inputs(3, 50, False)
    a = model("decoder", 512, 8)
    b = copy.deepcopy(a)
    want = step(a, ids, mask)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.to(DEV)):
        got = step(b, ids, mask)
    assert len(packed) >= 6 and torch.equal(got[0], want[0]) and all(torch.equal(got[1][n], want[1][n]) for n in want[1])


def hooked(kind, ff, att):
    """A hook of that kind that changes a gradient -> handles"""
    from torch.nn.modules import module as M
    half = lambda g: tuple(None if t is None else 0.5 * t for t in g)
    if kind == "full":
        return [ff.register_full_backward_hook(lambda m, gi, go: half(gi))]
    if kind == "pre":
        return [att.register_full_backward_pre_hook(lambda m, go: half(go))]
    if kind == "old":
        return [ff.register_backward_hook(lambda m, gi, go: None)]
    if kind == "global":
        return [M.register_module_full_backward_hook(lambda m, gi, go: half(gi) if m is ff else None)]
    return [M.register_module_full_backward_pre_hook(lambda m, go: half(go) if m is att else None)]


@pytest.mark.parametrize("kind", ["full", "pre", "old", "global", "global pre"])
def test_backward_hooks_see_their_modules(kind):
    """A hook that halves a gradient: what the modules one by one make of it."""
    ids, mask = inputs(2, 20, False)
    plain = model("decoder", 512, 8)
    results = []
    for one_by_one in (False, True):
        m = copy.deepcopy(plain)
        handles = hooked(kind, m.all_layer[1].feed_forward, m.all_layer[1].attention)
        try:
            results.append(step(m, ids, mask, one_by_one=one_by_one))
        finally:
            for h in handles:
                h.remove()
    (y, grads, calls), (y2, grads2, _) = results
    assert calls == ([] if "global" in kind else ["vy_text_layer_train_fwd", "vy_text_layer_bwd"])      # (the other layer's)
    assert torch.equal(y, y2)
    unhooked = step(plain, ids, mask)[1]
    changed = False
    for n in grads:
        bound = 2.0 ** -16 * grads2[n].abs().max() + 1e-12      # (as above: sums in atomics)
        assert (grads[n] - grads2[n]).abs().max() <= bound, n
        changed |= bool((grads[n] - unhooked[n]).abs().max() > bound)
    assert changed == (kind != "old"), kind


def test_what_waiting_weight_gradients_hold(monkeypatch):
    """Their operands and nothing else of the layer, 16 numbers of a row's width a token: x, o, a and the inner rows of four widths, and
    the gradients of both norms' inputs, of the inner rows and of the projections of three widths."""
    from vyomai_amd import autograd_train as AT
    B, L, d, layers = 8, 256, 512, 2
    ids, mask = inputs(B, L, False)
    held, real = [], AT.ops.linear_wgrad_grouped

    def launch(items):
        held.extend(t for dy, x, *_ in items for t in (dy, x))
        real(items)
    monkeypatch.setattr(AT.ops, "linear_wgrad_grouped", launch)
    calls = step(model("decoder", d, 8, layers=layers), ids, mask)[2]
    assert len(calls) == 2 * layers and len(held) >= 2 * 4 * layers
    storages = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for t in held}
    assert sum(storages.values()) <= layers * (16 * d * B * L * 2 + 16 * 128)     # (a segment is filled up to a line)
