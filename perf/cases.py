"""The work that users of this package have it do, as cases that can be timed and checked: training steps, text encoding, prompt
processing and token generation, through the package's public entry points, on synthetic inputs and random weights.

A case is a dict of plain values.  `listed` names the ones that are always measured, `draw` gives more of the same ranges, `prepare`
makes what a program has in hand before the call, `run` is one pass, `work` is what the pass cannot do without, `exact` computes the
same outputs in 64 bits with plain torch.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F

BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
D, HEADS, DH, VOCAB, POSITIONS = 768, 12, 64, 50265, 1024     # the text models of bench.py
IMAGE, PATCH = 224, 16                                        # ViT-B/16
PATCHES = (IMAGE // PATCH) ** 2
KV_HEADS = 4                                                  # of a grouped-query text model
LAYERS = 12
# the decoders that mix layer kinds, as bench.py --model sizes them: heads of 128, vocabulary 32000
HEAD, MIX_VOCAB, WINDOW = 128, 32000, 1024
LATENT = {1024: (8, 512, 256), 2048: (16, 1024, 512)}         # width -> heads, query latent, key/value latent
GATED_FF = {1024: 4096, 2048: 8192}
PLAIN_FF = {1024: 6144, 2048: 12288}
EXPERTS = {1024: (32, 4, 4, 2, 512, 1024), 2048: (64, 4, 8, 4, 1024, 2048)}   # experts, top, groups, kept, width, shared width
# the learning rate of a warm-up: full steps of a fresh AdamW move every weight by as much, whichever way rounding tips the tiny gradients
LR, BETAS, ADAM_EPS, DECAY = 1e-6, (0.9, 0.999), 1e-8, 0.01
LIMIT, ALPHA, CAP, TEMP, DIFF = 7.0, 1.702, 30.0, (0.1, 4096), 0.5


def listed():
    return [
        # one step of causal language model training at the benchmark's size: 16384 tokens a step
        {"name": "train 32x512", "kind": "train", "batch": 32, "length": 512, "grouped": False, "padded": False},
        # fine-tuning on few short rows of odd length with padding, grouped key/value heads
        {"name": "train 5x333 padded", "kind": "train", "batch": 5, "length": 333, "grouped": True, "padded": True},
        # caption training: 64 images (197 tokens each) and captions of 32 tokens, ViT-B/16 and a 12-layer decoder
        {"name": "caption 64", "kind": "caption", "batch": 64, "length": 32},
        # text encoding on arrival: a few short texts, where launches and latency count
        {"name": "encode 4x128", "kind": "encode", "batch": 4, "length": 128, "grouped": False, "padded": False},
        # text encoding in bulk: rows of unequal length
        {"name": "encode 61x500 padded", "kind": "encode", "batch": 61, "length": 500, "grouped": False, "padded": True},
        # a full batch of generation requests on the text decoder: prompts of 512, then token by token
        {"name": "serve 32x512+24", "kind": "serve", "batch": 32, "length": 512, "new": 24, "grouped": False},
        # one user, a short prompt
        {"name": "serve 1x60+24", "kind": "serve", "batch": 1, "length": 60, "new": 24, "grouped": True},
        # prompts of a batch through the decoder with latent and lightning attention
        {"name": "gisitar 8x1024", "kind": "gisitar", "width": 2048, "batch": 8, "length": 1024, "new": 0},
        # one conversation on it, smaller width
        {"name": "gisitar 1x700+24", "kind": "gisitar", "width": 1024, "batch": 1, "length": 700, "new": 24},
        # one long document through the decoder with gated linear, differential and windowed latent attention
        {"name": "biruvik 1x8192", "kind": "biruvik", "width": 2048, "batch": 1, "length": 8192, "new": 0},
        # a full batch of conversations on it
        {"name": "biruvik 32x250+16", "kind": "biruvik", "width": 1024, "batch": 32, "length": 250, "new": 16},
        # prompts through parallel layers of windowed attention and a mixture of experts
        {"name": "rivudra 3x2731", "kind": "rivudra", "width": 2048, "batch": 3, "length": 2731, "new": 0},
    ]


def spread(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["train", "train", "caption", "encode", "encode", "serve", "serve", "gisitar", "biruvik", "rivudra"])
    if kind in ("train", "encode"):
        length = spread(rng, 24, 512)
        batch = spread(rng, 1, min(64 if kind == "encode" else 32, 16384 // length))
        return {"kind": kind, "batch": batch, "length": length, "grouped": rng.random() < 0.5, "padded": rng.random() < 0.5}
    if kind == "caption":
        return {"kind": kind, "batch": spread(rng, 2, 64), "length": rng.randint(8, 32)}
    if kind == "serve":
        return {"kind": kind, "batch": spread(rng, 1, 32), "length": spread(rng, 20, 512), "new": rng.randint(4, 24),
                "grouped": rng.random() < 0.5}
    width = rng.choice([1024, 2048])
    if kind == "rivudra" or rng.random() < 0.5:      # prompts only
        length = spread(rng, 100, 8192)
        return {"kind": kind, "width": width, "batch": spread(rng, 1, max(1, min(16, 8192 // length))), "length": length, "new": 0}
    return {"kind": kind, "width": width, "batch": spread(rng, 1, 32), "length": spread(rng, 20, 256), "new": rng.randint(4, 16)}


# ---- weights and inputs ------------------------------------------------------------------------------

def text_shapes(case, causal, prefix=""):
    """Parameters of a text model (causal: a decoder, with the vocabulary head), in the reference's names."""
    kv = KV_HEADS * DH if case.get("grouped") else D
    s = {prefix + "word_embeddings.weight": (VOCAB, D)}
    for i in range(LAYERS):
        s.update(block_shapes(f"{prefix}all_layer.{i}.", {"query": D, "key": kv, "value": kv}))
    if causal:
        h = prefix + "lm_head."
        s.update({h + "dense.weight": (D, D), h + "dense.bias": (D,), h + "layer_norm.weight": (D,), h + "layer_norm.bias": (D,),
                  h + "decoder.weight": (VOCAB, D), h + "bias": (VOCAB,)})
    return s


def block_shapes(p, projections):
    s = {}
    for n, rows in projections.items():
        s[f"{p}attention.{n}.weight"], s[f"{p}attention.{n}.bias"] = (rows, D), (rows,)
    s.update({p + "attention.out.dense.weight": (D, D), p + "attention.out.dense.bias": (D,),
              p + "attention.out.layernorm.weight": (D,), p + "attention.out.layernorm.bias": (D,),
              p + "feed_forward.intermediate.weight": (4 * D, D), p + "feed_forward.intermediate.bias": (4 * D,),
              p + "feed_forward.layernorm.weight": (D,), p + "feed_forward.layernorm.bias": (D,),
              p + "feed_forward.out.weight": (D, 4 * D), p + "feed_forward.out.bias": (D,)})
    return s


def caption_shapes(case):
    s = text_shapes(case, True, "decoder.")
    p, patch = "encoder.", 3 * PATCH * PATCH
    s.update({p + "cls_token": (1, 1, patch), p + "position_embeddings.pos_embeddings": (1, PATCHES + 1, patch)})
    for i in range(LAYERS):
        s.update(block_shapes(f"{p}all_layer.{i}.", {"qkv": 3 * D}))
    s.update({p + "pixel_seq.weight": (D, 3, PATCH, PATCH), p + "pixel_seq.bias": (D,)})
    return s


def mixed_layers(case):
    """Layer descriptions of a decoder that mixes layer kinds, as its configuration takes them."""
    w = case["width"]
    H, qr, kr = LATENT[w]
    if case["kind"] == "gisitar":
        dense = {"kind": "dense", "ff": GATED_FF[w]}
        lat = {"type": "latent_attention", "mixer": {"heads": H, "dim": HEAD, "vdim": HEAD, "q_rank": qr, "kv_rank": kr,
                                                     "scale": HEAD ** -0.5}, "mlp": dense}
        lig = {"type": "lightning", "mixer": {"heads": H, "dim": HEAD, "vdim": HEAD,
                                              "decay": [math.exp(-(2.0 ** -(1 + 6 * h / H))) for h in range(H)]}, "mlp": dense}
        return [lat, lig] * 4
    if case["kind"] == "biruvik":
        dense = {"kind": "dense", "ff": PLAIN_FF[w]}
        gla = {"type": "hgrn2", "mixer": {"heads": H, "dim": HEAD, "vdim": HEAD}, "mlp": dense}
        dif = {"type": "attention", "mixer": {"heads": H, "kv_heads": H // 4, "dim": HEAD // 2, "vdim": HEAD, "scale": (HEAD // 2) ** -0.5,
                                              "diff": DIFF, "q_temp": {"coef": TEMP[0], "every": TEMP[1]}}, "mlp": dense}
        lat = {"type": "latent_attention", "mixer": {"heads": H, "dim": HEAD, "vdim": HEAD, "kv_rank": kr, "scale": HEAD ** -0.5,
                                                     "mask": {"size": WINDOW}}, "mlp": dense}
        return [gla, dif, gla, lat] * 2
    E, top, groups, keep, ff, shared = EXPERTS[w]
    # (two layers: a token whose two best experts are a rounding error apart takes another path, and each layer adds such tokens)
    return [{"type": "attention", "mixer": {"heads": H, "kv_heads": H // 4, "dim": HEAD, "vdim": HEAD, "scale": HEAD ** -0.5,
                                            "mask": {"size": WINDOW}, "rot": {"base": 10000.0, "dims": HEAD}},
             "mlp": {"kind": "moe", "router": {"experts": E, "top": top, "scale": 1.0, "groups": {"count": groups, "keep": keep}},
                     "expert": {"ff": ff, "limit": LIMIT}, "shared": {"ff": shared, "limit": LIMIT}}}] * 2


def mixed_shapes(case):
    w = case["width"]
    H, qr, kr = LATENT[w]
    n = H * HEAD
    s = {"word_embeddings.weight": (MIX_VOCAB, w), "head.weight": (MIX_VOCAB, w)}
    vec = () if case["kind"] == "biruvik" else (w,)
    s["final_norm.weight"] = vec
    for i, layer in enumerate(mixed_layers(case)):
        p, m, t = f"layers.{i}.", f"layers.{i}.mixer.", layer["type"]
        s.update({p + k + ".weight": vec for k in (["norm1"] if case["kind"] == "rivudra" else ["norm1", "norm1b", "norm2", "norm2b"])})
        s[m + "out.weight"] = (w, n)
        if t == "latent_attention":
            if "q_rank" in layer["mixer"]:
                s.update({m + "q_down.weight": (qr, w), m + "q_norm.weight": (qr,), m + "q_up.weight": (n, qr), m + "gate.weight": (n, w)})
            else:
                s.update({m + "query.weight": (n, w), m + "gate.weight": (H, w)})
            s.update({m + "kv_down.weight": (kr, w), m + "kv_norm.weight": (kr,), m + "k_up.weight": (n, kr), m + "v_up.weight": (n, kr)})
        elif t == "lightning":
            s.update({m + k + ".weight": (n, w) for k in ("query", "key", "value", "gate")})
            s[m + "norm.weight"] = (n,)
        elif t == "hgrn2":
            s.update({m + k + ".weight": (n, w) for k in ("query", "forget", "value")})
            s.update({m + "forget.bias": (n,), m + "lower": (n,), m + "norm.weight": (HEAD,)})
        elif case["kind"] == "biruvik":
            for k, rows in (("query", n), ("key", n // 4), ("value", n // 4)):
                s[m + k + ".weight"], s[m + k + ".bias"] = (rows, w), (rows,)
            s.update({m + k: (HEAD // 2,) for k in ("q_norm.weight", "k_norm.weight", "lq1", "lk1", "lq2", "lk2")})
        else:
            s.update({m + "query.weight": (n, w), m + "key.weight": (n // 4, w), m + "value.weight": (n // 4, w), m + "gate.weight": (n, w)})
        f = p + "mlp."
        if case["kind"] == "rivudra":
            E, _, _, _, ff, sh = EXPERTS[w]
            s.update({f + "router.weight": (E, w), f + "gate": (E, ff, w), f + "up": (E, ff, w), f + "down": (E, w, ff),
                      f + "shared.gate.weight": (sh, w), f + "shared.up.weight": (sh, w), f + "shared.down.weight": (w, sh)})
        else:
            ff = layer["mlp"]["ff"]
            s.update({f + "up.weight": (ff, w), f + "down.weight": (w, ff)})
            if case["kind"] == "gisitar":
                s[f + "gate.weight"] = (ff, w)
    return s


def shapes_of(case):
    kind = case["kind"]
    if kind == "caption":
        return caption_shapes(case)
    if kind in ("train", "encode", "serve"):
        return text_shapes(case, kind != "encode")
    return mixed_shapes(case)


def numbers(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + sum(ord(c) * (i + 1) for i, c in enumerate(case["kind"]))) % (1 << 62))
    return g


def weights(case, g):
    """Random weights with the spread of a trained model's: matrices keep the size of what they multiply, norms are near one (Rivudra
    stores them around zero), what is added to the residual stream of parallel layers is smaller than the stream."""
    dt = F32 if case["kind"] in ("train", "caption") else BF
    out = {}
    for name, shape in shapes_of(case).items():
        z = torch.randn(shape, generator=g, device="cuda", dtype=F32)
        leaf = name.rsplit(".", 1)[-1]
        if "norm" in name.split(".")[-2] and leaf == "weight":
            z = 0.1 * z + (0.0 if case["kind"] == "rivudra" else 1.0)
        elif leaf == "lower":                        # least forget gate of a channel: from none to long memory
            z = torch.sigmoid(2.0 * z)
        elif leaf in ("lq1", "lk1", "lq2", "lk2"):
            z = 0.1 * z
        elif leaf == "bias":
            z = 0.02 * z
        elif "embeddings" in name or leaf == "cls_token":
            z = 0.5 * z
        else:
            z = z * (0.6 / math.sqrt(math.prod(shape[1:] if leaf == "weight" else shape[2:])))
        out[name] = z.to(dt)
    return out


def lengths_of(case, g):
    """Tokens of each row: all of them, or (padded) from a third to the whole, the first row whole."""
    n = torch.full((case["batch"],), case["length"], dtype=torch.long, device="cuda")
    if case.get("padded"):
        n[1:] = torch.randint(max(2, case["length"] // 3), case["length"] + 1, (case["batch"] - 1,), generator=g, device="cuda")
    return n


def inputs(case, g):
    vocab = VOCAB if case["kind"] in ("train", "caption", "encode", "serve") else MIX_VOCAB
    B, L, new = case["batch"], case["length"], case.get("new", 0)
    s = SimpleNamespace()
    s.ids = torch.randint(3, vocab, (B, L + new), generator=g, device="cuda")
    s.mask = s.labels = s.pixels = None
    if case["kind"] in ("train", "encode"):
        keep = torch.arange(L, device="cuda")[None] < lengths_of(case, g)[:, None]
        s.mask = keep.long() if case["padded"] or case["kind"] == "encode" else None
        s.ids = s.ids.masked_fill(~keep, 1)
        s.labels = s.ids.masked_fill(~keep, -100)
    if case["kind"] == "caption":
        s.pixels = torch.rand(B, 3, IMAGE, IMAGE, generator=g, device="cuda").to(BF)
    return s


# ---- the package's side ------------------------------------------------------------------------------

def text_config():
    from vyomai_amd import EncoderConfig
    return EncoderConfig(num_hidden_layers=LAYERS, max_position_embeddings=POSITIONS, hidden_dropout_prob=0.0)


def build(case):
    """The model of a case, on the GPU."""
    import vyomai_amd as V
    kind = case["kind"]
    if kind in ("train", "encode", "serve", "caption"):
        cfg = text_config()
        heads = None
        if case.get("grouped"):
            heads, cfg.num_key_value_heads = "gqa", KV_HEADS
        if kind == "caption":
            from vyomai_amd.shapes import vit_b16_config
            return V.VisionLanguageModel(cfg, V.Vit(vit_b16_config(LAYERS, 0.0)), "rope", None)
        return (V.EncoderModel if kind == "encode" else V.DecoderModel)(cfg, "rope", heads)
    args = dict(vocab=MIX_VOCAB, width=case["width"], layers=mixed_layers(case))
    if kind == "gisitar":
        return V.GisitarModel(V.GisitarConfig(**args))
    if kind == "biruvik":
        return V.BiruvikModel(V.BiruvikConfig(logit_softcap=CAP, **args))
    return V.RivudraModel(V.RivudraConfig(**args))


def prepare(case, seed):
    import vyomai_amd as V
    from vyomai_amd.decode_plan import DecodePlan
    from vyomai_amd.training import FlatTrainer
    kind, g = case["kind"], numbers(case, seed)
    w = weights(case, g)
    s = inputs(case, g)
    s.case, dt = case, next(iter(w.values())).dtype
    before = torch.get_default_dtype()
    torch.set_default_dtype(dt)
    try:
        with torch.device("cuda"):
            s.model = build(case)
    finally:
        torch.set_default_dtype(before)
    if kind in ("train", "caption", "serve"):
        head = "decoder.lm_head." if kind == "caption" else "lm_head."
        w[head + "decoder.bias"] = w[head + "bias"]     # (one tensor under two names)
    s.model.load_state_dict(w)
    if kind in ("train", "caption"):
        s.model.train()
        s.trainer = FlatTrainer(s.model, lr=LR, betas=BETAS, eps=ADAM_EPS, weight_decay=DECAY)
        s.named = {n: p for n, p in s.model.named_parameters() if n in watched(case)}
        return s
    s.model.eval()
    B, total = case["batch"], case["length"] + case.get("new", 0)
    if kind == "serve":
        s.cache = V.StaticCacheOne(s.model.config, max_cache_len=total, batch_size=B, dtype=BF)
        s.plan = DecodePlan(s.model, s.cache, B, BF, torch.device("cuda", torch.cuda.current_device()))
    elif kind != "encode":
        s.cache = s.model.new_cache(B, total)
        s.next_ids = [s.ids[:, i].contiguous() for i in range(case["length"], total)]
        s.prompt = s.ids[:, : case["length"]].contiguous()
    return s


def watched(case):
    """Parameters whose gradients are compared one by one: embeddings, head, and the layers at both ends."""
    ends = ("all_layer.0.", f"all_layer.{LAYERS - 1}.")
    if case["kind"] == "caption":       # (of the first image layer and the last text layer: 64 outputs are the most)
        ends = ("encoder.all_layer.0.", f"decoder.all_layer.{LAYERS - 1}.")
    return {n for n in shapes_of(case) if "all_layer." not in n or any(e in n for e in ends)}


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "train":
        loss = s.trainer.train_step(lambda: s.model.clm_loss(s.ids, s.labels, s.mask))
    elif kind == "caption":
        loss = s.trainer.train_step(lambda: s.model.caption_loss(s.pixels, s.ids))
    if kind in ("train", "caption"):
        return {"loss": loss, "all gradients": s.trainer.arena.grad, "all weights": s.trainer.arena.master,
                "gradient": {n: p.grad for n, p in s.named.items()}}
    with torch.no_grad():
        if kind == "encode":
            return {"states": s.model(s.ids, s.mask).logits}
        B, L, new = case["batch"], case["length"], case["new"]
        if kind == "serve":
            h, _ = s.model.forward_hidden(s.ids[:, :L], None, True, s.cache, 0)
            logits = [s.model.lm_head(h[:, -1:].contiguous())[:, -1]]
            for i in range(L, L + new):
                logits.append(s.plan.step(s.model.word_embeddings(s.ids[:, i]), i)[0])
            return {"states": h, "logits": logits}
        slots = s.cache.allocate(B)
        x = s.model.prefill(s.prompt, [L] * B, s.cache, slots)
        logits = [s.model.logits(x[:, -1])]
        for ids in s.next_ids:
            logits.append(s.model.decode(ids, s.cache, slots))
        s.cache.free(slots)
        return {"stream": x, "logits": logits}


# ---- what a pass cannot do without -------------------------------------------------------------------

def work(case):
    """Every weight a pass needs is read once (a generated token: once more), every input and output moved once.  Matrix products and
    attention count as operations, causal attention by what is visible."""
    kind, B, L, new = case["kind"], case["batch"], case["length"], case.get("new", 0)
    params = {n: math.prod(s) for n, s in shapes_of(case).items()}
    total = sum(params.values())
    looked_up = sum(v for n, v in params.items() if "word_embeddings" in n)
    if kind in ("train", "caption"):
        tokens, pairs = B * L, B * L * (L + 1) / 2
        body = sum(v for n, v in params.items() if "all_layer." in n and not n.startswith("encoder."))
        head = D * D + VOCAB * D
        forward = 2 * tokens * (body + head) + 4 * D * LAYERS * pairs
        if kind == "caption":
            tokens, pairs, seen = B * (L + 1), B * (L + 1) * (L + 2) / 2, PATCHES + 1
            vit = sum(v for n, v in params.items() if n.startswith("encoder.all_layer."))
            forward = 2 * tokens * (body + head) + 4 * D * LAYERS * pairs + 2 * B * seen * vit + 4 * D * LAYERS * B * seen * seen
            forward += 2 * B * PATCHES * D * D * 2 / 3     # (the patches' projection needs no gradient of its input)
        # gradients twice the forward pass; AdamW reads and writes weight and two moments, and reads the gradient, in fp32
        return {"flops": 3 * forward, "bytes": total * (7 * 4 + 2)}
    if kind == "encode":
        return {"flops": 2 * B * L * (total - looked_up) + 4 * D * LAYERS * B * L * L, "bytes": 2 * (total - looked_up) + 4 * B * L * D}
    if kind == "serve":
        kv = 2 * LAYERS * (KV_HEADS * DH if case["grouped"] else D)     # cached numbers per token
        body = sum(v for n, v in params.items() if "all_layer." in n)
        head = total - body - looked_up
        ctx = L * new + new * (new + 1) / 2                             # cached tokens that the generated ones look at
        flops = 2 * B * (L * body + head) + 4 * D * LAYERS * B * L * (L + 1) / 2 + 2 * B * new * (body + head) + 4 * D * LAYERS * B * ctx
        nbytes = 2 * (body + head) * (1 + new) + 2 * B * kv * (L + ctx) + 2 * B * (L * D + (1 + new) * VOCAB)
        return {"flops": flops, "bytes": nbytes}
    w, layers = case["width"], mixed_layers(case)
    H, _, kr = LATENT[w]
    n, head = H * HEAD, params["head.weight"]
    body = total - looked_up - head
    active, used = body, lambda rows: body
    if kind == "rivudra":
        E, top, _, _, ff, _ = EXPERTS[w]
        expert = 3 * w * ff
        active = body - len(layers) * (E - top) * expert
        used = lambda rows: body - len(layers) * (E - min(E, rows * top)) * expert
    flops = 2 * B * L * active + 2 * B * head + 2 * B * new * (active + head)
    nbytes = 2 * (used(B * L) + head) + 2 * (used(B) + head) * new + B * L * w * 4 + 2 * B * (1 + new) * MIX_VOCAB
    for i in range(len(layers)):
        m = layers[i]["mixer"]
        window = m["mask"]["size"] if "mask" in m else None
        for count, first in [(L, 0)] + [(1, L + j) for j in range(new)]:
            seen = sum_seen(first, count, window)
            if layers[i]["type"] in ("hgrn2", "lightning"):
                flops += 4 * B * count * n * HEAD                       # the state's update and its product with the query
                nbytes += 8 * B * n * HEAD                              # the state, fp32, read and written
                continue
            flops += 2 * B * n * seen * (3 if "diff" in m else 2)       # (two maps: of half a head's columns, over whole values)
            rows = first + count if window is None else min(first + count, window)
            width = kr if layers[i]["type"] == "latent_attention" else 2 * n // 4
            nbytes += 2 * B * rows * width
    return {"flops": flops, "bytes": nbytes}


def sum_seen(first, count, window):
    """Pairs of a query (positions first .. first + count - 1) and a key that it sees."""
    if window is None or first + count <= window:
        return count * first + count * (count + 1) / 2
    return sum(min(window, p + 1) for p in range(first, first + count))


def tolerance(case):
    """bf16 storage and products with fp32 sums.  Against 64 bits the package is 0.006 to 0.011 off (states, logits), up to 0.024 on
    gradients and 0.017 where experts are chosen (a token between two of them may take the other one)."""
    loose = case["kind"] in ("train", "caption", "rivudra")
    return {"rel": 0.03, "max": 0.9} if loose else {"rel": 0.025, "max": 0.5}


# ---- the same in 64 bits -----------------------------------------------------------------------------

def exact(case, seed):
    g = numbers(case, seed)
    w = {n: t.to(F64) for n, t in weights(case, g).items()}
    s = inputs(case, g)
    kind, B, L, new = case["kind"], case["batch"], case["length"], case.get("new", 0)
    if kind in ("train", "caption"):
        for t in w.values():
            t.requires_grad_(True)
        if kind == "train":
            h = text_states(w, s.ids, s.mask, True, case["grouped"])
            loss = next_token_loss(w, "lm_head.", h[:, :-1], s.labels[:, 1:])
        else:
            img = image_states(w, s.pixels.to(F64))[:, 0]
            h = text_states(w, s.ids, None, True, False, "decoder.", img)
            loss = next_token_loss(w, "decoder.lm_head.", h[:, 1:-1], s.ids[:, 1:])
        loss.backward()
        return {"loss": loss.detach(), "all gradients": None, "all weights": None, "gradient": {n: w[n].grad for n in watched(case)}}
    with torch.no_grad():
        if kind == "encode":
            return {"states": text_states(w, s.ids, s.mask, False, case["grouped"])}
        if kind == "serve":
            h = text_states(w, s.ids, None, True, case["grouped"])
            return {"states": h[:, :L], "logits": list(vocabulary(w, "lm_head.", h[:, L - 1:]).unbind(1))}
        x = torch.stack([mixed_stream(case, w, ids) for ids in s.ids])
        z = norm(x[:, L - 1:], w["final_norm.weight"], case["kind"]) @ w["head.weight"].T
        z = CAP * torch.tanh(z / CAP) if kind == "biruvik" else z
        return {"stream": x[:, :L], "logits": list(z.unbind(1))}


def affine(w, p, x):
    return F.linear(x, w[p + ".weight"], w.get(p + ".bias"))


def layer_norm(w, p, x):
    return F.layer_norm(x, (D,), w[p + ".weight"], w[p + ".bias"], 1e-5)


def half_turned(x, positions):
    """Rotary positions, column c with column c + half."""
    half = x.shape[-1] // 2
    a = positions[:, None] * 10000.0 ** (-torch.arange(half, device=x.device, dtype=F64) / half)[None]
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)


def text_block(w, p, h, hidden, positions):
    """One layer; hidden: True where a key is not seen."""
    B, L, _ = h.shape
    heads = lambda t: t.view(B, L, -1, DH).transpose(1, 2)
    if p + "attention.qkv.weight" in w:
        q, k, v = (heads(t) for t in affine(w, p + "attention.qkv", h).chunk(3, -1))
    else:
        q, k, v = (heads(affine(w, p + "attention." + n, h)) for n in ("query", "key", "value"))
    if positions is not None:
        q, k = half_turned(q, positions), half_turned(k, positions)
    k, v = (t.repeat_interleave(HEADS // t.shape[1], 1) for t in (k, v))
    z = q @ k.transpose(-1, -2) / math.sqrt(DH)
    if hidden is not None:
        z = z.masked_fill(hidden, -math.inf)
    o = (z.softmax(-1) @ v).transpose(1, 2).reshape(B, L, D)
    a = layer_norm(w, p + "attention.out.layernorm", affine(w, p + "attention.out.dense", o) + h)
    f = affine(w, p + "feed_forward.out", F.gelu(affine(w, p + "feed_forward.intermediate", a)))
    return layer_norm(w, p + "feed_forward.layernorm", f + h)


def text_states(w, ids, mask, causal, grouped, p="", first=None):
    """Last hidden states; first: a vector per row ahead of the tokens."""
    h = w[p + "word_embeddings.weight"][ids]
    if first is not None:
        h = torch.cat([first[:, None], h], 1)
    L = h.shape[1]
    positions = torch.arange(L, device=h.device, dtype=F64)
    hidden = (positions[None] > positions[:, None])[None, None] if causal else None
    if mask is not None:
        pad = (mask == 0)[:, None, None, :]
        hidden = pad if hidden is None else hidden | pad
    for i in range(LAYERS):
        h = text_block(w, f"{p}all_layer.{i}.", h, hidden, positions)
    return h


def image_states(w, pixels):
    p = "encoder."
    x = F.conv2d(pixels, w[p + "pixel_seq.weight"], w[p + "pixel_seq.bias"], stride=PATCH).flatten(2).transpose(1, 2)
    x = torch.cat([w[p + "cls_token"].expand(x.shape[0], -1, -1), x], 1)
    h = 2 * (x + w[p + "position_embeddings.pos_embeddings"])       # (added twice, as the reference does)
    for i in range(LAYERS):
        h = text_block(w, f"{p}all_layer.{i}.", h, None, None)
    return h


def vocabulary(w, p, h):
    return F.linear(layer_norm(w, p + "layer_norm", F.gelu(affine(w, p + "dense", h))), w[p + "decoder.weight"], w[p + "bias"])


def next_token_loss(w, p, h, labels):
    return F.cross_entropy(vocabulary(w, p, h).flatten(0, 1), labels.flatten(), ignore_index=-100)


def norm(x, factor, kind):
    if kind == "gisitar":
        x = x - x.mean(-1, keepdim=True)
    eps = 1e-5 if kind == "gisitar" else 1e-6
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 + factor if kind == "rivudra" else factor)


def rms(x, eps, factor=1.0):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * factor


def mixed_stream(case, w, ids):
    """Residual stream behind the last layer, of one sequence."""
    kind = case["kind"]
    eps = 1e-5 if kind == "gisitar" else 1e-6
    mixers = {"latent_attention": latent_attention, "lightning": lightning, "hgrn2": gated_linear,
              "attention": differential if kind == "biruvik" else window_attention}
    x = w["word_embeddings.weight"][ids]
    for i, layer in enumerate(mixed_layers(case)):
        p = f"layers.{i}."
        v = {n[len(p):]: t for n, t in w.items() if n.startswith(p)}
        h = norm(x, v["norm1.weight"], kind)
        y = mixers[layer["type"]](h, {n[6:]: t for n, t in v.items() if n.startswith("mixer.")}, layer["mixer"], eps)
        if kind == "rivudra":
            x = x + y + mixture(h, v, layer["mlp"])
            continue
        x = x + norm(y, v["norm1b.weight"], kind)
        h = norm(x, v["norm2.weight"], kind)
        up = h @ v["mlp.up.weight"].T
        a = F.silu(h @ v["mlp.gate.weight"].T) * up if kind == "gisitar" else up.clamp(min=0.0) ** 2
        x = x + norm(a @ v["mlp.down.weight"].T, v["norm2b.weight"], kind)
    return x


def attend(q, k, v, scale, window=None, sink=False, step=1024):
    """(heads, tokens, columns) each; query i sees keys up to its own (window: the last so many of them)."""
    T, out = q.shape[1], []
    for lo in range(0, T, step):
        i = torch.arange(lo, min(T, lo + step), device=q.device)
        first = 0 if window is None else max(0, lo - window + 1)
        j = torch.arange(first, int(i[-1]) + 1, device=q.device)
        z = q[:, i] @ k[:, j].transpose(1, 2) * scale
        no = j[None] > i[:, None]
        if window is not None:
            no = no | (j[None] <= i[:, None] - window)
        z = z.masked_fill(no, -math.inf)
        if sink:
            z = torch.cat([z, torch.zeros_like(z[..., :1])], -1).softmax(-1)[..., :-1]
        else:
            z = z.softmax(-1)
        out.append(z @ v[:, j])
    return torch.cat(out, 1)


def heads_of(x, n):
    return x.view(x.shape[0], n, -1).transpose(0, 1)


def flat(x):
    return x.transpose(0, 1).reshape(x.shape[1], -1)


def latent_attention(h, p, cfg, eps):
    H = cfg["heads"]
    if "q_rank" in cfg:
        q = rms(h @ p["q_down.weight"].T, eps, p["q_norm.weight"]) @ p["q_up.weight"].T
    else:
        q = h @ p["query.weight"].T
    c = rms(h @ p["kv_down.weight"].T, eps, p["kv_norm.weight"])
    o = attend(heads_of(q, H), heads_of(c @ p["k_up.weight"].T, H), heads_of(c @ p["v_up.weight"].T, H), cfg["scale"],
               cfg["mask"]["size"] if "mask" in cfg else None)
    gate = torch.sigmoid(h @ p["gate.weight"].T)
    o = flat(o) * gate if "q_rank" in cfg else flat(o * gate.T[:, :, None])
    return o @ p["out.weight"].T


def lightning(h, p, cfg, eps, step=256):
    H, T = cfg["heads"], h.shape[0]
    q, k, v = (heads_of(F.silu(h @ p[n + ".weight"].T), H) for n in ("query", "key", "value"))
    log = torch.tensor(cfg["decay"], dtype=F64, device=h.device).log()[:, None]
    S, out = torch.zeros(H, q.shape[2], v.shape[2], dtype=F64, device=h.device), []
    for lo in range(0, T, step):
        a, b, c = q[:, lo:lo + step], k[:, lo:lo + step], v[:, lo:lo + step]
        i = torch.arange(a.shape[1], device=h.device, dtype=F64)
        apart = (i[:, None] - i[None]).clamp(min=0.0)
        inside = (a @ b.transpose(1, 2)) * torch.exp(log[:, :, None] * apart) * (i[:, None] >= i[None])
        out.append(inside @ c + torch.exp(log * (i + 1))[..., None] * (a @ S))
        S = torch.exp(log * len(i))[..., None] * S + (b * torch.exp(log * (len(i) - 1 - i))[..., None]).transpose(1, 2) @ c
    o = rms(flat(torch.cat(out, 1)), eps, p["norm.weight"])
    return (o * torch.sigmoid(h @ p["gate.weight"].T)) @ p["out.weight"].T


def gated_linear(h, p, cfg, eps):
    H, T = cfg["heads"], h.shape[0]
    q, v = heads_of(F.silu(h @ p["query.weight"].T), H), heads_of(h @ p["value.weight"].T, H)
    low = p["lower"]
    f = heads_of(low + (1.0 - low) * torch.sigmoid(h @ p["forget.weight"].T + p["forget.bias"]), H)
    S, out = torch.zeros(H, q.shape[2], v.shape[2], dtype=F64, device=h.device), torch.empty_like(v)
    for t in range(T):
        S.mul_(f[:, t, :, None]).baddbmm_(1.0 - f[:, t, :, None], v[:, t, None])
        out[:, t] = torch.bmm(q[:, t, None], S)[:, 0]
    return flat(rms(out, eps, p["norm.weight"])) @ p["out.weight"].T


def differential(h, p, cfg, eps):
    H, G, dim, T = cfg["heads"], cfg["kv_heads"], cfg["dim"], h.shape[0]
    q = rms(affine(p, "query", h).view(T, H, 2, dim), eps, p["q_norm.weight"])
    k = rms(affine(p, "key", h).view(T, G, 2, dim), eps, p["k_norm.weight"])
    v = heads_of(affine(p, "value", h), G).repeat_interleave(H // G, 0)
    t = torch.arange(1, T + 1, device=h.device, dtype=F64)
    q = q * (1.0 + TEMP[0] * torch.log(torch.floor(t / TEMP[1]) + 1))[:, None, None, None]
    a = [attend(q[:, :, m].transpose(0, 1), k[:, :, m].transpose(0, 1).repeat_interleave(H // G, 0), v, cfg["scale"]) for m in (0, 1)]
    lam = torch.exp((p["lq1"] * p["lk1"]).sum()) - torch.exp((p["lq2"] * p["lk2"]).sum()) + DIFF
    return flat(rms(a[0] - lam * a[1], eps) * (1.0 - DIFF)) @ p["out.weight"].T


def pair_turned(x, base):
    """Rotary positions, neighbouring columns."""
    i = torch.arange(x.shape[2] // 2, device=x.device, dtype=F64)
    a = torch.arange(x.shape[1], device=x.device, dtype=F64)[:, None] * base ** (-2.0 * i / x.shape[2])[None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1).flatten(2)


def window_attention(h, p, cfg, eps):
    H, G, base = cfg["heads"], cfg["kv_heads"], cfg["rot"]["base"]
    q, k, v = (heads_of(h @ p[n + ".weight"].T, c) for n, c in (("query", H), ("key", G), ("value", G)))
    q, k = pair_turned(q, base), pair_turned(k, base).repeat_interleave(H // G, 0)
    o = attend(q, k, v.repeat_interleave(H // G, 0), cfg["scale"], cfg["mask"]["size"], sink=True)
    return (flat(o) * torch.sigmoid(h @ p["gate.weight"].T)) @ p["out.weight"].T


def clamped(h, gate, up, down):
    g, u = (h @ gate.T).clamp(max=LIMIT), (h @ up.T).clamp(-LIMIT, LIMIT)
    return (g * torch.sigmoid(ALPHA * g) * (u + 1.0)) @ down.T


def mixture(h, v, cfg):
    r = cfg["router"]
    s = (h @ v["mlp.router.weight"].T).softmax(-1)
    groups, size = r["groups"]["count"], r["experts"] // r["groups"]["count"]
    kept = s.view(-1, groups, size).amax(-1).topk(r["groups"]["keep"], -1).indices
    open_ = torch.zeros(s.shape[0], groups, dtype=torch.bool, device=s.device).scatter_(1, kept, True).repeat_interleave(size, 1)
    best = s.masked_fill(~open_, -1.0).topk(r["top"], -1)
    share = best.values / best.values.sum(-1, keepdim=True) * r["scale"]
    y = clamped(h, v["mlp.shared.gate.weight"], v["mlp.shared.up.weight"], v["mlp.shared.down.weight"])
    for e in range(r["experts"]):
        row, place = (best.indices == e).nonzero(as_tuple=True)
        if len(row):
            y[row] += share[row, place, None] * clamped(h[row], v["mlp.gate"][e], v["mlp.up"][e], v["mlp.down"][e])
    return y
