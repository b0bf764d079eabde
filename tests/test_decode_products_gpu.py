"""The products of decode steps one by one and element by element, against fp64 on the operands they read: 1 to 4 rows with every prologue
and epilogue (vyomai_amd/csrc/vy_few.hip), 5 to 32 rows with every number of weight rows a workgroup takes and as K slices (vy_rows.hip).
Rows, columns and contractions end inside waves, tiles and slices; everything behind the results' last column must stay as it is."""
import ctypes as C
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV, NAN = torch.bfloat16, "cuda", float("nan")
STORE, QKV, GATED = range(3)
PLAIN, LAYER, STREAM = range(3)
NONE, GELU, GELU_TANH, SILU, RELU2, SOFTCAP = 0, 1, 2, 3, 4, 5
p, i32, i64, f32 = C.c_void_p, C.c_int, C.c_int64, C.c_float


def rnd(*shape, seed, scale=1.0, dtype=BF):
    return (torch.randn(*shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)) * scale).to(dtype)


def ptr(t):
    return None if t is None else t.data_ptr()


def entry(name, *argtypes):
    from vyomai_amd import _lib
    f = getattr(_lib.load(), name)
    f.argtypes, f.restype = list(argtypes), C.c_int
    return f


def stream():
    return torch.cuda.current_stream().cuda_stream


def act_of(v, act, cap):
    if act == GELU:
        return 0.5 * v * (1 + torch.erf(v / math.sqrt(2)))
    if act == GELU_TANH:
        return torch.nn.functional.gelu(v, approximate="tanh")
    if act == SILU:
        return v * torch.sigmoid(v)
    if act == RELU2:
        return v.clamp(min=0) ** 2
    return cap * torch.tanh(v / cap) if act == SOFTCAP else v


def sums(x, w):
    """x w^T and what fp32 sums of its K products may be off by: K roundings of 2^-24 of the sum of magnitudes."""
    x, w = x.double(), w.double().T.contiguous()
    return x @ w, x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs())


def within(got, want, off):
    """bf16 results of values that may be `off` away: half a unit in the last place on top."""
    got = got.double()
    bad = ~((got - want).abs() <= off + 2.0 ** -8 * (want.abs() + off))
    assert not bad.any(), (int(bad.sum()), bad.nonzero()[:4].tolist(), got[bad][:4].tolist(), want[bad][:4].tolist())


def slope(act, v):
    return 2 * v.abs() if act == RELU2 else 1.13      # of the activations; the GELUs' and SiLU's largest is 1.13


# the activations' own arithmetic, fp32 functions of the library and the erf of 7.1.26 (1.5e-7): 2^-18 of the argument at most
FN = 2.0 ** -18


def few(epi, pro, x, a, b, s_in, n, rms, w, N, bias=None, act=NONE, cap=0.0, residual=None, nq=0, nkv=0, tables=(None, None), pos=0):
    M, K = (x if x is not None else s_in).shape
    ldy = (nq if epi == QKV else N) + (0 if epi == QKV else 3)
    y = torch.full((M, ldy), NAN, dtype=BF, device=DEV)
    h = None if pro == PLAIN else torch.full((M, K), NAN, dtype=BF, device=DEV)
    s_out = torch.full((M, K), NAN, device=DEV) if pro == STREAM else None
    k, v = (torch.full((M, max(nkv, 1)), NAN, dtype=BF, device=DEV) for _ in range(2))
    go = entry("vy_debug_few", i32, i32, p, p, p, p, p, p, i32, i32, f32, p, p, i32, f32, p, p, i64, p, p, i32, i32, p, p, i32, i32, i32,
               i64, p)
    rc = go(epi, pro, ptr(x), ptr(a), ptr(b), ptr(s_in), ptr(s_out), ptr(h), n, rms, 1e-5, ptr(w), ptr(bias), act, cap, ptr(residual),
            ptr(y), ldy, ptr(k), ptr(v), nq, nkv, ptr(tables[0]), ptr(tables[1]), pos, M, N, K, stream())
    assert rc == 0, rc
    torch.cuda.synchronize()
    if epi != QKV:
        assert torch.isnan(y[:, N:]).all()
        y = y[:, :N]
    return y, h, s_out, k, v


def normed(v, n, rms, gain, shift):
    """The norm of rows of which the first n columns count, and how far fp32 arithmetic may be from it."""
    v = v.double()
    mean = 0.0 if rms else v[:, :n].sum(1, keepdim=True) / n
    d = v[:, :n] - mean
    r = (d.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt()
    out = torch.zeros_like(v)
    out[:, :n] = d * r * gain.double()[:n] + (shift.double()[:n] if shift is not None else 0.0)
    return out, 2.0 ** -18 * (out.abs() + 1.0)


PRO = [(PLAIN, 1024, 1024, 0), (LAYER, 768, 768, 0), (STREAM, 1024, 1020, 0), (STREAM, 2048, 2048, 1)]


def operands(pro, K, n, rms, M, seed):
    """-> (arguments of few, the fp64 stream and operand rows with what they may be off by)"""
    if pro == PLAIN:
        x = rnd(M, K, seed=seed)
        return (x, None, None, None, n, rms), None, (x, None)
    if pro == LAYER:
        x, g, b = rnd(M, K, seed=seed), rnd(K, seed=seed + 1, scale=0.3) + 1, rnd(K, seed=seed + 2, scale=0.2)
        return (x, g, b, None, n, rms), None, normed(x, n, rms, g, b)
    x, post, pre = rnd(M, K, seed=seed), rnd(K, seed=seed + 1, dtype=torch.float32) * 0.3 + 1, rnd(K, seed=seed + 2, dtype=torch.float32) * 0.3 + 1
    s = rnd(M, K, seed=seed + 3, dtype=torch.float32) * 2
    for t in (x, s):
        t[:, n:] = 0
    post[n:] = pre[n:] = 0
    add, off = normed(x, n, rms, post, None)
    total = s.double() + add
    return (x, post, pre, s, n, rms), (total, off), normed(total, n, rms, pre, None)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("pro,K,n,rms", PRO)
@pytest.mark.parametrize("N,act,extras", [(1003, NONE, "bias"), (1, GELU, "bias residual"), (7, GELU_TANH, ""), (50265, SOFTCAP, ""),
                                          (8205, RELU2, "bias"), (24, NONE, "bias residual")])
def test_few_rows_stored(pro, K, n, rms, M, N, act, extras):
    args, total, (rows, off) = operands(pro, K, n, rms, M, N + M)
    w = rnd(N, K, seed=5, scale=K ** -0.5)
    bias = rnd(N, seed=6, scale=0.5) if "bias" in extras else None
    res = rnd(M, N, seed=7) if "residual" in extras else None
    cap = 3.0 if act == SOFTCAP else 0.0
    y, h, s_out, _, _ = few(STORE, pro, *args, w, N, bias, act, cap, res)
    if total is not None:
        assert ((s_out.double() - total[0]).abs() <= total[1] + 2.0 ** -20 * total[0].abs()).all()
    if h is not None:
        within(h, rows, off)
        rows = h                                    # (what it multiplies: the bits that it wrote)
    want, e = sums(rows, w)
    if bias is not None:
        want = want + bias.double()
    e = (e + 2.0 ** -23 * want.abs()) * slope(act, want.abs() + e) + FN * (want.abs() + want.pow(2) * (act == RELU2))
    want = act_of(want, act, cap)
    if res is not None:
        want = want + res.double()
    within(y, want, e)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K,n,rms", [(1024, 1000, 0), (2048, 2048, 1)])
@pytest.mark.parametrize("N,act", [(1, SILU), (1496, SILU), (13, GELU_TANH), (8194, GELU_TANH)])
def test_few_rows_gated(K, n, rms, M, N, act):
    args, _, (rows, off) = operands(STREAM, K, n, rms, M, N)
    w = rnd(2 * N, K, seed=8, scale=1.5 * K ** -0.5)
    y, h, _, _, _ = few(GATED, STREAM, *args, w, N, act=act)
    within(h, rows, off)
    gate, eg = sums(h, w[:N])
    up, eu = sums(h, w[N:])
    eg, eu = eg + 2.0 ** -8 * (gate.abs() + eg), eu + 2.0 ** -8 * (up.abs() + eu)     # both are rounded to bf16 first
    a, ea = act_of(gate, act, 0.0), 1.13 * eg + FN * gate.abs()
    within(y, a * up, ea * (up.abs() + eu) + a.abs() * eu)


@pytest.mark.parametrize("M", [1, 3, 4])
@pytest.mark.parametrize("pro,K", [(PLAIN, 512), (PLAIN, 1024), (LAYER, 768), (LAYER, 1024)])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("heads,kv", [(12, 4), (1, 1), (16, 2)])
def test_few_rows_rotated(pro, K, heads, kv, M, rope):
    args, _, (rows, off) = operands(pro, K, K, 0, M, heads + M)
    N, pos = 64 * (heads + 2 * kv), 5
    w, bias = rnd(N, K, seed=9, scale=K ** -0.5), rnd(N, seed=10, scale=0.3)
    turn = torch.arange(8, device=DEV, dtype=torch.float32)[:, None] * 10000 ** (-torch.arange(32, device=DEV, dtype=torch.float32) / 32)
    tables = (turn.cos().contiguous(), turn.sin().contiguous()) if rope else (None, None)
    q, h, _, k, v = few(QKV, pro, *args, w, N, bias, nq=64 * heads, nkv=64 * kv, tables=tables, pos=pos)
    if h is not None:
        within(h, rows, off)
        rows = h
    want, e = sums(rows, w)
    want = want + bias.double()
    e = e + 2.0 ** -8 * (want.abs() + e)            # rounded to bf16 ahead of the rotation
    turned = want.view(M, -1, 2, 32).clone()
    te = e.view(M, -1, 2, 32).clone()
    if rope:
        c, s = (t[pos].to(BF).double() for t in tables)
        a, b = (turned[:, : heads + kv, j].clone() for j in (0, 1))
        ea, eb = (te[:, : heads + kv, j].clone() for j in (0, 1))
        # each factor of the sum is rounded once more
        more = 2.0 ** -8 * ((a * c).abs() + (b * s).abs() + (b * c).abs() + (a * s).abs())
        turned[:, : heads + kv, 0], turned[:, : heads + kv, 1] = a * c - b * s, b * c + a * s
        te[:, : heads + kv, 0] = ea * c.abs() + eb * s.abs() + 2 * more
        te[:, : heads + kv, 1] = eb * c.abs() + ea * s.abs() + 2 * more
    within(torch.cat([q, k, v], 1), turned.reshape(M, N), te.reshape(M, N))


@pytest.mark.parametrize("M", [5, 16, 17, 32])
@pytest.mark.parametrize("N,K,act,extras", [(17, 8, NONE, ""), (200, 1000, NONE, "bias"), (1003, 2056, NONE, "bias"),     # 16, 8 waves
                                            (4100, 1032, RELU2, ""), (6139, 200, NONE, "bias"),                          # 24
                                            (8189, 520, SOFTCAP, ""), (8197, 264, NONE, "bias"), (12011, 1032, RELU2, ""),   # 24 / 32, 48
                                            (16101, 520, NONE, ""), (32003, 264, SOFTCAP, "bias")])                      # 24 / 16, 64
def test_rows_of_wide_products(M, N, K, act, extras):
    x, w = rnd(M, K, seed=N), rnd(N, K, seed=12, scale=K ** -0.5)
    bias, cap = rnd(N, seed=13, scale=0.5) if extras else None, 3.0 if act == SOFTCAP else 0.0
    ldy = (N + 7) // 8 * 8 + 8
    y = torch.full((M, ldy), NAN, dtype=BF, device=DEV)
    go = entry("_Z14vy_rows_linearPKvS0_S0_ifPvllllP12ihipStream_t", p, p, p, i32, f32, p, i64, i64, i64, i64, p)
    assert go(ptr(x), ptr(w), ptr(bias), act, cap, ptr(y), ldy, M, N, K, stream()) == 0
    torch.cuda.synchronize()
    assert torch.isnan(y[:, N:]).all()
    want, e = sums(x, w)
    if bias is not None:
        want = want + bias.double()
    e = (e + 2.0 ** -23 * want.abs()) * slope(act, want.abs() + e) + FN * (want.abs() + want.pow(2) * (act == RELU2))
    within(y[:, :N], act_of(want, act, cap), e)


@pytest.mark.parametrize("M", [5, 16, 17, 32])
@pytest.mark.parametrize("N,K,slices", [(512, 1024, 8), (520, 1400, 8), (1000, 6144, 8), (520, 1032, 0), (1024, 1096, 0), (1032, 4104, 4), (2048, 8200, 8), (2001, 8200, 8),
                                        (2048, 1024, 4), (2056, 12288, 2), (4096, 1400, 2), (504, 1024, 0), (4104, 1024, 0),
                                        (1024, 1016, 0)])
def test_rows_in_slices(M, N, K, slices):
    """Every slice by itself: its own columns of the contraction, no others."""
    x, w = rnd(M, K, seed=N), rnd(N, K, seed=14, scale=K ** -0.5)
    parts = torch.full((8 * M * N + 64,), NAN, device=DEV)
    go = entry("_Z13vy_rows_partsPKvS0_PflllP12ihipStream_t", p, p, p, i64, i64, i64, p)
    assert go(ptr(x), ptr(w), ptr(parts), M, N, K, stream()) == slices
    torch.cuda.synchronize()
    assert torch.isnan(parts[slices * M * N:]).all()
    if not slices:
        return
    step = ((K + slices - 1) // slices + 63) // 64 * 64
    for i in range(slices):
        want, e = sums(x[:, i * step:(i + 1) * step], w[:, i * step:(i + 1) * step])
        got = parts[i * M * N:(i + 1) * M * N].view(M, N).double()
        assert ((got - want).abs() <= e).all()


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K,shares,bias", [(512, 1, True), (768, 4, True), (768, 12, False), (1024, 5, True), (1024, 16, True)])
def test_norm_of_a_sum_of_shares(M, K, shares, bias):
    """Operand rows LayerNorm(bf16(shares + bias + x)): the rounding moves a column by 2^-8 of it at most."""
    parts, x, xb = rnd(shares, M, K, seed=K + shares, scale=shares ** -0.5, dtype=torch.float32), rnd(M, K, seed=3), rnd(K, seed=4) if bias else None
    g, b, w, wb = rnd(K, seed=5, scale=0.3) + 1, rnd(K, seed=6, scale=0.2), rnd(205, K, seed=7, scale=K ** -0.5), rnd(205, seed=8)
    y, h, *_ = few(STORE, 3, x, g, b, parts, shares, 0, w, 205, wb, GELU, residual=xb)
    row = parts.double().sum(0) + x.double() + (xb.double() if bias else 0.0)
    want, e = normed(row, K, 0, g, b)
    d = row - row.mean(1, keepdim=True)
    r = (d.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt()
    moved = row.abs() + row.abs().mean(1, keepdim=True) + (d * r).abs() * row.pow(2).mean(1, keepdim=True).sqrt()
    within(h, want, e + 2.0 ** -8 * moved * r * g.double().abs())
    z, ez = sums(h, w)
    z = z + wb.double()
    within(y, act_of(z, GELU, 0.0), (ez + 2.0 ** -23 * z.abs()) * 1.13 + FN * z.abs())


@pytest.mark.parametrize("B,h,hk,S", [(1, 12, 4, 1), (1, 12, 12, 85), (1, 16, 2, 700), (2, 12, 4, 64), (2, 8, 8, 65), (3, 12, 6, 192), (4, 12, 12, 193),
                                      (4, 16, 4, 449), (4, 12, 3, 640), (2, 8, 1, 321), (4, 16, 4, 641), (1, 12, 12, 769)])
def test_attention_into_its_output_projection(B, h, hk, S):
    """The heads' shares of the projection, each by itself; contexts that no kernel holds, and four heads beside long ones, are left to others."""
    d, cap = 64 * h, S + 7
    q, wo = rnd(B, d, seed=S), rnd(d, d, seed=1, scale=d ** -0.5)
    k, v = rnd(B, hk, cap, 64, seed=2), rnd(B, hk, cap, 64, seed=3)
    together = h // hk if B > 1 and 2 <= h // hk <= 4 else 1
    units = h // together
    part = torch.full((units + 1, B, d), NAN, device=DEV)
    go = entry("_Z15vy_dec_attn_outPKvS0_S0_lllS0_PfliiillPKifP12ihipStream_t", p, p, p, i64, i64, i64, p, p, i64, i32, i32, i32, i64, i64, p,
               f32, p)
    n = go(ptr(q), ptr(k), ptr(v), hk * cap * 64, cap * 64, 64, ptr(wo), ptr(part), units * B * d * 4, B, h, hk, S, cap, None, 0.125, stream())
    torch.cuda.synchronize()
    assert n == (0 if S > 768 or (together == 4 and S > 640) else units)
    assert torch.isnan(part[n:]).all()
    assert go(ptr(q), ptr(k), ptr(v), hk * cap * 64, cap * 64, 64, ptr(wo), ptr(part), units * B * d * 4 - 4, B, h, hk, S, cap, None, 0.125, stream()) == 0
    if not n:
        return
    kk, vv = (t[:, :, :S].double().repeat_interleave(h // hk, 1) for t in (k, v))
    qq = q.double().view(B, h, 1, 64)
    score = (qq * kk).sum(-1) * 0.125
    prob = torch.softmax(score, -1)
    o = (prob[..., None] * vv).sum(2)                                     # B, h, 64
    # weights e^s of fp32 scores (64 roundings of 2^-24 of the terms), the result rounded to bf16
    off = 2.0 ** -18 * (1 + (qq.abs() * kk.abs()).sum(-1).amax(-1)[..., None] * 0.125) * (prob[..., None] * vv.abs()).sum(2) + 2.0 ** -8 * o.abs()
    for u in range(units):
        cols = slice(64 * together * u, 64 * together * (u + 1))
        x, e = (t.reshape(B, d)[:, cols] for t in (o, off))
        w = wo.double()[:, cols].T.contiguous()
        bound = e @ w.abs() + 64 * together * 2.0 ** -24 * (x.abs() @ w.abs())
        assert ((part[u].double() - x @ w).abs() <= bound + 1e-30).all()


@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("K,n,np_kv", [(512, 512, 256), (512, 500, 0), (1024, 1024, 8), (1024, 1000, 1024), (1024, 1001, 520)])
def test_rms_norm_of_rows_and_cache_rows_beside_it(M, K, n, np_kv):
    x, g = rnd(M, K, seed=K + n), rnd(K, seed=5, scale=0.3, dtype=torch.float32) + 1
    x[:, n:] = 0
    eye = torch.eye(K, dtype=BF, device=DEV)[: K - 3].contiguous()         # (the products are the operand rows themselves)
    kv = rnd(M, K, seed=7) if np_kv else None                             # (rows of the stride of x; their first np_kv columns)
    gk = rnd(max(np_kv, 1), seed=8, scale=0.3, dtype=torch.float32) + 1
    cache = torch.full((M, 2, np_kv), NAN, dtype=BF, device=DEV) if np_kv else None
    at = torch.tensor([1, 0, 2, 1][:M], dtype=torch.int32, device=DEV)    # (row 2 is past the capacity)
    y = torch.full((M, K - 3), NAN, dtype=BF, device=DEV)
    go = entry("vy_debug_few", i32, i32, p, p, p, p, p, p, i32, i32, f32, p, p, i32, f32, p, p, i64, p, p, i32, i32, p, p, i32, i32, i32, i64, p)
    assert go(STORE, 4, ptr(x), None, ptr(gk), None, None, None, n, 1, 1e-5, ptr(eye), None, NONE, 0.0, None, ptr(y), K - 3, ptr(cache), ptr(kv),
              2, np_kv, ptr(at), ptr(g), 0, M, K - 3, K, stream()) == 0
    torch.cuda.synchronize()
    want, e = normed(x, n, 1, g, None)
    within(y, want[:, : K - 3], e[:, : K - 3] + 2.0 ** -18 * want[:, : K - 3].abs())
    if not np_kv:
        return
    rows, ek = normed(kv[:, :np_kv], np_kv, 1, gk, None)
    for m in range(M):
        for r in (0, 1):
            if r == int(at[m]):
                within(cache[m, r], rows[m], ek[m])
            else:
                assert torch.isnan(cache[m, r]).all()


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K,n,np_kv,ring", [(512, 508, 256, 0), (512, 512, 504, 1), (1024, 1020, 512, 1), (1024, 1024, 1024, 0)])
def test_rms_norm_of_rows_and_slots_of_a_cache(M, K, n, np_kv, ring):
    """Slots that are not the rows' numbers, rings that have turned, three rows (a wave has none)."""
    x, g = rnd(M, K, seed=K + n), rnd(K, seed=5, scale=0.3, dtype=torch.float32) + 1
    x[:, n:] = 0
    eye = torch.eye(K, dtype=BF, device=DEV)
    kv, gk = rnd(M, K, seed=7), rnd(np_kv, seed=8, scale=0.3, dtype=torch.float32) + 1
    cache = torch.full((M, 2, np_kv), NAN, dtype=BF, device=DEV)
    slots = torch.tensor([[0], [1, 0], [2, 0, 1], [3, 1, 0, 2]][M - 1], dtype=torch.int32, device=DEV)
    start = torch.tensor(([5, 2, 8, 3] if ring else [1, 0, 2, 1])[:M], dtype=torch.int32, device=DEV)     # of the slots
    y = torch.full((M, K), NAN, dtype=BF, device=DEV)
    go = entry("vy_debug_few", i32, i32, p, p, p, p, p, p, i32, i32, f32, p, p, i32, f32, p, p, i64, p, p, i32, i32, p, p, i32, i32, i32, i64, p)
    assert go(STORE, 4, ptr(x), None, ptr(gk), None, None, ptr(slots), n, 1, 1e-5, ptr(eye), None, NONE, 0.0, None, ptr(y), K, ptr(cache), ptr(kv),
              -2 if ring else 2, np_kv, ptr(start), ptr(g), 0, M, K, K, stream()) == 0
    torch.cuda.synchronize()
    want, e = normed(x, n, 1, g, None)
    within(y, want, e + 2.0 ** -18 * want.abs())
    rows, ek = normed(kv[:, :np_kv], np_kv, 1, gk, None)
    at = {(int(slots[m]), int(start[slots[m]]) % 2): m for m in range(M) if ring or int(start[slots[m]]) < 2}
    for s in range(M):
        for r in (0, 1):
            if (s, r) in at:
                within(cache[s, r], rows[at[s, r]], ek[at[s, r]])
            else:
                assert torch.isnan(cache[s, r]).all()


def microseconds(launch, n=50):
    """Of a launch among others: the least of several replays of a graph that holds n of them."""
    launch()
    torch.cuda.synchronize()
    graph, best = torch.cuda.CUDAGraph(), float("inf")
    with torch.cuda.graph(graph):
        for _ in range(n):
            launch()
    for _ in range(9):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) / n * 1e3)
    return best


@pytest.mark.parametrize("K", [3072, 4096])
def test_what_four_plain_rows_cost(K):
    """The operand rows are requested together: four of them take 1.3 and 1.4 times what one takes (one trip after the other: 1.9 and
    2.2)."""
    go = entry("vy_debug_few", i32, i32, p, p, p, p, p, p, i32, i32, f32, p, p, i32, f32, p, p, i64, p, p, i32, i32, p, p, i32, i32, i32, i64, p)
    w, y, us = rnd(768, K, seed=1), torch.empty(4, 768, dtype=BF, device=DEV), {}
    for M in (1, 4):
        x = rnd(M, K, seed=M)

        def launch():
            assert go(STORE, PLAIN, ptr(x), None, None, None, None, None, K, 0, 1e-5, ptr(w), None, NONE, 0.0, None, ptr(y), 768, None, None, 0, 0,
                      None, None, 0, M, 768, K, stream()) == 0
        us[M] = microseconds(launch)
    assert us[4] <= 1.7 * us[1], us


@pytest.mark.parametrize("M", [5, 8])
def test_what_the_bias_of_a_wide_product_costs(M):
    """Nothing: it is there before the weights are (converted as it came, ahead of them, it took a tenth of the product's time)."""
    go = entry("_Z14vy_rows_linearPKvS0_S0_ifPvllllP12ihipStream_t", p, p, p, i32, f32, p, i64, i64, i64, i64, p)
    x, w, b, y = rnd(M, 1024, seed=1), rnd(32000, 1024, seed=2), rnd(32000, seed=3), torch.empty(M, 32000, dtype=BF, device=DEV)

    def launch(bias):
        assert go(ptr(x), ptr(w), ptr(bias), NONE, 0.0, ptr(y), 32000, M, 32000, 1024, stream()) == 0
    without, beside = (microseconds(lambda: launch(bias), 20) for bias in (None, b))
    assert beside <= 1.06 * without, (without, beside)
