"""Products of 1 to 4 rows that make their operand rows, on workgroups of four, eight and sixteen waves (more of them for wider products): against
fp64, element by element, and the columns of a wide product have the bits of a narrow one's."""
import pytest
import torch

from tests.test_decode_products_gpu import (BF, DEV, FN, GATED, GELU, LAYER, NAN, NONE, QKV, SILU, STORE, STREAM, act_of, entry, f32, few, i32, i64, normed, operands, p, ptr,
                                            rnd, slope, stream, sums, within)

pytestmark = pytest.mark.gpu
PARTS, RMS = 3, 4


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("pro,K,N,act", [(LAYER, 768, 2051, GELU), (LAYER, 1024, 1025, NONE), (STREAM, 1024, 1025, NONE), (STREAM, 1024, 3072, NONE),
                                         (STREAM, 1024, 3089, NONE), (STREAM, 2048, 4101, NONE), (PARTS, 512, 2048, GELU), (PARTS, 512, 3087, GELU),
                                         (PARTS, 768, 3072, GELU), (PARTS, 768, 6147, GELU), (PARTS, 1024, 1031, GELU), (PARTS, 1024, 4096, GELU)])
def test_stored(pro, K, N, act, M):
    if pro == PARTS:
        args = (rnd(M, K, seed=3), rnd(K, seed=4, scale=0.3) + 1, rnd(K, seed=5, scale=0.2), rnd(K // 64, M, K, seed=6, scale=0.3, dtype=torch.float32), K // 64, 0)
        extra = rnd(K, seed=7)
        row = args[3].double().sum(0) + args[0].double() + extra.double()     # (rounded to bf16 ahead of the norm)
        rows, off = normed(row, K, 0, args[1], args[2])
        d = row - row.mean(1, keepdim=True)
        r = (d.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt()
        moved = row.abs() + row.abs().mean(1, keepdim=True) + (d * r).abs() * row.pow(2).mean(1, keepdim=True).sqrt()
        off = off + 2.0 ** -8 * moved * r * args[1].double().abs()
    else:
        (args, _, (rows, off)), extra = operands(pro, K, K - 4 if pro == STREAM else K, 1 if pro == STREAM else 0, M, N), None
    w, bias = rnd(N, K, seed=8, scale=K ** -0.5), rnd(N, seed=9)
    wide = few(STORE, pro, *args, w, N, bias, act, residual=extra)
    within(wide[1], rows, off)
    z, e = sums(wide[1], w)
    z = z + bias.double()
    within(wide[0], act_of(z, act, 0.0), (e + 2.0 ** -23 * z.abs()) * slope(act, z) + FN * z.abs())
    for first, n in ((0, 200), (N - 131, 131)):
        narrow = few(STORE, pro, *args, w[first:first + n].contiguous(), n, bias[first:first + n].contiguous(), act, residual=extra)
        assert torch.equal(wide[0][:, first:first + n], narrow[0])
        assert all(a is None or torch.equal(a, b) for a, b in zip(wide[1:3], narrow[1:3]))


@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("K,N", [(1024, 1030), (1024, 4096), (2048, 3080)])
def test_gated(K, N, M):
    args, _, (rows, off) = operands(STREAM, K, K, 1, M, N)
    w = rnd(2 * N, K, seed=8, scale=K ** -0.5)
    wide = few(GATED, STREAM, *args, w, N, act=SILU)
    within(wide[1], rows, off)
    (gate, eg), (up, eu) = sums(wide[1], w[:N]), sums(wide[1], w[N:])
    eg, eu = eg + 2.0 ** -8 * (gate.abs() + eg), eu + 2.0 ** -8 * (up.abs() + eu)     # both are rounded to bf16 first
    a, ea = act_of(gate, SILU, 0.0), 1.13 * eg + FN * gate.abs()
    within(wide[0], a * up, ea * (up.abs() + eu) + a.abs() * eu)
    narrow = few(GATED, STREAM, *args, torch.cat([w[N - 72:N], w[2 * N - 72:]]), 72, act=SILU)
    assert torch.equal(wide[0][:, -72:], narrow[0]) and torch.equal(wide[2], narrow[2])


@pytest.mark.parametrize("M", [1, 3, 4])
@pytest.mark.parametrize("K,heads,kv", [(768, 12, 12), (1024, 32, 1)])
def test_rotated(K, heads, kv, M):
    """More than 1024 waves: the query columns of the narrow product are the first of the wide one's."""
    args = operands(LAYER, K, K, 0, M, heads)[0]
    N = 64 * (heads + 2 * kv)
    w, bias = rnd(N, K, seed=9, scale=K ** -0.5), rnd(N, seed=10, scale=0.3)
    turn = torch.arange(8, device=DEV, dtype=torch.float32)[:, None] * 10000 ** (-torch.arange(32, device=DEV, dtype=torch.float32) / 32)
    tables = (turn.cos().contiguous(), turn.sin().contiguous())
    q, h, _, k, v = few(QKV, LAYER, *args, w, N, bias, nq=64 * heads, nkv=64 * kv, tables=tables, pos=5)
    z, e = sums(h, w)
    z = z + bias.double()
    within(v, z[:, 64 * (heads + kv):], e[:, 64 * (heads + kv):])
    rows = torch.cat([torch.arange(192), 64 * heads + torch.arange(64), 64 * (heads + kv) + torch.arange(64)]).to(DEV)
    q2, _, _, k2, v2 = few(QKV, LAYER, *args, w[rows].contiguous(), 320, bias[rows].contiguous(), nq=192, nkv=64, tables=tables, pos=5)
    assert torch.equal(q[:, :192], q2) and torch.equal(k[:, :64], k2) and torch.equal(v[:, :64], v2)


@pytest.mark.parametrize("M", [1, 2, 4])
def test_norm_of_a_query_latent_and_the_cache_row_beside_it(M):
    K, N, cap, nkv = 1024, 2051, 9, 512
    x, w, gain, kv, kv_gain = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(K, seed=3, dtype=torch.float32), rnd(M, K, seed=4), rnd(nkv, seed=5, dtype=torch.float32)
    start = torch.arange(3, 3 + M, device=DEV, dtype=torch.int32) % 2
    go = entry("vy_debug_few", i32, i32, p, p, p, p, p, p, i32, i32, f32, p, p, i32, f32, p, p, i64, p, p, i32, i32, p, p, i32, i32, i32, i64, p)

    def product(rows, n):
        y, cache = torch.full((M, n), NAN, dtype=BF, device=DEV), torch.zeros(M, 2, nkv, dtype=BF, device=DEV)
        assert go(STORE, RMS, ptr(x), None, ptr(kv_gain), None, None, None, K, 1, 1e-5, ptr(rows), None, NONE, 0.0, None, ptr(y), n, ptr(cache), ptr(kv), cap, nkv,
                  ptr(start), ptr(gain), 0, M, n, K, stream()) == 0
        torch.cuda.synchronize()
        return y, cache
    (y, cache), (y2, cache2) = product(w, N), product(w[1000:1300].contiguous(), 300)
    assert torch.isfinite(y.float()).all() and torch.equal(y[:, 1000:1300], y2) and torch.equal(cache, cache2)
    row = kv[:, :nkv].double()
    want = row * (row.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt() * kv_gain.double()
    for m in range(M):
        assert ((cache[m, int(start[m])].double() - want[m]).abs() <= 2.0 ** -8 * want[m].abs() + 1e-6).all()
        assert not cache[m, 1 - int(start[m])].any()
