"""Projections of the text decoder's steps (vyomai_amd/csrc/vy_decode.hip) one by one, against fp64: a row count that leaves groups of 8
rows out, row blocks together or by themselves, one or two column blocks a workgroup, each number of k-steps a wave.  Rows give the same
bits in every form."""
import pytest
import torch

from tests.test_decode_products_gpu import BF, DEV, FN, GELU, NAN, NONE, act_of, entry, f32, i32, i64, p, ptr, rnd, stream, sums, within

pytestmark = pytest.mark.gpu


def linear_ex(x, w, bias, residual, gain, shift, eps, act):
    M, (N, K) = x.shape[0], w.shape
    y = torch.full((M, N + 8), NAN, dtype=BF, device=DEV)
    go = entry("_Z16vy_dec_linear_exPKviS0_S0_S0_iS0_S0_fPviiiiiP12ihipStream_t", p, i32, p, p, p, i32, p, p, f32, p, i32, i32, i32, i32, i32, p)
    assert go(ptr(x), x.stride(0), ptr(w), ptr(bias), ptr(residual), N, ptr(gain), ptr(shift), eps, ptr(y), N + 8, M, N, K, act, stream()) == 0
    torch.cuda.synchronize()
    assert torch.isnan(y[:, N:]).all()
    return y[:, :N]


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("K", [512, 768, 1024])
@pytest.mark.parametrize("N", [16, 768, 2048, 2064, 3072])     # (two row blocks of 128 column blocks and fewer: by themselves)
def test_rows(N, K, norm):
    full = rnd(32, K + 16, seed=N + K)
    w, bias, residual = rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3, scale=0.5), None if norm else rnd(32, N, seed=4)
    gain, shift = (rnd(K, seed=5), rnd(K, seed=6, scale=0.3)) if norm else (None, None)
    act = GELU if norm else NONE
    parts = [linear_ex(full[a:b, :K], w, bias, None if norm else residual[a:b], gain, shift, 1e-5, act) for a, b in [(0, 1), (1, 9), (9, 25), (25, 32)]]
    whole = torch.cat(parts)
    for M in (8, 16, 17, 24, 32):
        assert torch.equal(linear_ex(full[:M, :K], w, bias, residual, gain, shift, 1e-5, act), whole[:M]), M
    x = full[:, :K].double()
    extra = 0
    if norm:
        x = (x - x.mean(1, keepdim=True)) / (x.var(1, unbiased=False, keepdim=True) + 1e-5).sqrt() * gain.double() + shift.double()
        near = x.to(BF)
        extra = 2.0 ** -7 * near.abs().double() @ w.double().abs().T.contiguous()    # (a value beside a rounding edge may go the other way)
        x = near
    want, e = sums(x, w)
    want, e = want + bias.double(), e + extra + 2.0 ** -23 * want.abs()
    out = act_of(want, act, 0) + (0 if norm else residual.double())
    within(whole, out, 1.13 * e + FN * want.abs() + 2.0 ** -23 * out.abs())


@pytest.mark.parametrize("heads,kv", [(8, 2), (12, 12), (16, 4)])
@pytest.mark.parametrize("rope", [True, False])
def test_rotated_rows(heads, kv, rope):
    K, N, cap = 64 * heads, 64 * (heads + 2 * kv), 5
    x, w, bias = rnd(32, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3, scale=0.5)
    angle = torch.arange(8, device=DEV, dtype=torch.float32)[:, None] * 10000 ** (-torch.arange(32, device=DEV, dtype=torch.float32) / 32)
    cos, sin = angle.cos().contiguous(), angle.sin().contiguous()
    go = entry("_Z10vy_dec_qkvPKvS0_S0_PKfS2_lPKiPvS5_S5_llliiiiP12ihipStream_t", p, p, p, p, p, i64, p, p, p, p, i64, i64, i64, i32, i32, i32, i32, p)

    def run(rows):
        M = rows.shape[0]
        q = torch.full((M, K), NAN, dtype=BF, device=DEV)
        k, v = (torch.full((M, kv, cap, 64), NAN, dtype=BF, device=DEV) for _ in range(2))
        at = torch.tensor([3], dtype=torch.int32, device=DEV)
        assert go(ptr(rows), ptr(w), ptr(bias), ptr(cos) if rope else None, ptr(sin) if rope else None, 0, ptr(at), ptr(q), ptr(k), ptr(v), kv * cap * 64,
                  cap * 64, 64, M, K, heads, kv, stream()) == 0
        torch.cuda.synchronize()
        for c in (k, v):
            assert torch.isnan(c[:, :, [0, 1, 2, 4]]).all()
        return torch.cat([q, k[:, :, 3].reshape(M, -1), v[:, :, 3].reshape(M, -1)], 1)

    whole = torch.cat([run(x[a:b].contiguous()) for a, b in [(0, 1), (1, 9), (9, 25), (25, 32)]])
    for M in (8, 16, 17, 24, 32):
        assert torch.equal(run(x[:M].contiguous()), whole[:M]), M
    want, e = sums(x, w)
    want, e = want + bias.double(), e + 2.0 ** -23 * want.abs()
    if rope:
        t, n = want.view(32, -1, 64), heads + kv
        c, s = cos[3].to(BF).double(), sin[3].to(BF).double()
        a, b = t[:, :n, :32], t[:, :n, 32:]
        want = torch.cat([torch.cat([a * c - b * s, b * c + a * s], 2), t[:, n:]], 1).reshape(32, -1)
        # both factors and both products are rounded to bf16 ahead of the last rounding
        size = torch.cat([torch.cat([a.abs() + b.abs()] * 2, 2), t[:, n:].abs()], 1).reshape(32, -1)
        e = 2 * e.view(32, -1, 64).amax(2, keepdim=True).expand(-1, -1, 64).reshape(32, -1) + 2.0 ** -7 * size
    within(whole, want, e)


@pytest.mark.parametrize("K", [256, 512, 768, 1024, 3072])
@pytest.mark.parametrize("N", [64, 768])
def test_parts_and_norm(N, K):
    x, w, bias, residual = rnd(32, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3, scale=0.5), rnd(32, N, seed=4)
    gain, shift = rnd(N, seed=5), rnd(N, seed=6, scale=0.3)
    go = entry("_Z20vy_dec_linear_res_lnPKviS0_S0_S0_iS0_S0_fPviPfiiiiP12ihipStream_t", p, i32, p, p, p, i32, p, p, f32, p, i32, p, i32, i32, i32, i32, p)

    def run(a, b):
        part = torch.full((24, 32, N), NAN, device=DEV)
        y = torch.full((b - a, N + 8), NAN, dtype=BF, device=DEV)
        assert go(ptr(x[a:b]), K, ptr(w), ptr(bias), ptr(residual[a:b]), N, ptr(gain), ptr(shift), 1e-5, ptr(y), N + 8, ptr(part), b - a, N, K, NONE, stream()) == 0
        torch.cuda.synchronize()
        assert torch.isnan(y[:, N:]).all()
        return y[:, :N]

    whole = torch.cat([run(a, b) for a, b in [(0, 1), (1, 9), (9, 25), (25, 32)]])
    for M in (8, 16, 17, 24, 32):
        assert torch.equal(run(0, M), whole[:M]), M
    want, e = sums(x, w)
    want = want + bias.double() + residual.double()
    e = (e + 2.0 ** -8 * want.abs() + 2.0 ** -22 * want.abs()).amax(1, keepdim=True)
    sd = (want.var(1, unbiased=False, keepdim=True) + 1e-5).sqrt()
    z = (want - want.mean(1, keepdim=True)) / sd
    # |dz| of a change of at most e in each value: (2 + |z|) e / sd
    within(whole, z * gain.double() + shift.double(), gain.double().abs() * (2 + z.abs()) * e / sd + 2.0 ** -20)
