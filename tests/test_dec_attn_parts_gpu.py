"""Decode attention's softmax over keys of any place: contexts at the edges of the register counts (64 keys a pass of 64-wide heads, 32
of 256-wide ones), the largest score in the first, a middle or the last key, keys that weigh nothing, streamed and cached keys, shared
key heads; against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


def check(B, h, hk, S, dh, where, spread=1.0):
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(S + 7 * h + B)
    q = torch.randn(B, h, 1, dh, device=DEV, generator=g).to(BF)
    k, v = (torch.randn(B, hk, S, dh, device=DEV, generator=g) for _ in range(2))
    k = k * spread
    if where is not None:       # keys along the first query of their group: scores of about 8 * dh ** 0.5 there, or far below the others'
        at, size = where
        k[:, :, at] = size * q[:, ::h // hk, 0].float()
    k, v = k.to(BF), v.to(BF)
    got = ops.attention_decode(q, k, v, S).view(B, h, dh).double()
    rep = lambda t: t.double().repeat_interleave(h // hk, 1)
    z = (q.double() @ rep(k).transpose(2, 3).contiguous()) / dh ** 0.5
    want = (z.softmax(-1) @ rep(v)).view(B, h, dh)
    # the result's rounding, and scores of up to 100 in fp32: weights off by 64 * 100 * 2^-24
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -10 * v.double().abs().amax()).all()


@pytest.mark.parametrize("S", [1, 2, 63, 64, 65, 192, 193, 320, 321, 383, 448, 449, 640, 641, 767, 768])
@pytest.mark.parametrize("B,h,hk", [(1, 12, 12), (20, 12, 12), (24, 8, 4), (16, 12, 4), (9, 16, 4)])
def test_heads_of_64(B, h, hk, S):
    check(B, h, hk, S, 64, None, 3.0)
    for at in {0, S // 3, S - 1}:
        check(B, h, hk, S, 64, (at, 8.0))
        check(B, h, hk, S, 64, (at, -8.0))


@pytest.mark.parametrize("S", [1, 32, 33, 160, 161, 224, 225, 320, 321, 384])
@pytest.mark.parametrize("B,h,hk", [(1, 8, 1), (12, 8, 2)])
def test_heads_of_256(B, h, hk, S):
    check(B, h, hk, S, 256, None)
    check(B, h, hk, S, 256, (S - 1, 4.0))


@pytest.mark.parametrize("S", [5, 400, 700])
def test_values_without_a_finite_weight(S):
    """A NaN or an infinite score of the first or the last key: NaN in its head's result, and nowhere else."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(S)
    for at in (0, S - 1):
        for bad in (float("nan"), float("inf")):
            q, k, v = (torch.randn(2, 4, n, 64, device=DEV, generator=g).to(BF) for n in (1, S, S))
            k[1, 2, at, 5] = bad
            out = ops.attention_decode(q, k, v, S).view(2, 4, 64)
            z = (q.float() @ k.float().transpose(2, 3).contiguous())[..., 0, :]
            nan = ~torch.isfinite(z).all(-1) & ~(z == -float("inf")).any(-1)      # (a score of -inf weighs nothing)
            assert torch.equal(torch.isnan(out).all(-1), nan) and torch.equal(torch.isnan(out).any(-1), nan)
