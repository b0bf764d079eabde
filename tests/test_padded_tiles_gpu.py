"""Key padding that hides whole 64-key tiles: attention and its gradients walk only the tiles between the first and the last visible key, so
they equal the same call on those keys alone, bit by bit, and hidden keys get zero gradients."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("S,first,last", [(500, 0, 3), (500, 3, 5), (512, 0, 1), (512, 7, 8), (320, 2, 4), (64, 0, 1), (130, 2, 3)])
def test_hidden_tiles(dh, S, first, last):
    from vyomai_amd import ops
    B, h, hk, L = 2, 4, 2, 150
    g = torch.Generator().manual_seed(S + first)
    q, k, v, dout = (torch.randn(B, n, t, dh, generator=g).to(BF).to(DEV) for n, t in ((h, L), (hk, S), (hk, S), (h, L)))
    lo, hi = 64 * first, min(64 * last, S)
    keep = torch.zeros(B, S, dtype=torch.uint8)
    keep[:, lo:hi] = torch.rand(B, hi - lo, generator=g) > 0.2
    keep[:, lo] = 1
    keep[1, lo + 1:hi - 1] = 0
    keep[:, hi - 1] = 1
    keep = keep.to(DEV)

    def go(k, v, keep):
        lse = torch.empty(B, h, L, device=DEV)
        out = ops.attention(q, k, v, keypad=keep, lse=lse)
        if dh != 64:
            return (out,)
        do = dout.transpose(1, 2).reshape(B, L, h * dh).contiguous()
        dq, dk, dv = (torch.full_like(t, 7.0) for t in (q, k, v))
        ops.attention_bwd(q, k, v, out, do, lse, dq, dk, dv, causal=False, keypad=keep)
        return out, lse, dq, dk, dv

    got = go(k, v, keep)
    want = go(k[:, :, lo:hi].contiguous(), v[:, :, lo:hi].contiguous(), keep[:, lo:hi].contiguous())
    for a, b in zip(got[:3], want[:3]):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)
    for a, b in zip(got[3:], want[3:]):
        assert torch.equal(a[:, :, lo:hi], b) and not a[:, :, :lo].any() and not a[:, :, hi:].any()


def test_nothing_visible():
    """A sequence without a visible key: the mean over all of its values, and no gradients from it; the one beside it is as alone."""
    from vyomai_amd import ops
    B, h, L, S, dh = 2, 2, 130, 200, 64
    g = torch.Generator().manual_seed(5)
    q, k, v, dout = (torch.randn(B, h, t, dh, generator=g).to(BF).to(DEV) for t in (L, S, S, L))
    keep = torch.ones(B, S, dtype=torch.uint8, device=DEV)
    keep[0] = 0
    lse = torch.empty(B, h, L, device=DEV)
    out = ops.attention(q, k, v, keypad=keep, lse=lse)
    mean = v[0].double().mean(1)                                   # fp32 sums, rounded to bf16 once
    assert ((out[0].double().view(L, h, dh) - mean).abs() <= 2 ** -8 * mean.abs() + 1e-6).all()
    do = dout.transpose(1, 2).reshape(B, L, h * dh).contiguous()
    grads = [torch.full_like(t, 7.0) for t in (q, k, v)]
    ops.attention_bwd(q, k, v, out, do, lse, *grads, causal=False, keypad=keep)
    assert not any(t[0].any() for t in grads)
    lse1 = torch.empty(1, h, L, device=DEV)
    assert torch.equal(ops.attention(q[1:], k[1:], v[1:], keypad=keep[1:], lse=lse1), out[1:]) and torch.equal(lse1, lse[1:])
