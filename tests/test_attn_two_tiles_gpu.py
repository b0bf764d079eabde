"""Attention over heads of 128 bf16 columns (two K/V tiles of 64 keys in LDS) where its ring can go wrong: no, one, two and more tiles
of keys, a last tile with one key, with the masks that change which tiles a workgroup walks.  Against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("mask", ["none", "causal", "keypad", "causal+keypad", "add"])
@pytest.mark.parametrize("L,S", [(1, 1), (33, 64), (128, 65), (129, 128), (130, 129), (64, 192), (257, 321)])
def test_tiles_of_keys(L, S, mask):
    from vyomai_amd import ops
    B, h, hk, dh = 2, 4, 2, 128
    g = torch.Generator().manual_seed(S * 1000 + L)
    q, k, v = (torch.randn(B, n, t, dh, generator=g).to(BF) for n, t in ((h, L), (hk, S), (hk, S)))
    start = max(0, S - L)
    kw, seen = {}, torch.ones(B, 1, L, S, dtype=torch.bool)
    if "causal" in mask:
        kw.update(causal=True, start_pos=start)
        seen = seen & (torch.arange(S)[None, :] <= start + torch.arange(L)[:, None])
    if "keypad" in mask:
        keep = torch.rand(B, S, generator=g) > 0.3
        keep[:, 0] = True                                    # (every row sees a key)
        keep[1, 1:max(1, S - 1)] = False                     # whole tiles without one
        kw["keypad"] = keep.to(torch.uint8).to(DEV)
        seen = seen & keep[:, None, None, :]
    add = torch.zeros(B, 1, L, S)
    if mask == "add":
        add = torch.randn(B, 1, L, S, generator=g)
        kw["addmask"] = add.to(DEV)
    got = ops.attention(q.to(DEV), k.to(DEV), v.to(DEV), **kw).double().cpu()
    kd, vd = (t.double().repeat_interleave(h // hk, 1) for t in (k, v))
    s = (q.double() @ kd.transpose(2, 3)) * dh ** -0.5 + add.double()
    p = torch.softmax(s.masked_fill(~seen, float("-inf")), -1)
    want, size = p @ vd, p @ vd.abs()
    flat = lambda t: t.transpose(1, 2).reshape(B, L, h * dh)
    # the probabilities and the result are rounded to bf16 once each: 2^-8 of every term and of the sum; the scores' fp32 error is a
    # hundredth of that
    assert ((got - flat(want)).abs() <= 2.02 * 2 ** -8 * flat(size) + 1e-6).all()
