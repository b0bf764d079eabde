"""Differential attention over prompts, heads of 64 and 128 columns in bf16: the two maps' waves meet in the epilogue.  Sizes at the edges
of 32-row waves, 64-key tiles and 128-row workgroups, with a past and with unequal lengths.  Against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("L,start,count", [(2, (0, 0), None), (33, (0, 31), None), (64, (0, 64), (64, 1)), (65, (63, 0), (2, 65)),
                                           (128, (0, 1), None), (129, (127, 0), (129, 33)), (200, (0, 190), (199, 200))])
def test_two_maps(D, L, start, count):
    from vyomai_amd import _lib, ops
    B, h, hk, lam, out_scale, eps = 2, 4, 2, 0.37, 0.6, 1e-5
    R = max(start) + L
    g = torch.Generator().manual_seed(1000 * D + L)
    q, ring = torch.randn(B * L, h * D, generator=g).to(BF), torch.randn(B, hk, R, 2 * D, generator=g).to(BF)
    at = dict(start=torch.tensor(start, dtype=torch.int32, device=DEV), count=None if count is None else torch.tensor(count, dtype=torch.int32, device=DEV))
    scale = (D // 2) ** -0.5
    got = ops.diff_attention(q.to(DEV), B, L, h, hk, D, D, ring.to(DEV), scale, _lib.VyDiff(lam, out_scale, eps, D), at["start"], count=at["count"])
    got = got.double().cpu().view(B, L, h, D)
    for b in range(B):
        n = L if count is None else count[b]
        S = start[b] + n
        seen = torch.arange(S)[None] <= start[b] + torch.arange(n)[:, None]
        for a in range(h):
            k, v = ring[b, a // (h // hk), :S, :D].double(), ring[b, a // (h // hk), :S, D:].double()
            x = q.view(B, L, h, 2, D // 2)[b, :n, a].double()
            p = [(x[:, m] @ k[:, m * (D // 2): (m + 1) * (D // 2)].T * scale).masked_fill(~seen, float("-inf")).softmax(-1) for m in (0, 1)]
            o = p[0] @ v - lam * (p[1] @ v)
            r = (o.square().mean(-1, keepdim=True) + eps).sqrt()
            want = o / r * out_scale
            # the probabilities are rounded to bf16 once: 2^-8 of every term; the norm passes an error e of its columns on as at most
            # max(e) / r (1 + |o| / r), and the result is rounded once more
            e = 2 ** -8 * ((p[0] + lam * p[1]) @ v.abs()).amax(-1, keepdim=True)
            bound = 1.05 * e / r * (1 + o.abs() / r) * out_scale + 2 ** -8 * want.abs() + 1e-6
            assert ((got[b, :n, a] - want).abs() <= bound).all()
