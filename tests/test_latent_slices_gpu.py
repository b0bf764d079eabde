"""Latent decode where the key range is cut: one tile of keys a slice up to 64 slices, two and more tiles beyond, empty slices of the shorter
sequence, more slices than one batch of loads.  Against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("gate_heads", [False, True])
@pytest.mark.parametrize("R", [64, 256, 512])
@pytest.mark.parametrize("keys", [(1,), (64, 1), (65, 64), (33, 2048), (2049, 130), (4096, 4097), (4160, 8000)])
def test_slices(keys, R, gate_heads):
    from vyomai_amd import ops
    B, h, dh, dv, scale = len(keys), 3, 64, 72, 0.05
    g = torch.Generator().manual_seed(sum(keys) + R)
    q, wk, wv = (torch.randn(*n, generator=g).to(BF) for n in ((B, h * dh), (h, R, dh), (h, dv, R)))
    wk = (wk * 0.1).to(BF)
    cache, gate = torch.randn(B, max(keys), R, generator=g).to(BF), torch.randn(B, 8 if gate_heads else h * dv, generator=g).to(BF)
    got = ops.latent_decode(q.to(DEV), wk.to(DEV), wv.to(DEV), cache.to(DEV), torch.tensor(keys, dtype=torch.int32, device=DEV) - 1, max(keys), scale,
                            gate=gate.to(DEV), gate_heads=gate_heads).double().cpu().view(B, h, dv)
    for b, n in enumerate(keys):
        c = cache[b, :n].double()
        for a in range(h):
            qa = q[b, a * dh:(a + 1) * dh].double()
            ql = wk[a].double() @ qa
            p = (c @ ql * scale).softmax(0)
            s = torch.sigmoid(gate[b, a].double() if gate_heads else gate[b, a * dv:(a + 1) * dv].double())
            want = wv[a].double() @ (p @ c) * s
            size = wv[a].double().abs() @ (p @ c.abs()) * s
            # latent queries as two bf16 halves: 2^-16 of every term of a score, an error of the exponent; weights and result are rounded
            # to bf16 once each
            d = 2 * scale * 2 ** -16 * (c.abs() @ (wk[a].double().abs() @ qa.abs())).max()
            assert ((got[b, a] - want).abs() <= (1.02 * 2 ** -8 + 2 * d) * size + 2 ** -8 * want.abs() + 1e-6).all(), (b, a)
