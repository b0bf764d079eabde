"""Values of latent decode: 16 and 64 value columns a workgroup (64 workgroups of 64 columns are the line between them), several sequences a
workgroup, latents and values that end inside lines and blocks.  Rows are the same whatever else is in the batch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("R", [8, 64, 72, 248, 264, 512])
@pytest.mark.parametrize("dv", [8, 64, 72, 136])
def test_batches(dv, R):
    from vyomai_amd import ops
    h, dh, keys, scale, B = 5, 64, 70, 0.05, 300       # (rows 0 .. 4 of 5 heads and two column blocks are 50 workgroups)
    g = torch.Generator().manual_seed(R + dv)
    q, wk, wv = (torch.randn(*n, generator=g).to(BF) for n in ((B, h * dh), (h, R, dh), (h, dv, R)))
    wk = (wk * 0.1).to(BF)
    cache, gate = torch.randn(B, keys, R, generator=g).to(BF), torch.randn(B, h * dv, generator=g).to(BF)

    def run(n):
        return ops.latent_decode(q[:n].to(DEV), wk.to(DEV), wv.to(DEV), cache[:n].to(DEV), torch.full((n,), keys - 1, dtype=torch.int32, device=DEV), keys, scale,
                                 gate=gate[:n].to(DEV)).cpu()

    whole = run(B)
    for n in (1, 5, 16, 100):
        # (the number of key slices falls with the batch: sums of one slice or two)
        assert (run(n).double() - whole[:n].double()).abs().max() <= 2 ** -6 * whole[:n].double().abs().max(), n
    got = whole.double().view(B, h, dv)
    for b in (0, 7, B - 1):
        c = cache[b].double()
        for a in range(h):
            qa = q[b, a * dh:(a + 1) * dh].double()
            p = (c @ (wk[a].double() @ qa) * scale).softmax(0)
            s = torch.sigmoid(gate[b, a * dv:(a + 1) * dv].double())
            want = wv[a].double() @ (p @ c) * s
            size = wv[a].double().abs() @ (p @ c.abs()) * s
            # latent queries as two bf16 halves: 2^-16 of every term of a score; weights and result are rounded to bf16 once each
            d = 2 * scale * 2 ** -16 * (c.abs() @ (wk[a].double().abs() @ qa.abs())).max()
            assert ((got[b, a] - want).abs() <= (1.02 * 2 ** -8 + 2 * d) * size + 2 ** -8 * want.abs() + 1e-6).all(), (b, a)
