"""The router's logits by lines through LDS, up to 256 tokens and 32, 48 or 64 tokens a workgroup: short last lines and tiles, lines for some waves
only.  The weights of the chosen experts against fp64."""
import pytest
import torch

from tests.test_decode_products_gpu import BF, DEV, rnd, sums

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 17, 256, 257, 4097, 8193, 12300])      # (8193: 48 tokens a workgroup, 12300: 64)
@pytest.mark.parametrize("E,K", [(24, 64), (64, 1160), (70, 520), (130, 72)])
@pytest.mark.parametrize("normalize", [True, False])
def test_chosen_experts(E, K, M, normalize):
    from vyomai_amd.layers.ffn import MixtureFeedForward
    top = 5
    m = MixtureFeedForward(K, E, top, 8, 1.0, normalize=normalize).to(BF).cuda()
    h, w = rnd(M, K, seed=M + E), rnd(E, K, seed=2, scale=2 * K ** -0.5)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(rnd(*p.shape, seed=3, scale=0.1))
        m.router.weight.copy_(w)
    r = m.routed(h)
    ids, weight = r.ids.long(), r.weight.double()
    z, e = sums(h, w)
    e = e.amax(1, keepdim=True)
    p = z.softmax(1)
    want, best = p.topk(top, 1)
    # what is chosen is no more than two errors behind what should be, in each place, and no expert twice
    assert ((z.gather(1, best) - z.gather(1, ids)).abs() <= 2 * e).all()
    assert (ids.sort(1).values.diff(dim=1) > 0).all()
    exact = p.gather(1, ids)
    if normalize:
        exact = exact / exact.sum(1, keepdim=True)
    # exponentials of sums that are e away, in numerator and denominator; a few fp32 functions besides
    assert ((weight - exact).abs() <= exact * (4 * e + 2.0 ** -19)).all()
