"""The experts' products of many tokens on their two tile sizes: experts without a row, with one, with a whole tile and with one row
more, contractions and outputs that end inside a stage and a tile, against the same products in fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("act", ["clamped", "gelu"])
@pytest.mark.parametrize("width,ff", [(136, 200), (1096, 1032)])
@pytest.mark.parametrize("counts", [[0, 1, 128, 129], [190, 190, 190, 197], [0, 1, 256, 511], [257, 700, 64, 65], [0, 1, 9000, 257]])
def test_rows_of_uneven_experts(act, width, ff, counts):
    """One expert per token, forced by the token's first columns.  A row's activations and its outputs are rounded to bf16 (half a unit in the
    last of 8 bits: at most 2^-8 of the value), the sums are fp32."""
    from vyomai_amd.layers.ffn import MixtureFeedForward
    E, M = len(counts), sum(counts)
    g = torch.Generator().manual_seed(M + width)
    more = {} if act == "clamped" else {"act": "gelu", "score": "sigmoid", "group_best": 1}
    m = MixtureFeedForward(width, E, 1, ff, 1.5 if act == "clamped" else 0.0, **more).to(BF).cuda()
    with torch.no_grad():
        m.router.weight.zero_()
        m.router.weight[:, :E] = 8.0 * torch.eye(E)
        for n in (("gate",) if act == "clamped" else ()) + ("up", "down"):
            p = getattr(m, n)
            p.copy_(torch.randn(p.shape, generator=g) / p.shape[-1] ** 0.5)
    want_ids = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(M, generator=g)]
    h = torch.randn(M, width, generator=g)
    h[:, :E] = torch.nn.functional.one_hot(want_ids, E).float()
    h = h.to(BF)
    weights = {n: getattr(m, n).detach().double().cpu() for n in ("gate", "up", "down") if getattr(m, n, None) is not None}
    r = m.routed(h.cuda())
    assert r.ids.cpu()[:, 0].tolist() == want_ids.tolist()
    pos = r.pos.cpu()[:, 0].long()
    assert sorted(pos.tolist()) == list(range(M))
    rows = r.rows.double().cpu()[pos]
    for e in range(E):
        x = h[want_ids == e].double()
        u = x @ weights["up"][e].T
        if act == "clamped":
            gate = (x @ weights["gate"][e].T).clamp(max=1.5)
            a = gate * torch.sigmoid(1.702 * gate) * (u.clamp(-1.5, 1.5) + 1)
        else:
            a = torch.nn.functional.gelu(u)
        want = a @ weights["down"][e].T
        bound = 2.0 ** -8 * (a.abs() @ weights["down"][e].abs().T + want.abs()) * 1.01 + 1e-4
        assert ((rows[want_ids == e] - want).abs() <= bound).all(), e
