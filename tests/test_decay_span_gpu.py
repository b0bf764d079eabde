"""The chunked linear attention with all value columns in one workgroup (enough chunks for the chip) and with 64 a workgroup: a batch
that takes the former equals its sequences alone, which take the latter, bit by bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("k_scale", [1.0, 0.37])
@pytest.mark.parametrize("dk,dv", [(128, 128), (40, 200), (24, 72), (104, 64), (64, 136)])
def test_a_batch_equals_its_sequences_alone(dk, dv, k_scale):
    from vyomai_amd import ops
    B, H, L = 6, 5, 600                              # 300 chunks together, 50 each
    g = torch.Generator(device=DEV).manual_seed(dk + dv)
    p = torch.randn(B * L, H * (2 * dk + dv) + 8, device=DEV, generator=g).to(BF)
    state = torch.randn(B, H, dk, dv, device=DEV, generator=g)
    start = torch.tensor([0, 3, 700, 0, 1, 2], dtype=torch.int32, device=DEV)
    counts = torch.tensor([600, 1, 599, 64, 130, 513], dtype=torch.int32, device=DEV)
    pw = torch.tensor([[d ** i for i in range(65)] for d in (0.9, 1.0, 0.0, 0.999, 0.5)], device=DEV)
    s = state.clone()
    got = ops.decay_attention(p, H, dk, dv, s, pw, B, L, start=start, count=counts, k_scale=k_scale).view(B, L, -1)
    for b in range(B):
        n = int(counts[b])
        one = state[b:b + 1].clone()
        want = ops.decay_attention(p[b * L:(b + 1) * L], H, dk, dv, one, pw, 1, L, start=start[b:b + 1].contiguous(),
                                   count=counts[b:b + 1].contiguous(), k_scale=k_scale)
        assert torch.equal(got[b, :n], want[:n]) and torch.equal(s[b], one[0])
        assert torch.isfinite(want[:n].float()).all()
