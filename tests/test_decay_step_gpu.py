"""One token of the linear attentions, 16 bytes of state a lane, against the kernel with a column a lane, which takes states that are not
aligned to 16 bytes: the same new states bit by bit, outputs that differ by the order of one sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("dt", [BF, torch.float32])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("dk,dv", [(8, 8), (64, 32), (72, 40), (128, 128), (136, 72), (256, 200)])
def test_both_kernels(dk, dv, gated, dt):
    from vyomai_amd import ops
    B, h, slots = 3, 2, 5
    g = torch.Generator(device=DEV).manual_seed(dk + dv)
    rand = lambda *n: torch.randn(*n, generator=g, device=DEV)
    p, held = rand(B, h * (2 * dk + dv)).to(dt), rand(slots * h * dk * dv + 4)
    held[4 + h * dk * dv:][:8] = float("nan")                       # slot 1 is empty: whatever lies there
    start = torch.tensor([3, 0, 700, 9, 1], dtype=torch.int32, device=DEV)
    at = dict(start=start, slots=torch.tensor([4, 1, 2], dtype=torch.int32, device=DEV), count=torch.tensor([1, 1, 0], dtype=torch.int32, device=DEV))
    lower, bias = torch.rand(h * dk, generator=g, device=DEV), rand(h * dk)
    powers = torch.tensor([[d ** i for i in range(65)] for d in (0.9, 0.99)], device=DEV)
    half = min(dk, 64) // 2
    rotary = rand(800, half, 2)

    def go(offset):
        s = torch.empty(held.numel(), device=DEV)
        state = s[offset:offset + slots * h * dk * dv].view(slots, h, dk, dv)
        state.copy_(held[4:].view_as(state))
        assert state.data_ptr() % 16 == 4 * offset
        o = ops.gated_attention(p, h, dk, dv, state, lower, bias, B, 1, **at) if gated else \
            ops.decay_attention(p, h, dk, dv, state, powers, B, 1, rotary=rotary, k_scale=0.37, **at)
        return o.float(), state

    (got, new), (want, old) = go(0), go(1)
    assert torch.equal(new.nan_to_num(7.0), old.nan_to_num(7.0))
    assert torch.isfinite(new[[1, 2, 4]]).all() and not got[2].any() and torch.isfinite(got).all()
    # sums of dk products in another order, 2^-24 each of at most the sum of their sizes (|q| < 10 and a rotation's factor), and a rounding
    size = 40 * new[[4, 1, 2]].abs().sum(2).reshape(B, h * dv)
    eps = 2 ** -8 if dt == BF else 2 ** -24
    assert ((got - want).abs() <= 2 ** -24 * dk * size + eps * want.abs() + 1e-9).all()
