"""Steps of 5 to 32 sequences through the sublayers' output products that leave their sums in slices: widths and batches at the edges of
the rule that takes them (one slice short of it, ragged last slices, a last tile of 8 columns), against the products and norms one by
one in fp64."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


def model(width, ff, heads, dim):
    from vyomai_amd import GisitarConfig, GisitarModel
    lig = {"type": "lightning", "mixer": {"heads": heads, "dim": dim, "vdim": dim, "decay": [0.9] * heads}, "mlp": {"kind": "dense", "ff": ff}}
    torch.manual_seed(width + ff)
    with torch.device(DEV):
        torch.set_default_dtype(BF)
        try:
            m = GisitarModel(GisitarConfig(vocab=200, width=width, layers=[lig, lig]))
        finally:
            torch.set_default_dtype(torch.float32)
    return m.eval()


@pytest.mark.parametrize("B", [4, 5, 16, 17, 32, 33])
@pytest.mark.parametrize("width,ff,heads,dim", [(1024, 1024, 8, 128), (520, 1032, 8, 128), (1000, 2200, 9, 120), (2048, 1016, 8, 128),
                                                (2056, 3000, 8, 136)])
def test_a_step_equals_the_same_rows_as_a_prompt(B, width, ff, heads, dim):
    """A batch's next token through the step and through the prompt path (other product and norm kernels): the logits agree within
    bf16 roundings of the sublayers' inputs, 2^-9 relative each, two sublayers and a norm per layer and a vocabulary product."""
    m = model(width, ff, heads, dim)
    ids = torch.randint(0, 200, (B, 4), device=DEV, generator=torch.Generator(device=DEV).manual_seed(B))
    got, want = [], []
    cache = m.new_cache(B, 8)
    slots = cache.allocate(B)
    m.prefill(ids[:, :2].contiguous(), [2] * B, cache, slots)
    for t in (2, 3):
        got.append(m.decode(ids[:, t].contiguous(), cache, slots))
        other = m.new_cache(B, 8)
        s = other.allocate(B)
        x = m.prefill(ids[:, :t + 1].contiguous(), [t + 1] * B, other, s)
        want.append(m.logits(x[:, -1]))
    for a, b in zip(got, want):
        a, b = a.double(), b.double()
        assert torch.isfinite(a).all()
        assert (a - b).norm() <= 24 * 2.0 ** -9 * b.norm(), float((a - b).norm() / b.norm())


@pytest.mark.parametrize("B", [5, 16, 17, 32])
@pytest.mark.parametrize("ff", [1400, 2603, 4096, 5203, 8003])
def test_a_step_through_wide_products(B, ff):
    """[gate; up] products of 2800 to 16016 columns: 16, 24, 32, 48 and 64 weight rows a workgroup, the last ones ragged."""
    test_a_step_equals_the_same_rows_as_a_prompt(B, 520, ff, 8, 128)
