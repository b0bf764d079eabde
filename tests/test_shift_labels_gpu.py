"""Labels of a shifted loss, their count and the logits' padding columns in one launch, against the operations it stands for."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,L,V,ld", [(1, 1, 8, 8), (1, 2, 5, 8), (3, 333, 50257, 50264), (7, 64, 1000, 1000), (1, 1025, 11, 16), (64, 512, 31, 32)])
@pytest.mark.parametrize("layout", ["rows", "columns", "spaced"])
def test_shift_labels(B, L, V, ld, layout):
    from vyomai_amd import ops
    g = torch.Generator().manual_seed(B * L)
    labels = torch.randint(-2, V + 2, (B, L), generator=g)        # (-1, -2, V and V + 1: neither counted nor ignored)
    labels[torch.rand(B, L, generator=g) < 0.3] = -100
    if layout == "columns":
        dev = labels.t().contiguous().to(DEV).t()
    elif layout == "spaced":
        dev = torch.stack((labels, labels + 7), -1).to(DEV)[..., 0]
    else:
        dev = labels.to(DEV)
    buf = torch.full((B * L, ld), 3.0, dtype=torch.bfloat16, device=DEV)
    shifted, acc = ops.shift_labels(dev, -100, buf[:, :V], ld)
    want = torch.full((B, L), -100)
    want[:, :-1] = labels[:, 1:]
    assert torch.equal(shifted.cpu(), want.view(-1))
    counted = ((want != -100) & (want >= 0) & (want < V)).sum()
    assert acc.tolist() == [0.0, float(counted)]
    assert (buf[:, :V] == 3).all() and (buf[:, V:] == 0).all()


@pytest.mark.parametrize("kind", ["int32", "cpu", "one row for all"])
def test_other_labels_take_the_general_way(kind):
    """The loss accepts what indexing accepts: other integers, labels on the host, one row for every sequence."""
    from vyomai_amd.autograd_train import LMHeadLossFn
    g = torch.Generator().manual_seed(1)
    B, L, d, V = 3, 10, 64, 101
    bf = lambda *s: (0.2 * torch.randn(*s, generator=g)).to(torch.bfloat16).to(DEV)
    args = (bf(d, d), bf(d), torch.ones(d, dtype=torch.bfloat16, device=DEV), bf(d), bf(V, d), bf(V), 1e-5)
    h, labels = bf(B, L, d), torch.randint(0, V, (B, L), generator=g)
    if kind == "one row for all":
        labels = labels[:1].expand(B, L).contiguous()
    want = LMHeadLossFn.apply(h, labels.to(DEV), -100, *args)
    other = labels.to(DEV).to(torch.int32) if kind == "int32" else labels if kind == "cpu" else labels[:1].to(DEV)
    got = LMHeadLossFn.apply(h, other, -100, *args)
    assert abs(float(got) - float(want)) <= B * L * 2.0 ** -23 * float(want)       # (positive terms, added up in either order)
