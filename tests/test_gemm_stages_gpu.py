"""Products on the 256-row, 224-row and 160-row tiles: one to five stages of K, short last ones, and the order in which an XCD walks tiles
of many columns (strips of row panels of equal and unequal height), against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16


def check(M, N, K, seed):
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).to(BF)
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF)
    y = torch.full((M, N), 7.0, dtype=BF, device=DEV)
    ops.linear(x, w, out=y)
    # half an ulp of a bf16 result (2^-9), twice where it lies at a power of two, and the fp32 sum's own error
    bound = 2.0 ** -8 * (x.double() @ w.double().T).abs() + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30
    worst = ((y.double() - x.double() @ w.double().T).abs() / bound).max()
    assert worst <= 1, float(worst)


@pytest.mark.parametrize("K", [8, 56, 64, 72, 128, 136, 192, 200, 256, 264, 320])
@pytest.mark.parametrize("M,N", [(4096, 4096), (12600, 768), (5000, 1536), (8000, 1032), (6000, 3072), (4200, 2048)])
def test_few_stages(M, N, K):
    check(M, N, K, K)


# column tiles 16 to 65, W up to and beyond what stays near L2, row panels in strips of 6, of 5 and 6, of 1
@pytest.mark.parametrize("M,N,K", [(1665, 4096, 2048), (2500, 5128, 72), (6300, 4100, 264), (200, 16384, 1032), (4608, 16384, 200),
                                   (3333, 8200, 1600), (2600, 16640, 64), (1111, 16392, 520)])
def test_strips_of_row_panels(M, N, K):
    check(M, N, K, N)
