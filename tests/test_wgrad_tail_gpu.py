"""Weight gradients whose 256 x 256 tiles end in a partly filled round, cut in two along the rows: against fp64, and twice the same."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("M,N,K", [(4096, 22016, 768), (4129, 32760, 712), (4500, 50265, 776), (4097, 8200, 2056), (4200, 70000, 256)])
def test_against_fp64(M, N, K, accumulate):
    """258, 384, 788, 297 and 274 tiles: remainders of 2 and 128 (both cut), 20 (of 4 columns), 41 and 18.  Sums of M products in fp32,
    at most M rounding errors of 2^-24 of the sum of their magnitudes."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(N)
    dy = torch.randn(M, (N + 7) // 8 * 8, device=DEV, generator=g).to(BF)[:, :N]
    x = torch.randn(M, K, device=DEV, generator=g).to(BF)
    got = []
    for _ in range(2):
        dw = torch.full((N, K), 0.5 if accumulate else 7.0, device=DEV)
        db = torch.full((N,), -0.25 if accumulate else 7.0, device=DEV)
        ops.linear_wgrad(dy, x, dw, db, accumulate)
        got.append((dw, db))
    (dw, db), (dw2, db2) = got
    if not accumulate:   # two contributions to zero: in either order the same sum
        assert torch.equal(dw, dw2)
    for n0 in range(0, N, 8192):
        d = dy[:, n0:n0 + 8192].double()
        want = d.T.contiguous() @ x.double() + (0.5 if accumulate else 0.0)
        size = d.abs().T.contiguous() @ x.double().abs() + 1.0
        assert ((dw[n0:n0 + 8192].double() - want).abs() <= M * 2.0 ** -24 * size).all()
        assert ((db[n0:n0 + 8192].double() - d.sum(0) - (-0.25 if accumulate else 0.0)).abs() <= M * 2.0 ** -24 * (d.abs().sum(0) + 1.0)).all()
