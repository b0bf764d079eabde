"""Weight gradients whose 256 x 256 tiles end in a partly filled round, which goes out in quarters of 128 x 128: against fp64, twice
the same whatever the gradient held before, and the bits of whole tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("M,N,K", [(4096, 22016, 768), (4129, 32760, 712), (4500, 50265, 776), (4097, 8200, 2056), (4200, 70000, 256)])
def test_against_fp64(M, N, K, accumulate):
    """258, 384, 788, 297 and 274 tiles: remainders of 2 and 128, 20 (of 4 tiles a row, the last 8 columns wide), 41 and 18.  Sums of M
    products in fp32, at most M rounding errors of 2^-24 of the sum of their magnitudes."""
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
    assert torch.equal(dw, dw2) and torch.equal(db, db2)   # one contribution an element
    for n0 in range(0, N, 8192):
        d = dy[:, n0:n0 + 8192].double()
        want = d.T.contiguous() @ x.double() + (0.5 if accumulate else 0.0)
        size = d.abs().T.contiguous() @ x.double().abs() + 1.0
        assert ((dw[n0:n0 + 8192].double() - want).abs() <= M * 2.0 ** -24 * size).all()
        assert ((db[n0:n0 + 8192].double() - d.sum(0) - (-0.25 if accumulate else 0.0)).abs() <= M * 2.0 ** -24 * (d.abs().sum(0) + 1.0)).all()


@pytest.mark.parametrize("M,N,K", [(4160, 50265, 768), (4097, 22016, 712)])
def test_quarters_have_the_bits_of_whole_tiles(M, N, K):
    """The last 15 k columns of dY alone are 180 tiles at most, none of them in quarters."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    dy = torch.randn(M, (N + 7) // 8 * 8, device=DEV, generator=g).to(BF)[:, :N]
    x = torch.randn(M, K, device=DEV, generator=g).to(BF)
    before = torch.randn(N, K, device=DEV, generator=g)
    dw, db = before.clone(), torch.zeros(N, device=DEV)
    ops.linear_wgrad(dy, x, dw, db, True)
    n0 = (N - 15000) // 8 * 8
    part, pdb = before[n0:].clone(), torch.zeros(N - n0, device=DEV)
    ops.linear_wgrad(dy[:, n0:], x, part, pdb, True)
    assert torch.equal(dw[n0:], part) and torch.equal(db[n0:], pdb)


@pytest.mark.parametrize("n", [9, 12])
def test_more_than_a_layer_in_one_launch(n):
    """Gradients of several layers, ragged and of different rows, in one launch (one piece a tile, or several): against fp64."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n)
    items = []
    for i in range(n):
        M, N, K = (2112, 2200)[i % 2] + i, (768, 520, 1032)[i % 3], (768, 264, 1024)[i % 3 - 1]
        dy = torch.randn(M, (N + 7) // 8 * 8, device=DEV, generator=g).to(BF)[:, :N]
        x = torch.randn(M, K, device=DEV, generator=g).to(BF)
        items.append((dy, x, torch.full((N, K), 0.5, device=DEV), torch.full((N,), -0.25, device=DEV) if i % 4 else None))
    ops.linear_wgrad_grouped(items)
    for dy, x, dw, db in items:
        M, d = dy.shape[0], dy.double()
        size = d.abs().T.contiguous() @ x.double().abs() + 1.0
        assert ((dw.double() - (d.T.contiguous() @ x.double() + 0.5)).abs() <= M * 2.0 ** -24 * size).all()
        if db is not None:
            assert ((db.double() - (d.sum(0) - 0.25)).abs() <= M * 2.0 ** -24 * (d.abs().sum(0) + 1.0)).all()


def test_pending_gradients_fill_a_launch_and_no_more():
    """autograd_train._WgradGroup: a launch takes the gradients whose tiles the chip has CUs for; the next one starts the next launch."""
    from vyomai_amd import autograd_train as AT
    sizes = []
    real = AT.ops.linear_wgrad_grouped
    AT.ops.linear_wgrad_grouped = lambda items: sizes.append(sum(-(-i[2].shape[0] // 256) * -(-i[2].shape[1] // 256) for i in items))
    try:
        group = AT._WgradGroup()
        group.armed = True   # (no backward pass to flush it)
        for layer in range(5):
            for N, K in ((768, 3072), (3072, 768), (768, 768), (2304, 768)):
                group.add_tensors(None, None, torch.empty(N, K, device="meta"), None, [])
        assert sizes == [252, 252] and group.tiles == 36
        group.flush()
        for _ in range(13):
            group.add_tensors(None, None, torch.empty(512, 512, device="meta"), None, [])
        assert sizes == [252, 252, 36, 48] and len(group.items) == 1
        group.add_tensors(None, None, torch.empty(8191, 8192, device="meta"), None, [])   # alone more than the chip
        assert sizes == [252, 252, 36, 48, 4, 1024] and not group.items
    finally:
        AT.ops.linear_wgrad_grouped = real
