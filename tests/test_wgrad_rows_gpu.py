"""Weight gradients of several layers over few rows in one launch: each summed up as a launch of its own sums it up."""
import pytest
import torch

BF, DEV = torch.bfloat16, "cuda"
SHAPES = [(768, 3072), (3072, 768), (768, 768), (2304, 768), (512, 520), (255, 1032), (130, 8)]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 24, 63, 256, 257, 512, 700, 1665, 2047])
def test_rows(M):
    """Slices of 64 to 256 rows and their remainders, tiles that end in the last row or column but eight, gradients smaller than a tile, 1 to
    20 gradients.  Up to two slices the sums of a launch of its own arrive in either order with the same result; more of them are added in
    their order here, in any there: a rounding each, at most 8, of the sum of magnitudes."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    for shapes in (SHAPES, (SHAPES * 3)[:20], SHAPES[:1]):
        items, alone = [], []
        for i, (N, K) in enumerate(shapes):
            dy = torch.randn(M, (N + 7) // 8 * 8, device=DEV, generator=g).to(BF)[:, :N]
            x = torch.randn(M, K, device=DEV, generator=g).to(BF)
            new = lambda: (torch.zeros(N, K, device=DEV), torch.zeros(N, device=DEV) if i % 2 == 0 else None)
            items.append((dy, x, *new()))
            alone.append(new())
            ops.linear_wgrad(dy, x, *alone[-1], True)
        ops.linear_wgrad_rows(items)
        for (dy, x, dw, db), (dw1, db1) in zip(items, alone):
            d = dy.double()
            size, want = d.abs().T.contiguous() @ x.double().abs(), d.T.contiguous() @ x.double()
            assert ((dw.double() - want).abs() <= (M + 2) * 2.0 ** -24 * size).all()
            assert ((dw - dw1).double().abs() <= 8 * 2.0 ** -24 * size).all()
            if M <= 512:
                assert torch.equal(dw, dw1)
            if db is not None:
                assert ((db.double() - d.sum(0)).abs() <= (M + 2) * 2.0 ** -24 * d.abs().sum(0)).all()
                assert M > 512 or torch.equal(db, db1)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [200, 400, 1665])
def test_rows_are_added_to_fractions(M):
    """Gradients that are not zero: g + (s1 + s2) here, (g + s1) + s2 or (g + s2) + s1 by launches of their own.  The same bits from one slice; else
    a rounding for each slice and its sum, at most 8 slices, apart, and so is the only gradient of a launch."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    for shapes in (SHAPES, SHAPES[:1]):
        items, alone = [], []
        for N, K in shapes:
            dy = torch.randn(M, (N + 7) // 8 * 8, device=DEV, generator=g).to(BF)[:, :N]
            x, start = torch.randn(M, K, device=DEV, generator=g).to(BF), torch.randn(N, K, device=DEV, generator=g)
            items.append((dy, x, start.clone(), None))
            alone.append((start, start.clone()))
            ops.linear_wgrad(dy, x, alone[-1][1], None, True)
        ops.linear_wgrad_rows(items)
        for (dy, x, dw, _), (start, dw1) in zip(items, alone):
            d = dy.double()
            size, want = d.abs().T.contiguous() @ x.double().abs() + start.double().abs(), start.double() + d.T.contiguous() @ x.double()
            assert ((dw.double() - want).abs() <= (M + 3) * 2.0 ** -24 * size).all()
            assert ((dw - dw1).double().abs() <= 16 * 2.0 ** -24 * size).all()
            if M <= 256:
                assert torch.equal(dw, dw1)


@pytest.mark.gpu
def test_rows_are_added_to_what_is_there():
    """Two gradients of one weight in one launch, and launches on two streams: whole numbers, exact in any order."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(1)
    dy = torch.randint(-2, 3, (700, 520), device=DEV, generator=g).to(BF)
    x = torch.randint(-3, 4, (700, 264), device=DEV, generator=g).to(BF)
    dw, db = torch.full((520, 264), 5.0, device=DEV), torch.full((520,), -7.0, device=DEV)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for s in streams:
        with torch.cuda.stream(s):
            ops.linear_wgrad_rows([(dy, x, dw, db)] * 3)
    torch.cuda.synchronize()
    assert torch.equal(dw, 5.0 + 6 * (dy.float().T.contiguous() @ x.float())) and torch.equal(db, -7.0 + 6 * dy.float().sum(0))


def test_refused_on_the_host():
    from vyomai_amd import _lib
    d = (_lib.VyWgradDesc * 21)()
    import ctypes as C
    buf = (C.c_char * 64)()
    a = (C.addressof(buf) + 15) // 16 * 16

    def fill(i, dy=a, lddy=8, K=8):
        d[i].dy, d[i].lddy, d[i].x, d[i].ldx, d[i].dw, d[i].lddw, d[i].db = dy, lddy, a, 8, a, 8, None
        d[i].M, d[i].N, d[i].K = 1, 8, K
    ref = C.cast(d, C.c_void_p)
    for n, kind, match in ((0, _lib.dtype_code(BF), "1..20"), (21, _lib.dtype_code(BF), "1..20"), (1, _lib.dtype_code(torch.float32), "dtype")):
        with pytest.raises(_lib.VyomHipError, match=match):
            _lib.call("vy_linear_wgrad_rows", ref, n, kind, None)
    fill(1)
    for bad in ({"K": 12}, {"lddy": 12}, {"dy": a + 2}, {"lddy": 0}):
        fill(0, **bad)
        with pytest.raises(_lib.VyomHipError, match="multiples of 8"):
            _lib.call("vy_linear_wgrad_rows", ref, 2, _lib.dtype_code(BF), None)
        with pytest.raises(_lib.VyomHipError, match="multiples of 8"):
            _lib.call("vy_linear_wgrad_rows", ref, 1, _lib.dtype_code(BF), None)


def test_which_gradients_wait():
    from vyomai_amd import autograd_train as AT
    g, p = AT._WgradRows(), torch.nn.Parameter(torch.zeros(4))
    rows = lambda n, N, dt=BF: torch.empty(n, N, dtype=dt)
    assert g.gathers(rows(24, 768), (768, 768), [p]) and g.gathers(rows(2047, 2304), (2304, 768), [p, p])
    assert not g.gathers(rows(2048, 768), (768, 768), [p]) and not g.gathers(rows(24, 768, torch.float32), (768, 768), [p])
    assert not g.gathers(rows(4, 50265), (50265, 768), [p]) and not g.gathers(rows(24, 64), (64, 64), [p])
    assert not g.gathers(rows(24, 768), (768, 772), [p]) and not g.gathers(rows(24, 768), (768, 768), [p], torch.ones(1))
    p._vy_exchanged = True
    assert not g.gathers(rows(24, 768), (768, 768), [p])


def test_a_launch_takes_whole_layers(monkeypatch):
    """Four layers' gradients, or what comes before them and four layers'; never more than twenty."""
    from vyomai_amd import autograd_train as AT
    sizes = []
    monkeypatch.setattr(AT.ops, "wgrad_rows", lambda descs: sizes.append(len(descs)))
    monkeypatch.setattr(AT.ops, "_raw_stream", lambda: 1)
    g = AT._WgradRows()
    g.armed = True   # (no backward pass to flush it)
    keep = (torch.empty(4, dtype=BF),)
    g.add_descs([(None, [])], keep)
    for _ in range(12):
        g.add_descs([(None, [])] * 4, keep)
    assert sizes == [17, 16, 16] and not g.items
    for _ in range(15):
        g.add_descs([(None, [])], keep)
    g.add_descs([(None, [])] * 6, keep)
    assert sizes == [17, 16, 16, 15] and len(g.items) == 6
