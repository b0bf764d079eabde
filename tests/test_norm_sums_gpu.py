"""Column sums of several norms' gradients in one launch: the partials that vy_layernorm_bwd leaves when it is given no gradient to add to."""
import pytest
import torch

BF, DEV = torch.bfloat16, "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(1, 768)], [(3, 8), (4096, 768)], [(255, 520), (256, 64), (257, 72), (5000, 1024)], [(700, 768)] * 16])
def test_sums(shapes):
    """1 to 512 rows of partials, below and above the 64 from which they are cut in slices, and ragged column blocks."""
    from vyomai_amd import _lib, ops
    g = torch.Generator(device=DEV).manual_seed(len(shapes))
    items, want = [], []
    for M, N in shapes:
        x, dy = (torch.randn(M, N, device=DEV, generator=g).to(BF) for _ in range(2))
        gamma = torch.randn(N, device=DEV, generator=g).to(BF)
        mean, rstd = x.float().mean(1), 1.0 / (x.float().var(1, unbiased=False) + 1e-5).sqrt()
        rows = _lib.load().vy_layernorm_bwd_ws_rows(M)
        ws, dx = torch.empty(2 * rows * N, device=DEV), torch.empty_like(x)
        ops.call("vy_layernorm_bwd", dy.data_ptr(), N, x.data_ptr(), N, gamma.data_ptr(), mean.data_ptr(), rstd.data_ptr(), dx.data_ptr(), N, None, None,
                 1.0, ws.data_ptr(), M, N, _lib.dtype_code(BF), ops._stream())
        dg, db = torch.full((N,), 2.0, device=DEV), torch.full((N,), -1.0, device=DEV)
        items.append((ws, rows, dg, db))
        xh = (x.double() - mean.double()[:, None]) * rstd.double()[:, None]
        want.append((dy.double() * xh, dy.double()))
        dg1, db1 = torch.full((N,), 2.0, device=DEV), torch.full((N,), -1.0, device=DEV)
        dx1 = ops.layernorm_bwd(dy, x, gamma, mean, rstd, dg1, db1, accumulate=True)
        assert torch.equal(dx, dx1)
    ops.layernorm_sums(items)
    for (_, _, dg, db), (a, b) in zip(items, want):
        # M terms of a few roundings each, summed in fp32
        for got, t, start in ((dg, a, 2.0), (db, b, -1.0)):
            assert ((got.double() - start - t.sum(0)).abs() <= (t.shape[0] + 8) * 2.0 ** -24 * (t.abs().sum(0) + 3.0)).all()


def test_refused_on_the_host():
    import ctypes as C
    from vyomai_amd import _lib
    d = (_lib.VyNormSums * 17)()
    ref = C.cast(d, C.c_void_p)
    for n in (0, 17):
        with pytest.raises(_lib.VyomHipError, match="1..16"):
            _lib.call("vy_layernorm_sums", ref, n, None)
    with pytest.raises(_lib.VyomHipError, match="bad arguments"):
        _lib.call("vy_layernorm_sums", ref, 1, None)


def test_backward_refuses_other_factors():
    """Of what is there, all or nothing is kept; without gradients to add to as well."""
    import ctypes as C
    from vyomai_amd import _lib
    buf = (C.c_char * 256)()
    a = (C.addressof(buf) + 63) // 64 * 64
    for grads in ((None, None), (a, a)):
        for beta in (0.5, -1.0, float("nan")):
            with pytest.raises(_lib.VyomHipError, match="beta must be 0 or 1"):
                _lib.call("vy_layernorm_bwd", a, 8, a, 8, a, a, a, a, 8, *grads, beta, a, 1, 8, _lib.dtype_code(BF), None)


def test_when_sums_go_out(monkeypatch):
    """With the weight gradients of their layers, sixteen at the most; on another stream, or exchanged, at once; never reported ready before."""
    from vyomai_amd import autograd_train as AT
    out, ready, stream = [], [], [1]
    monkeypatch.setattr(AT.ops, "layernorm_sums", lambda items: out.append(len(items)))
    monkeypatch.setattr(AT.ops, "wgrad_rows", lambda descs: None)
    monkeypatch.setattr(AT.ops, "_raw_stream", lambda: stream[0])
    sums, rows = AT._NormSums(), AT._WgradRows()
    monkeypatch.setattr(AT, "_norm_sums", sums)
    sums.armed = rows.armed = True   # (no backward pass to flush them)

    def norm(exchanged=False):
        ps = [torch.nn.Parameter(torch.zeros(4)) for _ in range(2)]
        for p in ps:
            p.grad, p._vy_ready, p._vy_exchanged = torch.zeros(4), ready.append, exchanged
        return (torch.empty(8), 1, ps[0].grad, ps[1].grad, ps)
    sums.add_norms([norm(), norm()])
    assert not out and not ready and all(p._vy_deferred for item in sums.items for p in item[4])
    stream[0] = 2
    sums.add_norms([norm()])
    assert out == [1] and len(ready) == 2
    rows.add_descs([(None, [])], (torch.empty(4, dtype=BF),))
    rows.flush()                    # (of the other stream)
    assert out == [1]
    stream[0] = 1
    rows.add_descs([(None, [])], (torch.empty(4, dtype=BF),))
    rows.flush()
    assert out == [1, 2] and len(ready) == 6 and not any(p._vy_deferred for p in ready if hasattr(p, "_vy_deferred"))
    sums.add_norms([norm(True), norm(True)])
    assert out == [1, 2, 2] and not sums.items
    for _ in range(17):
        sums.add_norms([norm()])
    assert out == [1, 2, 2, 16] and len(sums.items) == 1
