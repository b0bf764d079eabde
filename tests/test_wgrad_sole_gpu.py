"""Weight gradients of which a launch adds one sum to an element, by themselves and several in one launch: against fp64; and launches on two
streams that add to one gradient."""
import types

import pytest
import torch

BF, DEV = torch.bfloat16, "cuda"


def check(dy, x, dw, db, before):
    """Sums of M products in fp32: at most M rounding errors of 2^-24 of the sum of their magnitudes, and one of what was there."""
    M, d = dy.shape[0], dy.double()
    size = d.abs().T.contiguous() @ x.double().abs() + before.abs().double() + 1.0
    assert ((dw.double() - (d.T.contiguous() @ x.double() + before.double())).abs() <= (M + 2) * 2.0 ** -24 * size).all()
    if db is not None:
        assert ((db.double() - (d.sum(0) - 0.25)).abs() <= (M + 2) * 2.0 ** -24 * (d.abs().sum(0) + 1.0)).all()


def problem(g, M, N, K):
    dy = torch.randn(M, (N + 7) // 8 * 8, device=DEV, generator=g).to(BF)[:, :N]
    x = torch.randn(M, K, device=DEV, generator=g).to(BF)
    before = torch.randn(N, K, device=DEV, generator=g)
    return dy, x, before


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 31, 64, 200, 257, 1000])
def test_grouped(M):
    """Whole tiles of 256 x 256, tiles that end in the last row or column but eight, and gradients smaller than a tile; up to 256 rows
    every element gets one sum, beyond that the 11 tiles of the first launch take several pieces a tile and the 264 of the second one."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    for shapes in ([(256, 256), (248, 264), (768, 512), (255, 8), (520, 256)], [(4096, 4096), (264, 768), (512, 256)]):
        items, olds = [], []
        for i, (N, K) in enumerate(shapes):
            dy, x, before = problem(g, M, N, K)
            items.append((dy, x, before.clone(), torch.full((N,), -0.25, device=DEV) if i % 2 == 0 else None))
            olds.append(before)
        ops.linear_wgrad_grouped(items)
        for (dy, x, dw, db), before in zip(items, olds):
            check(dy, x, dw, db, before)


@pytest.mark.gpu
def test_two_sums_for_one_gradient():
    """A weight that is used twice, and one whose gradient is a block of columns of another's, in one launch."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(3)
    (dy, x, before), (dy2, x2, _), (dy3, x3, _) = problem(g, 100, 512, 768), problem(g, 77, 512, 768), problem(g, 200, 512, 256)
    dw = before.clone()
    ops.linear_wgrad_grouped([(dy, x, dw, None), (dy2, x2, dw, None), (dy3, x3, dw[:, 256:512], None)])
    part = torch.zeros(512, 768, device=DEV, dtype=torch.float64)
    size = before.abs().double() + 1.0
    for a, b, cols in ((dy, x, slice(0, 768)), (dy2, x2, slice(0, 768)), (dy3, x3, slice(256, 512))):
        part[:, cols] += a.double().T.contiguous() @ b.double()
        size[:, cols] += a.double().abs().T.contiguous() @ b.double().abs()
    assert ((dw.double() - before.double() - part).abs() <= 400 * 2.0 ** -24 * size).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(40, 50265, 256), (200, 16384, 264), (300, 8192, 768)])
def test_by_itself(M, N, K):
    """More tiles than the chip takes at once, one piece each: whole ones and the last of an odd count of rows."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(N)
    dy, x, before = problem(g, M, N, K)
    dw, db = before.clone(), torch.full((N,), -0.25, device=DEV)
    ops.linear_wgrad(dy, x, dw, db, True)
    check(dy, x, dw, db, before)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(64, 512, 512), (200, 16384, 256), (4096, 32768, 520)])
def test_two_streams_add_to_one_gradient(M, N, K):
    """Launches of one and of several gradients on two streams at once, with nothing between them.  Whole numbers: the sums, up to
    12 * 2 * 4096 * 6, and every sum on the way are exact in fp32, in whatever order they are added."""
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    operands = []
    for _ in streams:
        dy = torch.randint(-2, 3, (M, N), device=DEV, generator=g).to(BF)
        x = torch.randint(-3, 4, (M, K), device=DEV, generator=g).to(BF)
        operands.append((dy, x))
    once = [a.float().T.contiguous() @ b.float() for a, b in operands]
    dw, db = torch.full((N, K), 5.0, device=DEV), torch.full((N,), -7.0, device=DEV)
    torch.cuda.synchronize()
    for _ in range(6):
        for s, (dy, x) in zip(streams, operands):
            with torch.cuda.stream(s):
                ops.linear_wgrad(dy, x, dw, db, True)
                if N < 16384:
                    ops.linear_wgrad_grouped([(dy, x, dw, db)])
    torch.cuda.synchronize()
    n = 12 if N < 16384 else 6
    assert torch.equal(dw, 5.0 + n * (once[0] + once[1]))
    assert torch.equal(db, -7.0 + n * sum(a.float().sum(0) for a, _ in operands))


def test_operands_of_another_type_go_out_by_themselves(monkeypatch):
    from vyomai_amd import autograd_train as AT
    alone, together = [], []
    monkeypatch.setattr(AT.ops, "linear_wgrad", lambda dy, x, dw, db, accumulate: alone.append((dy.dtype, accumulate)))
    monkeypatch.setattr(AT.ops, "linear_wgrad_grouped", lambda items: together.append(len(items)))
    monkeypatch.setattr(AT.ops, "_raw_stream", lambda: 7)
    g = AT._WgradGroup()
    g.armed = True   # (no backward pass to flush it)
    dw = torch.empty(512, 512, device="meta")
    for dt in (torch.bfloat16, torch.float32, torch.bfloat16):
        g.add_tensors(torch.empty(4, 512, dtype=dt), None, dw, None, [])
    g.flush()
    assert alone == [(torch.float32, True)] and together == [2]


def test_what_waits_goes_out_on_the_stream_of_its_operands(monkeypatch):
    """The end of a backward pass that was called on another stream than the forward pass ran on."""
    import contextlib
    from vyomai_amd import autograd_train as AT
    now, done = [5], []

    class Stream:
        def __init__(self, raw):
            self.raw = raw

        def wait_stream(self, other):
            done.append(("wait", self.raw, other.raw))

    @contextlib.contextmanager
    def inside(s):
        before, now[0] = now[0], s.raw
        yield
        now[0] = before
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: Stream(now[0]))
    monkeypatch.setattr(torch.cuda, "stream", inside)
    monkeypatch.setattr(AT.ops, "_raw_stream", lambda: now[0])
    monkeypatch.setattr(AT.ops, "linear_wgrad_grouped", lambda items: done.append(("launch", now[0])))
    g = AT._WgradGroup()
    g.armed = True
    dy = types.SimpleNamespace(dtype=torch.bfloat16, is_cuda=True)
    for caller, want in ((0, [("launch", 5), ("wait", 0, 5)]), (5, [("launch", 5)])):
        now[0] = 5
        g.add_tensors(dy, None, torch.empty(512, 512, device="meta"), None, [])
        now[0] = caller
        g._end_of_backward()
        assert done == want and not g.items
        done.clear()
        g.armed = True


@pytest.mark.gpu
def test_backward_called_on_another_stream():
    from vyomai_amd import autograd_train as AT
    from vyomai_amd.training import FlatTrainer
    from tests.test_text_layer_train_gpu import inputs, model
    ids, _ = inputs(8, 256, False)
    grads = []
    for apart in (False, True):
        m = model("decoder", 512, 8)
        tr = FlatTrainer(m, lr=0.0)
        tr.zero_grad()
        side = torch.cuda.Stream() if apart else torch.cuda.current_stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            out = m.forward_hidden(ids, None)[0]
            loss = (out.float() * torch.randn(out.shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(9))).mean()
        torch.cuda.current_stream().wait_stream(side)
        loss.backward()
        grads.append({n: p.grad.clone() for n, p in m.named_parameters() if "all_layer" in n})
        assert not AT._wgrad_group.items
        torch.cuda.synchronize()
    for n, a in grads[0].items():
        assert a.abs().max() > 0 and (a - grads[1][n]).abs().max() <= 2.0 ** -16 * a.abs().max(), n      # (sums in atomics)
