"""Weight gradients and norms' sums that wait for others belong to their backward pass.  Real backward passes on the CPU, the launches replaced by
the sums that they stand for."""
import gc
import threading
import weakref

import pytest
import torch

from vyomai_amd import autograd_train as AT

BF = torch.bfloat16
KINDS = ["rows", "many rows", "norms"]
M = {"rows": 8, "many rows": 2048}


@pytest.fixture(autouse=True)
def launches(monkeypatch):
    """Sizes of the launches; a descriptor is the gradient's tensors."""
    out = []

    def add(items):
        out.append(len(items))
        for dy, x, dw, db in items:
            dw.add_(dy.float().T @ x.float())

    def norms(items):
        out.append(len(items))
        for _, _, dg, db in items:
            dg.add_(1.0), db.add_(1.0)
    monkeypatch.setattr(AT.ops, "_raw_stream", lambda: 0)
    monkeypatch.setattr(AT.ops, "wgrad_desc", lambda dy, x, dw, db: ((dy, x, dw, db), (dy, x)))
    monkeypatch.setattr(AT.ops, "wgrad_rows", add)
    monkeypatch.setattr(AT.ops, "linear_wgrad_grouped", add)
    monkeypatch.setattr(AT.ops, "linear_wgrad", lambda dy, x, dw, db, accumulate, alpha=None: add([(dy, x, dw, db)]))
    monkeypatch.setattr(AT.ops, "layernorm_sums", norms)
    return out


class Product(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return x @ w.to(x.dtype).T

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dw, _ = AT._wgrad(dy.contiguous(), x, w, None)
        return dy @ w.to(dy.dtype), dw


class Norm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, b):
        ctx.params = w, b
        return x * 1.0

    @staticmethod
    def backward(ctx, dy):
        w, b = ctx.params
        AT._norm_sums.add_norms([(torch.zeros(2), 1, w.grad, b.grad, (w, b))])
        return dy, None, None


class Then(torch.autograd.Function):
    """Calls something in the middle of the backward pass."""
    @staticmethod
    def forward(ctx, x, act):
        ctx.act = act
        return x * 1.0

    @staticmethod
    def backward(ctx, dy):
        ctx.act()
        return dy, None


def parameter(shape, ready=None):
    p = torch.nn.Parameter(torch.ones(shape))
    p.grad, p._vy_direct = torch.zeros(shape), True
    if ready is not None:
        p._vy_ready = lambda q: ready.append(q)
    return p


def layer(kind, ready=None):
    """-> its parameters, and what it makes of a tensor (of no tensor: of an input of its size)."""
    if kind == "norms":
        w, b = parameter((4,), ready), parameter((4,), ready)
        return (w, b), lambda x=None: Norm.apply(torch.ones(2, 4, requires_grad=True) if x is None else x, w, b)
    w = parameter((512, 512), ready)
    return (w,), lambda x=None: Product.apply(torch.ones(M[kind], 512, dtype=BF, requires_grad=True) if x is None else x, w)


def written(params):
    return all(bool((p.grad != 0).all()) for p in params) and not any(getattr(p, "_vy_deferred", False) for p in params)


def untouched(params):
    return all(bool((p.grad == 0).all()) for p in params)


@pytest.mark.parametrize("other", KINDS)
@pytest.mark.parametrize("kind", KINDS)
def test_two_passes_at_a_time(kind, other):
    """One holds a gradient while the other begins and ends, and a trainer of the other clears its gradients."""
    ready = []
    pa, fa = layer(kind, ready)
    pb, fb = layer(other, ready)
    held, go, errors = threading.Event(), threading.Event(), []

    def wait():
        held.set()
        assert go.wait(60)

    def first():
        try:
            fa(Then.apply(torch.ones(M.get(kind, 2), 512 if kind in M else 4, dtype=BF if kind in M else None, requires_grad=True), wait)).float().sum().backward()
        except BaseException as e:
            errors.append(e)
    t = threading.Thread(target=first)
    t.start()
    assert held.wait(60)
    assert untouched(pa) and all(p._vy_deferred for p in pa)
    fb().float().sum().backward()
    assert written(pb) and {id(p) for p in ready} == {id(p) for p in pb}
    assert untouched(pa) and all(p._vy_deferred for p in pa)
    go.set()
    t.join(60)
    assert not errors and written(pa) and {id(p) for p in ready} == {id(p) for p in pa + pb}


@pytest.mark.parametrize("kind", KINDS)
def test_a_pass_that_raises(kind, launches):
    """It launches nothing, holds nothing, and the next one's gradients are written, those of the same parameters too."""
    def fail():
        raise RuntimeError("out of memory")
    ready = []
    p1, f1 = layer(kind, ready)
    p2, f2 = layer(kind, ready)
    x = Then.apply(torch.ones(M.get(kind, 2), 512 if kind in M else 4, dtype=BF if kind in M else None, requires_grad=True), fail)
    kept = weakref.ref(x)
    with pytest.raises(RuntimeError, match="out of memory"):
        f1(x).float().sum().backward()
    del x
    gc.collect()
    assert kept() is None and not launches and not ready and untouched(p1) and not any(p._vy_deferred for p in p1)
    f2().float().sum().backward()
    assert written(p2) and launches == [1]
    f1().float().sum().backward()
    assert written(p1) and launches == [1, 1] and len(ready) == len(p1) + len(p2)


@pytest.mark.parametrize("kind", KINDS)
def test_a_pass_inside_another(kind):
    """A checkpoint that runs its own backward pass in the middle of one."""
    from torch.utils.checkpoint import checkpoint
    (p1, f1), (p2, f2), (p3, f3) = layer(kind), layer(kind), layer(kind)
    y = f1()
    f3(checkpoint(f2, y, use_reentrant=True)).float().sum().backward()
    assert written(p1) and written(p2) and written(p3)


@pytest.mark.parametrize("kind", KINDS)
def test_a_backward_function_called_by_hand(kind):
    """There is no end of a pass to wait for."""
    class Ctx:
        pass
    ctx, (params, _) = Ctx(), layer(kind)
    if kind == "norms":
        ctx.params = params
        Norm.backward(ctx, torch.ones(2, 4))
    else:
        ctx.saved_tensors = torch.ones(M[kind], 512, dtype=BF), params[0]
        Product.backward(ctx, torch.ones(M[kind], 512, dtype=BF))
    assert written(params)


@pytest.mark.parametrize("accumulate", [1, 3])
@pytest.mark.parametrize("kind", KINDS)
def test_trainers_that_clear_their_gradients(kind, accumulate):
    """Another trainer's zero_grad() in the middle of a backward pass takes nothing away from it, and a micro-batch whose pass raised, nothing from
    the next one, whether zero_grad() comes between them at the start of an accumulation window or inside of one."""
    from vyomai_amd.training import FlatTrainer

    def fail():
        raise RuntimeError("out of memory")
    mine = torch.nn.ParameterList(layer(kind)[0])
    other = FlatTrainer(torch.nn.Linear(8, 8), compute_dtype=torch.float32)
    tr = FlatTrainer(mine, compute_dtype=torch.float32, accumulate_steps=accumulate)

    def loss(act):
        x = Then.apply(torch.ones(M.get(kind, 2), 512 if kind in M else 4, dtype=BF if kind in M else None, requires_grad=True), act)
        return (Norm.apply(x, *mine) if kind == "norms" else Product.apply(x, mine[0])).float().sum()
    tr.zero_grad()
    tr.backward(loss(other.zero_grad))
    assert written(mine) and len(tr.reducer.touched) == len(mine)
    tr.zero_grad()
    before = [p.grad.clone() for p in mine]
    with pytest.raises(RuntimeError, match="out of memory"):
        tr.backward(loss(fail))
    assert all(torch.equal(p.grad, g) for p, g in zip(mine, before))
    tr.zero_grad()
    tr.backward(loss(lambda: None))
    assert written(mine) and all(bool((p.grad != g).all()) for p, g in zip(mine, before))


@pytest.mark.parametrize("kind", KINDS)
def test_two_devices_in_a_pass(kind, monkeypatch):
    """A launch has the gradients of one device: streams of two have the same handles, and the engine calls each one's backward functions in a
    thread of its own."""
    out = []
    of = lambda items: {t.device.type for item in items for t in (item if kind != "norms" else item[2:])}
    for name in ("wgrad_rows", "linear_wgrad_grouped", "layernorm_sums"):
        monkeypatch.setattr(AT.ops, name, lambda items: out.append((len(items), *of(items))))

    def hold():
        for device in ("cpu", "meta") * 3:
            if kind == "norms":
                AT._norm_sums.add_norms([(None, 1, torch.zeros(4, device=device), torch.zeros(4, device=device), ())])
            else:
                dy, x, dw = (torch.zeros(512, 512, dtype=t, device=device) for t in (BF, BF, None))
                (AT._wgrad_rows if kind == "rows" else AT._wgrad_group).add_tensors(dy, x, dw, None, [])
    if kind == "rows":
        monkeypatch.setattr(AT.ops, "wgrad_desc", lambda dy, x, dw, db: ((dy, x, dw), (dy, x)))
    else:
        real = AT.ops.linear_wgrad_grouped
        monkeypatch.setattr(AT.ops, "linear_wgrad_grouped", lambda items: real([item[:3] for item in items]))
    Then.apply(torch.ones(2, requires_grad=True), hold).sum().backward()
    assert sorted(out) == [(3, "cpu"), (3, "meta")]


@pytest.mark.parametrize("which", ["dy", "x"])
@pytest.mark.parametrize("kind", ["rows", "many rows"])
def test_operands_that_no_launch_takes(kind, which, launches, monkeypatch):
    """Rows that do not start on 16 bytes are refused where their layer is reached, not with those of other layers that waited."""
    def refuse(dy, x, dw, db, accumulate, alpha=None):
        assert accumulate and any(t.data_ptr() % 16 or t.stride(0) % 8 for t in (dy, x))
        raise AT._lib.VyomHipError("vy_linear_wgrad: operands")
    monkeypatch.setattr(AT.ops, "linear_wgrad", refuse)
    w = parameter((512, 512))
    odd, even = torch.ones(M[kind], 520, dtype=BF)[:, 1:513], torch.ones(M[kind], 512, dtype=BF)
    for pair in ((odd, even), (torch.ones(M[kind], 513, dtype=BF)[:, :512], even)):
        with pytest.raises(AT._lib.VyomHipError, match="operands"):
            Then.apply(torch.ones(2, requires_grad=True), lambda: AT._wgrad(*(pair if which == "dy" else pair[::-1]), w, None)).sum().backward()
    assert not launches and not getattr(w, "_vy_deferred", False)


@pytest.mark.parametrize("kind", KINDS)
def test_a_launch_that_fails(kind, monkeypatch):
    """Nothing is left marked as waiting."""
    def fail(items):
        raise AT._lib.VyomHipError("launch failed")
    for name in ("wgrad_rows", "linear_wgrad_grouped", "layernorm_sums"):
        monkeypatch.setattr(AT.ops, name, fail)
    params, apply = layer(kind)
    with pytest.raises(AT._lib.VyomHipError, match="launch failed"):
        apply().float().sum().backward()
    assert not any(p._vy_deferred for p in params)
