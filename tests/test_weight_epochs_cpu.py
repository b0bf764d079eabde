"""Transposed weights of models that are trained in turn: an epoch for each trainer, one launch for all of its matrices, none for the others'."""
import copy

import pytest
import torch

from vyomai_amd import autograd_train as AT


class Batch:
    launches = []

    def __init__(self, pairs):
        self.pairs, self.keys = pairs, [(a.data_ptr(), b.data_ptr()) for a, b in pairs]

    def run(self):
        Batch.launches.append(len(self.pairs))
        for src, dst in self.pairs:
            dst.copy_(src.T)


@pytest.fixture
def alone(monkeypatch):
    done = []
    monkeypatch.setattr(AT.ops, "transpose", lambda src, dst: (done.append(src.shape), dst.copy_(src.T)))
    monkeypatch.setattr(AT.ops, "TransposeBatch", Batch)
    monkeypatch.setattr(AT, "_WT", AT._WtRegistry())
    Batch.launches = []
    return done


def params(reg, n=3):
    ps = [torch.nn.Parameter(torch.randn(6, 4)) for _ in range(n)]
    for p in ps:
        p._vy_weights = reg
    return ps


def use(ps):
    for p in ps:
        assert torch.equal(AT._wt(p, torch.float32), p.detach().T)


def step(reg, ps):
    """Weights rewritten behind the versions' back, as the optimizer's kernel does."""
    for p in ps:
        p.data.add_(1.0)
    reg.bump()


def test_models_in_turn(alone):
    regs = [AT._WtRegistry() for _ in range(3)]
    models = [params(r) for r in regs]
    for r, ps in zip(regs, models):
        use(ps)
        step(r, ps)
    assert len(alone) == 9 and not Batch.launches
    for _ in range(2):
        for r, ps in zip(regs, models):
            use(ps)
            step(r, ps)
    assert len(alone) == 9 and Batch.launches == [3] * 6
    use(models[0][:1])                      # (an evaluation's backward pass: the rest is not needed, and refreshed with it)
    use(models[0])
    assert Batch.launches == [3] * 7
    step(regs[0], models[0])
    use(models[0][:1])
    step(regs[0], models[0])
    step(regs[0], models[0])
    use(models[0])                          # (two were last used two epochs ago)
    assert torch.equal(models[0][2]._vy_wt_view, models[0][2].detach().T)


def test_a_parameter_of_another_trainer(alone):
    a, b = AT._WtRegistry(), AT._WtRegistry()
    ps = params(a)
    use(ps)
    step(a, ps)
    use(ps)
    for p in ps:
        p.data = p.data.clone().add_(2.0)   # (its arena; the version stays)
        p._vy_weights = b
    use(ps)
    step(b, ps)
    use(ps)
    step(a, [])                             # (what the first one does from now on does not matter)
    use(ps)
    assert Batch.launches[-1] == 3 and not [e for e in a.entries if e[0]() is not None and e[0]()._vy_wt_entry is e]
    plain = torch.nn.Parameter(torch.randn(6, 4))   # of no trainer
    use([plain])
    with torch.no_grad():
        plain.add_(1.0)
    use([plain])


def test_a_copy_of_a_module_has_matrices_of_its_own(alone):
    class Attention(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.w = torch.nn.Parameter(torch.randn(6, 4))

        def _params(self):
            return [self.w]

        def _packed_shadow(self, dtype, packed=None, members=None):
            return self.w.detach(), None
    m, reg = Attention(), AT._WtRegistry()
    m.w._vy_weights = reg
    AT._wt_packed(m, torch.float32)
    c = copy.deepcopy(m)
    assert len(reg.entries) == 1
    for mod, r in ((m, reg), (c, AT._WT), (m, reg), (c, AT._WT)):
        mod.w.data.add_(1.0)
        r.bump()
        assert torch.equal(AT._wt_packed(mod, torch.float32), mod.w.detach().T)
    assert m._vy_wt_view.data_ptr() != c._vy_wt_view.data_ptr() and torch.equal(c._vy_wt_view, c.w.detach().T) and torch.equal(m._vy_wt_view, m.w.detach().T)


def test_trainers_have_epochs_of_their_own():
    from vyomai_amd.training import FlatTrainer
    models = [torch.nn.Sequential(torch.nn.Linear(8, 8), torch.nn.Linear(8, 8)) for _ in range(2)]
    first, second = (FlatTrainer(m, compute_dtype=torch.float32) for m in models)
    assert first.weights is not second.weights and all(p._vy_weights is first.weights for p in models[0].parameters())
    before = first.weights.epoch, second.weights.epoch, AT._WT.epoch
    first.resync()
    assert first.weights.epoch != before[0] and second.weights.epoch == before[1] and AT._WT.epoch != before[2]
    assert len({first.weights.epoch, second.weights.epoch, AT._WT.epoch}) == 3
