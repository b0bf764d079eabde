"""A backward pass that raises between its layers, and the passes after it: the gradients are those of a model without it."""
import time

import pytest
import torch

from tests.test_text_layer_train_gpu import DEV, inputs, model

pytestmark = pytest.mark.gpu


class Raise(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, on):
        ctx.on = on
        return x * 1.0

    @staticmethod
    def backward(ctx, dy):
        if ctx.on[0]:
            raise RuntimeError("in the middle")
        return dy, None


@pytest.mark.parametrize("settle", [False, True])
@pytest.mark.parametrize("accumulate", [1, 2])
@pytest.mark.parametrize("B,L", [(3, 65), (8, 256)])
def test_a_pass_that_raises(B, L, accumulate, settle):
    """settle: the next pass begins when nothing of the one that raised is left, or at once."""
    from vyomai_amd import autograd_train as AT
    from vyomai_amd.training import FlatTrainer
    groups = AT._wgrad_group, AT._wgrad_rows, AT._norm_sums
    ids, _ = inputs(B, L, False)
    grads = []
    for fails in (False, True):
        m, on = model("decoder", 512, 8, layers=3), [False]
        m.all_layer[1].register_forward_pre_hook(lambda mod, args: (Raise.apply(args[0], on), *args[1:]))
        k = accumulate * (2 if fails else 1)       # (powers of two: the losses are scaled exactly)
        tr = FlatTrainer(m, lr=0.0, accumulate_steps=k)

        def backward():
            out = m.forward_hidden(ids, None)[0]
            tr.backward((out.float() * torch.randn(out.shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(9))).mean() * k)
        tr.zero_grad()
        if fails:       # (above the raise two layers' gradients wait)
            on[0] = True
            with pytest.raises(RuntimeError, match="in the middle"):
                backward()
            on[0] = False
            if settle:          # (the engine's thread lets go of the pass when it next has the interpreter)
                end = time.monotonic() + 30
                while time.monotonic() < end and any(g.passes for g in groups):
                    time.sleep(0.01)
                assert not any(g.passes for g in groups) and not any(getattr(p, "_vy_deferred", False) for p in m.parameters())
            assert not any(p.grad.any() for n, p in m.named_parameters() if "all_layer.2" in n and p.dim() == 2)
            tr.zero_grad()      # (in an accumulation window: nothing)
            tr.arena.grad.zero_()
        for _ in range(accumulate):
            backward()
        torch.cuda.synchronize()
        grads.append({n: p.grad.clone() for n, p in m.named_parameters() if "all_layer" in n})
    for n, a in grads[0].items():
        assert a.abs().max() > 0 and (a - grads[1][n]).abs().max() <= 2.0 ** -14 * a.abs().max(), n
        # (the same products, their sums in atomics of up to 16 slices and 512 partials of a norm: 2^-20 of the sum of magnitudes, which for
        # random signs is about the root of 2048 rows, 45 times, the gradient)
