"""The AdamW kernel over ranges that end inside a quad, inside a workgroup's pass and behind the second pass of all workgroups: every element
once, against the update in fp64."""
import pytest
import torch

DEV = "cuda"
PASS = 512 * 256 * 4     # elements that all workgroups take with a quad a thread


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 2048, 2051, PASS - 1, PASS, PASS + 5, 2 * PASS - 4, 2 * PASS + 1, 3 * PASS + 6, 5 * PASS + 2])
def test_sizes(n):
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n % 1000)
    p, gr, m = (torch.randn(n + 8, device=DEV, generator=g) for _ in range(3))
    v = torch.rand(n + 8, device=DEV, generator=g)
    pb = torch.zeros(n + 8, device=DEV, dtype=torch.bfloat16)
    lr, b1, b2, eps, wd, step = 1e-3, 0.9, 0.999, 1e-8, 0.01, 3
    old = [t.double() for t in (p, gr, m, v)]
    keep = [t[n:].clone() for t in (p, m, v, pb)]
    ops.adamw_step(p[:n], gr[:n], m[:n], v[:n], pb[:n], lr, b1, b2, eps, wd, step, 0.5)
    for t, k in zip((p, m, v, pb), keep):
        assert torch.equal(t[n:], k)
    q, h, a, c = (t[:n] for t in old)
    h = 0.5 * h
    a, c = b1 * a + (1 - b1) * h, b2 * c + (1 - b2) * h * h
    q = q * (1 - lr * wd) - lr / (1 - b1 ** step) * a / (c.sqrt() / (1 - b2 ** step) ** 0.5 + eps)
    # a dozen roundings of 2^-24 of terms that are at most ten times the result, and factors that are powf's
    for got, want in ((p[:n], q), (m[:n], a), (v[:n], c)):
        assert ((got.double() - want).abs() <= 2.0 ** -19 * (want.abs() + 0.1)).all()
    assert torch.equal(pb[:n], p[:n].to(torch.bfloat16))
