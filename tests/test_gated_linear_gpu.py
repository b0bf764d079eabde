"""Gated products of more than 32 rows in one launch, on every tile that may take them: rows, outputs and contractions that end inside
a tile, a block of 16 outputs and a stage, strided operands, against the product and the activation as two launches -- the same sums in
the same order and the same roundings, so the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"
# 64 x 64 (once and twice), 256 x 128, 256 x 192, 256 x 256, 128 x 128, K split over workgroups (two launches)
SHAPES = [(33, 8, 8), (65, 24, 72), (513, 520, 200), (264, 1024, 4096), (4000, 1000, 1032), (5000, 520, 1032), (3000, 1544, 520),
          (9000, 520, 264), (6200, 1000, 520), (8192, 1024, 256), (2000, 1000, 2056), (300, 1024, 8192)]


def act_code(name):
    from vyomai_amd import _lib
    return {"silu": _lib.ACT_SILU, "gelu_tanh": _lib.ACT_GELU_TANH}[name]


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,K", SHAPES)
def test_one_launch_equals_two(M, I, K, act):
    from vyomai_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + I + K)
    x = torch.randn(M, K + 8, device=DEV, generator=g).to(BF)[:, :K]
    w = (2 * torch.randn(2 * I, K + 16, device=DEV, generator=g) / K ** 0.5).to(BF)[:, :K]
    got = ops.gated_linear(x, w, act_code(act))
    want = ops.gated_act(ops.linear(x, w), act_code(act))
    assert got.shape == (M, I) and torch.equal(got, want)
    # against fp64: the two factors' roundings (half a unit in the last of 8 bits: 2^-8 of the value, on the activation's slope of at most 1.13) and the result's
    p = x.double() @ w.double().T
    a, u = p[:, :I], p[:, I:]
    f = torch.nn.functional.silu(a) if act == "silu" else torch.nn.functional.gelu(a, approximate="tanh")
    sums = 2.0 ** -20 * (x.double().abs() @ w.double().abs().T)   # of the fp32 accumulation
    da, du = 2.0 ** -8 * a.abs() + sums[:, :I], 2.0 ** -8 * u.abs() + sums[:, I:]
    bound = 1.13 * da * (u.abs() + du) + f.abs() * du + 2.0 ** -8 * (f * u).abs() + 1e-5
    assert ((got.double() - f * u).abs() <= 1.02 * bound).all()


def test_calls_that_take_two_launches():
    """fp32, few rows, the erf GELU and widths that are no multiple of 8."""
    from vyomai_amd import _lib, ops
    for M, I, K, dt, act in ((100, 24, 64, torch.float32, _lib.ACT_SILU), (32, 64, 64, BF, _lib.ACT_SILU), (100, 64, 64, BF, _lib.ACT_GELU_ERF)):
        x, w = torch.randn(2, M // 2, K, device=DEV).to(dt), torch.randn(2 * I, K, device=DEV).to(dt)
        got = ops.gated_linear(x, w, act)
        assert got.shape == (2, M // 2, I) and torch.equal(got, ops.gated_act(ops.linear(x, w), act))
    with pytest.raises(_lib.VyomHipError):
        ops.gated_linear(torch.randn(100, 64, device=DEV).to(BF), torch.randn(24, 64, device=DEV).to(BF), _lib.ACT_SILU)
