"""Activations looked up in the epilogue of the 256-row tiles: every bf16 as a pre-activation, through a product that passes them on
unchanged, has the bits that the tiles that evaluate the same expressions give it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"
# M, N, K on 256 x 256 and 256 x 128 tiles (and, without a table, 256 x 192)
SHAPES = [(16384, 3072, 768), (4000, 2000, 1032), (9000, 1040, 264)]


def patterns(rows, K):
    """(rows, K), zero but for the first eight columns: all bf16 bit patterns in order, from 2^-20 on (where the table starts), then
    the negative ones, infinities and NaNs included, repeated."""
    bits = torch.arange(65536, dtype=torch.int32)
    bits = torch.cat([bits[0x3580:0x4180], bits[0xB580:0xC180], bits]).to(torch.int16).view(BF)
    n = rows * 8
    vals = bits.repeat(-(-n // bits.numel()))[:n].view(rows, 8)
    x = torch.zeros(rows, K, dtype=BF)
    x[:, :8] = vals
    return x.to(DEV)


def pass_on(N, K, first=0, step=1):
    w = torch.zeros(N, K, dtype=BF, device=DEV)
    n = torch.arange(N, device=DEV)
    w[n, first + (n % 8) * step] = 1.0
    return w


def same(a, b):
    return torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16)) or bool(
        ((a == b) | (a.isnan() & b.isnan())).all())


@pytest.mark.parametrize("act", ["GELU_ERF", "GELU_TANH"])
@pytest.mark.parametrize("save", [None, "pre", "derivative"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_every_value(M, N, K, save, act):
    from vyomai_amd import _lib, ops
    code = getattr(_lib, "ACT_" + act) | (_lib.ACT_SAVE_DERIV if save == "derivative" else 0)
    x, w = patterns(M, K), pass_on(N, K)
    bias = torch.zeros(N, dtype=BF, device=DEV)
    pre = torch.empty(M, N, dtype=BF, device=DEV) if save else None
    got = ops.linear(x, w, bias, act=code, pre_out=pre)
    few = 64   # columns; as many as a 64 x 64 tile has: evaluated
    pre64 = torch.empty(M, few, dtype=BF, device=DEV) if save else None
    want = ops.linear(x[:, :8].contiguous(), w[:few, :8].contiguous(), bias[:few], act=code, pre_out=pre64)
    for c in range(0, N, few):
        n = min(few, N - c)
        assert same(got[:, c:c + n], want[:, :n])
        if save:
            assert same(pre[:, c:c + n], pre64[:, :n])


@pytest.mark.parametrize("act", ["SILU", "GELU_TANH"])
@pytest.mark.parametrize("M,I,K", [(8192, 1024, 256), (4000, 1000, 1032)])
def test_every_gate(M, I, K, act):
    from vyomai_amd import _lib, ops
    x = patterns(M, K)
    x[:, 8:16] = torch.randn(M, 8, device=DEV).to(BF)
    w = torch.cat([pass_on(I, K), pass_on(I, K, 8)])
    code = getattr(_lib, "ACT_" + act)
    assert same(ops.gated_linear(x, w, code), ops.gated_act(ops.linear(x, w), code))
