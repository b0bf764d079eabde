"""Products of 5 to 32 rows: operands requested as they are needed (up to 160 columns of K) and by lines through LDS, 512 columns at a time: one
k-step, lines for some waves only, whole chunks, one more column block, one more chunk; every epilogue.  Against fp64 on the bf16 operands."""
import pytest
import torch

from tests.test_gemm_tiles_gpu import BF, DEV, close, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [5, 16, 17, 32])
@pytest.mark.parametrize("K", [32, 96, 160, 192, 480, 512, 544, 768, 1024, 1056, 3072])
@pytest.mark.parametrize("N", [16, 784])
def test_linear(M, N, K):
    from vyomai_amd import _lib, ops
    x, w, b, r = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3), rnd(M, N, seed=4)
    product = x.double() @ w.double().T
    close(ops.linear(x, w), product, x, w)
    close(ops.linear(x, w, b), product + b.double(), x, w)
    close(ops.linear(x, w, b, residual=r), product + b.double() + r.double(), x, w)
    y = ops.linear(x, w, b, act=_lib.ACT_GELU_ERF).double()
    gelu = torch.nn.functional.gelu(product + b.double())
    # slope of the GELU: 1.13; the fp32 sums are K roundings of 2^-24 of the sum of magnitudes away, the polynomial for Phi 1e-6
    off = 1.13 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-5 * (product + b.double()).abs() + 1e-6
    assert ((y - gelu).abs() <= 2.0 ** -8 * gelu.abs() + off).all()


@pytest.mark.parametrize("B,L", [(1, 5), (3, 7), (2, 16)])
@pytest.mark.parametrize("K", [64, 160, 512, 768])
@pytest.mark.parametrize("rope", [True, False])
def test_qkv(B, L, K, rope):
    from vyomai_amd import ops
    h, hk = 3, 1
    N, M = 64 * (h + 2 * hk), B * L
    x, w, b = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3)
    cos, sin = ops.rope_tables(64, L, DEV) if rope else (None, None)
    q, k, v = (torch.empty(B, n, L, 64, dtype=BF, device=DEV) for n in (h, hk, hk))
    ops.qkv_rope(x.view(B, L, K), w, b, h, hk, 64, cos, sin, 0, q, k, v)
    t = (x.double() @ w.double().T + b.double()).view(B, L, h + 2 * hk, 64).transpose(1, 2)
    turn = lambda u: u
    if rope:
        c, s = (a[:L].double() for a in (cos, sin))
        turn = lambda u: torch.cat([u[..., :32] * c - u[..., 32:] * s, u[..., 32:] * c + u[..., :32] * s], -1)
    # rounded to bf16: the projection, both factors, both products and their sum -- 2^-9 of at most |a| + |b| each
    for got, exact in ((q, turn(t[:, :h])), (k, turn(t[:, h:h + hk])), (v, t[:, h + hk:])):
        assert ((got.double() - exact).abs() <= 8 * 2.0 ** -9 * t.abs().max()).all()


@pytest.mark.parametrize("K", [64, 160, 256])
def test_more_workgroups_than_compute_units(K):
    """4608 columns are 288 workgroups of 16, 4096 are 256: several of few columns of K share a compute unit, so an eighth more columns take no
    second round -- less than 1.25 times as long (measured: 1.03 to 1.08; one on a unit, 1.43 to 1.5)."""
    from vyomai_amd import ops
    x, times = rnd(32, K, seed=1), []
    for N in (4096, 4608):
        w, y = rnd(N, K, seed=2), torch.empty(32, N, dtype=BF, device=DEV)
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            for _ in range(50):
                ops.linear(x, w, out=y)
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        graph.replay()
        best = 1e9
        for _ in range(10):
            a.record(); graph.replay(); b.record(); b.synchronize()
            best = min(best, a.elapsed_time(b))
        times.append(best)
    assert times[1] < 1.25 * times[0], times
