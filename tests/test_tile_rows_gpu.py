"""Products whose K slices two groups of waves of one workgroup take, on tiles of 32, 96 and 128 rows: at the edges of a tile, with short
last stages and columns, odd and even numbers of slices; every epilogue.  Against fp64 on the bf16 operands."""
import ctypes as C

import pytest
import torch

from tests.test_gemm_tiles_gpu import BF, DEV, close, rnd
from tests.test_product_tiles_cpu import tiling

#: rows, columns, K, rows of a tile
SHAPES = [(33, 64, 512, 32), (63, 768, 768, 32), (64, 2304, 768, 32), (65, 192, 456, 32), (512, 768, 3072, 32), (481, 768, 3072, 32),
          (333, 1024, 1024, 32), (180, 2048, 2048, 32), (512, 2304, 768, 96), (480, 2304, 768, 96), (481, 2304, 768, 96),
          (1665, 768, 3072, 96), (641, 2112, 1992, 96), (1537, 768, 712, 96), (2112, 768, 3072, 128), (2049, 768, 3072, 128), (640, 3136, 1160, 128)]


def tile_rows(M, N, K):
    from vyomai_amd import _lib
    f = _lib.load().vy_debug_tile_rows
    f.argtypes, f.restype = [C.c_int64] * 4 + [C.c_double], C.c_int
    return f(M, N, K, 64 << 20, 0.0)


def test_rows_follow_what_the_fullest_CU_takes_in():
    for M, N, K, rows in SHAPES:
        assert tiling(M, N, K)[0] in ("64 twice", "64 many") and tile_rows(M, N, K) == rows, (M, N, K, tiling(M, N, K), tile_rows(M, N, K))
    assert tile_rows(1000, 768, 3072) == 64 and tile_rows(16384, 768, 768) == 256


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,rows", SHAPES)
def test_against_fp64(M, N, K, rows):
    from vyomai_amd import _lib, ops
    x, w, b, r = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3), rnd(M, N, seed=4)
    want = x.double() @ w.double().T
    close(ops.linear(x, w), want, x, w)
    product = want + b.double()
    close(ops.linear(x, w, b, residual=r), product + r.double(), x, w, 2.0 ** -8 * product.abs())   # (staged in bf16 ahead of the residual)
    pre, y = (torch.empty(M, N, dtype=BF, device=DEV) for _ in range(2))
    ops.linear(x, w, b, act=_lib.ACT_GELU_ERF, pre_out=pre, out=y)
    close(pre, product, x, w)
    gelu = torch.nn.functional.gelu(pre.double())   # (of the rounded product; the polynomial for Phi is 1e-6 off at most)
    assert ((y.double() - gelu).abs() <= 2.0 ** -8 * gelu.abs() + 2e-6 * pre.double().abs() + 1e-30).all()
    close(ops.linear_dgrad(x, w, add_to=r), want + r.double(), x, w, 2.0 ** -8 * want.abs())
    if N % 192 == 0:
        heads = N // 192
        cos, sin = ops.rope_tables(64, M, DEV)
        q, k, v = (torch.empty(1, heads, M, 64, dtype=BF, device=DEV) for _ in range(3))
        ops.qkv_rope(x.view(1, M, K), w, b, heads, heads, 64, cos, sin, 0, q, k, v)
        t = product.view(M, 3, heads, 64).permute(1, 2, 0, 3)
        c, s = (a.double() for a in (cos, sin))
        turn = lambda u: torch.cat([u[..., :32] * c - u[..., 32:] * s, u[..., 32:] * c + u[..., :32] * s], -1)
        # rounded to bf16: the projection, both factors, both products and their sum -- 2^-9 of at most |a| + |b| each
        for got, exact in ((q, turn(t[0])), (k, turn(t[1])), (v, t[2])):
            assert ((got[0].double() - exact).abs() <= 8 * 2.0 ** -9 * t.abs().max()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(64, 2304, 768), (481, 2304, 768), (640, 3136, 1160), (333, 1024, 1024)])
def test_gated(M, N, K):
    from vyomai_amd import _lib, ops
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5)
    y = ops.gated_linear(x, w, _lib.ACT_SILU)
    gate, up = ((x.float() @ w.float().T).to(BF).double()).chunk(2, -1)
    want = torch.nn.functional.silu(gate) * up
    # both factors rounded, either the other way: 2^-8 of each, SiLU's slope at most 1.1
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -7 * (1.1 * gate.abs() * up.abs() + want.abs()) + 1e-4).all()
