"""Products of more than 32 rows on every tile the launcher chooses from, at the sizes where a tile can go wrong: its edges, ragged
rows and columns, a K that is no multiple of a stage, one stage only, fewer stages than the ring holds, odd numbers of stages for
the two groups of a 64 x 64 workgroup.  Against fp64 on the bf16 operands."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

BF, DEV = torch.bfloat16, "cuda"


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(BF)


def close(got, want, x, w, extra=0.0):
    """A bf16 result of an fp32 sum: half an ulp of the result (2^-9 of it, twice where it is rounded ahead of a sum too) and the
    fp32 sum's own error, at most K 2^-24 of the terms' magnitudes; tiny results have the spacing 2^-133."""
    K = x.shape[1]
    bound = 2.0 ** -8 * want.abs() + extra + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30
    assert torch.isfinite(got).all()
    worst = ((got.double() - want).abs() / bound).max()
    assert worst <= 1, float(worst)


#: rows, columns, K: 64 x 64 tiles (one and two groups), 128 x 128, 256 x 128, 256 x 192, 256 x 256, K split over workgroups
SHAPES = [(33, 8, 8), (63, 64, 64), (64, 72, 72), (65, 200, 136), (127, 64, 192), (129, 520, 200), (512, 768, 768), (300, 2304, 760),
          (1000, 776, 320), (2111, 1032, 448), (1665, 3080, 128), (4096, 768, 3072), (4100, 1000, 1024), (8000, 1024, 1600),
          (3000, 2048, 2048), (8193, 1030, 64), (9000, 776, 832), (130, 768, 6144), (257, 1024, 4160), (700, 1024, 6144),
          # slices of K added up in order inside a tile, by one group of waves or two: two to eight, short last ones (more of them: SLICED, below)
          (512, 768, 576), (512, 776, 704), (700, 1024, 1024), (2112, 768, 3072), (1700, 1544, 392), (512, 768, 840)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_linear_on_every_tile(M, N, K):
    from vyomai_amd import ops
    x, w, b, r = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3), rnd(M, N, seed=4)
    y = ops.linear(x, w)
    close(y, x.double() @ w.double().T, x, w)
    y = ops.linear(x, w, b, residual=r)
    product = x.double() @ w.double().T + b.double()
    close(y, product + r.double(), x, w, 2.0 ** -8 * product.abs())      # (the product is staged in bf16 ahead of the residual)


@pytest.mark.parametrize("M,N,K", [(64, 768, 768), (333, 3072, 768), (512, 3080, 136), (1100, 2304, 768)])
def test_activation_and_its_saved_derivative_on_small_tiles(M, N, K):
    from vyomai_amd import ops, _lib
    x, w, b = rnd(M, K, seed=5), rnd(N, K, seed=6, scale=K ** -0.5), rnd(N, seed=7)
    y = torch.empty(M, (N + 7) // 8 * 8, dtype=BF, device=DEV)[:, :N]
    pre = torch.empty(M, (N + 7) // 8 * 8, dtype=BF, device=DEV)[:, :N]
    ops.linear(x, w, b, act=_lib.ACT_GELU_ERF, pre_out=pre, out=y)
    z = x.double() @ w.double().T + b.double()
    close(pre, z, x, w)
    zb = pre.double()                                       # the activation is of the staged bf16 value
    want = 0.5 * zb * (1 + torch.erf(zb / math.sqrt(2)))
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()       # 1e-5: the epilogue's fast erf


def test_what_a_residual_behind_an_activation_costs():
    """Requested ahead like a residual by itself, it costs as much: 1.02 times (requested where it is added: 1.13)."""
    from tests.test_decode_products_gpu import microseconds
    from vyomai_amd import ops, _lib
    M, N, K = 30500, 768, 768
    x, w, b, r = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3), rnd(M, N, seed=4)
    y = torch.empty(M, N, dtype=BF, device=DEV)
    plain, behind = (microseconds(lambda: ops.linear(x, w, b, act=a, residual=r, out=y), 10) for a in (_lib.ACT_NONE, _lib.ACT_RELU2))
    assert behind <= 1.08 * plain, (plain, behind)


@pytest.mark.parametrize("B,L,h,hk", [(3, 37, 12, 12), (1, 65, 12, 4), (5, 333, 12, 4), (2, 1000, 12, 12)])
def test_rotary_heads_on_small_tiles(B, L, h, hk):
    from vyomai_amd import ops
    K, N, pos0 = 768, (h + 2 * hk) * 64, 3
    x, w, b = rnd(B, L, K, seed=8), rnd(N, K, seed=9, scale=K ** -0.5), rnd(N, seed=10)
    cos, sin = ops.rope_tables(64, pos0 + L, DEV)
    q = torch.empty(B, h, L, 64, dtype=BF, device=DEV)
    cache = torch.zeros(2, B, hk, pos0 + L + 2, 64, dtype=BF, device=DEV)
    k, v = cache[0, :, :, pos0:pos0 + L], cache[1, :, :, pos0:pos0 + L]
    ops.qkv_rope(x, w, b, h, hk, 64, cos, sin, pos0, q, k, v)
    y = (x.double() @ w.double().T + b.double()).view(B, L, -1, 64).transpose(1, 2)
    c, s = (t[pos0:pos0 + L].double() for t in (cos, sin))
    turn = lambda t: torch.cat([t[..., :32] * c - t[..., 32:] * s, t[..., 32:] * c + t[..., :32] * s], -1)
    size = y.abs().amax(-1, keepdim=True)
    # rounded to bf16: the projection, both factors, both products and their sum -- 2^-9 of at most |a| + |b| each
    for got, want in ((q, turn(y[:, :h])), (k, turn(y[:, h:h + hk])), (v, y[:, h + hk:])):
        assert ((got.double() - want).abs() <= 8 * 2.0 ** -9 * size.amax()).all()
    assert float(cache[:, :, :, :pos0].abs().max()) == 0 and float(cache[:, :, :, pos0 + L:].abs().max()) == 0


def test_workspaces_that_come_and_go():
    """Another thread registers the stream's workspace and takes it back (the memory itself stays) while products are launched."""
    import threading
    from vyomai_amd import ops
    from vyomai_amd._lib import call
    g = torch.Generator(device=DEV).manual_seed(3)
    x, w = (torch.randn(n, 8192, device=DEV, generator=g).to(BF) for n in (264, 1024))
    st, size = torch.cuda.current_stream().cuda_stream, 64 << 20
    buf = torch.empty(size, dtype=torch.uint8, device=DEV)
    register = ops._mid_ws
    ops._mid_ws = lambda rows: None
    done = threading.Event()

    def turn():
        while not done.is_set():
            call("vy_workspace_set", st, None, 0)
            call("vy_workspace_set", st, buf.data_ptr(), size)
    other = threading.Thread(target=turn)
    try:
        call("vy_workspace_set", st, buf.data_ptr(), size)
        want = ops.linear(x, w)
        other.start()
        got = [ops.linear(x, w) for _ in range(400)]
        done.set()
        other.join()
        assert all(torch.equal(y, want) for y in got)
    finally:
        done.set()
        ops._mid_ws = register
        call("vy_workspace_set", st, None, 0)
        ops._WS.pop((torch.cuda.current_device(), st), None)


@pytest.mark.parametrize("M,N,K,act", [(5000, 768, 768, 1), (4097, 256, 4104, 0), (8192, 512, 2048, 0), (12001, 128, 1536, 0),
                                       (4096, 768, 3072, 0), (2112, 768, 768, 1), (264, 1024, 8192, 0), (200, 1152, 4304, 1),
                                       (33, 64, 1000, 0), (512, 768, 3080, 0)])
def test_bits_before_and_behind_a_smaller_product(M, N, K, act):
    """The first product on a stream, the same one behind a product for which the stream gets a workspace, the same one on a stream
    with a workspace that is too small: equal bits, as plain, gated and rotary products."""
    from vyomai_amd import ops
    from vyomai_amd._lib import call
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=1 / math.sqrt(K))
    heads = N // 192

    def products():
        out = [ops.linear(x, w, act=act), ops.gated_linear(x, w, 3)]
        if heads:
            qkv = [torch.empty(1, heads, M, 64, dtype=BF, device=DEV) for _ in range(3)]
            ops.qkv_rope(x.view(1, M, K), w[:192 * heads].contiguous(), None, heads, heads, 64, None, None, 0, *qkv)
            out += qkv
        return out
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        st, key = stream.cuda_stream, (torch.cuda.current_device(), stream.cuda_stream)
        register, small = ops._mid_ws, torch.empty(1 << 16, dtype=torch.uint8, device=DEV)
        try:
            ops._mid_ws = lambda rows: None
            call("vy_workspace_set", st, None, 0)     # (torch hands streams out again)
            ops._WS.pop(key, None)
            first = products()
            call("vy_workspace_set", st, small.data_ptr(), 1 << 16)
            narrow = products()
            ops._mid_ws = register
            ops.linear(rnd(64, 512, seed=3), rnd(64, 512, seed=4))
            assert key in ops._WS
            behind = products()
            stream.synchronize()
        finally:
            ops._mid_ws = register
            call("vy_workspace_set", st, None, 0)
            ops._WS.pop(key, None)
    assert all(torch.equal(a, b) and torch.equal(a, c) for a, b, c in zip(first, behind, narrow))


#: rows, columns, K, slices of K, kernel that adds them up inside a workgroup, kernels over which they are spread with a workspace
SLICED = [(640, 1536, 6152, 4, "64 twice", "128 split"), (200, 384, 1096, 6, "64 many", "128 split"), (900, 576, 3080, 7, "64 many", "128 split"),
          (900, 768, 4304, 8, "64 many", "128 split"), (257, 3072, 5000, 8, "64 many", "320 split"), (640, 384, 2056, 11, "64 many", "128 split"),
          (900, 384, 4104, 13, "64 many", "128 split"), (65, 192, 4304, 14, "64 many", "128 split"), (640, 576, 5000, 16, "64 many", "128 split"),
          (257, 1536, 5000, 16, "64 many", "320 split")]


@pytest.mark.parametrize("M,N,K,S,inside,over", SLICED)
def test_slices_inside_a_workgroup_and_over_workgroups(M, N, K, S, inside, over):
    """Odd and even numbers of slices (the second group of waves has one less of the odd ones), last slices and stages that are short: plain,
    behind a residual, gradient, gated and rotary products on the two kinds of kernels, bit by bit."""
    from tests.test_product_tiles_cpu import tiling
    from vyomai_amd import ops, _lib
    from vyomai_amd._lib import call
    assert tiling(M, N, K, 0) == (inside, S) and tiling(M, N, K) == (over, S)
    x, w, b, r = rnd(M, K, seed=1), rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3), rnd(M, N, seed=4)
    heads = N // 192
    cos, sin = ops.rope_tables(64, M, DEV)

    def products():
        out = [ops.linear(x, w), ops.linear(x, w, b, act=_lib.ACT_GELU_ERF, residual=r), ops.linear_dgrad(x, w, pre=r, act=_lib.ACT_GELU_ERF),
               ops.linear_dgrad(x, w, add_to=r), ops.gated_linear(x, w, _lib.ACT_SILU)]
        qkv = [torch.empty(1, heads, M, 64, dtype=BF, device=DEV) for _ in range(3)]
        ops.qkv_rope(x.view(1, M, K), w, b, heads, heads, 64, cos, sin, 0, *qkv)
        return out + qkv
    st, key = torch.cuda.current_stream().cuda_stream, (torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)
    register = ops._mid_ws
    try:
        spread = products()
        ops._mid_ws = lambda rows: None
        torch.cuda.synchronize()
        call("vy_workspace_set", st, None, 0)
        ops._WS.pop(key, None)
        held = products()
        torch.cuda.synchronize()
    finally:
        ops._mid_ws = register
    close(held[0], x.double() @ w.double().T, x, w)
    assert all(torch.equal(a, b) for a, b in zip(held, spread))
