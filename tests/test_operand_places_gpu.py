"""Operands that do not start on 16 bytes, where kernels bring lines to LDS in 16-byte pieces: read otherwise, or refused on the host."""
import ctypes as C

import pytest
import torch

BF, DEV = torch.bfloat16, "cuda"


def moved(t):
    """The same numbers, 2 bytes behind a multiple of 16."""
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    out = flat[1:1 + t.numel()].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == 2 and out.is_contiguous()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows", [(1, True), (7, True), (7, False), (300, False), (5000, False)])
@pytest.mark.parametrize("E,K", [(24, 64), (70, 520)])
def test_router(E, K, M, rows):
    """rows: those of the tokens start elsewhere (few of them: many go through the experts' products, which ask for 16 bytes), else the router's."""
    from tests.test_decode_products_gpu import rnd, sums
    from vyomai_amd.layers.ffn import MixtureFeedForward
    top = 5
    m = MixtureFeedForward(K, E, top, 8, 1.0).to(BF).cuda()
    h, w = rnd(M, K, seed=M + E), rnd(E, K, seed=2, scale=2 * K ** -0.5)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(rnd(*p.shape, seed=3, scale=0.1))
        m.router.weight.copy_(w)
        if rows:
            h = moved(h)
        else:
            m.router.weight.data = moved(w)
    r = m.routed(h)
    assert rows or m.packed().w_router.data_ptr() % 16
    z, e = sums(h, w)
    e = e.amax(1, keepdim=True)
    ids, weight, best = r.ids.long(), r.weight.double(), z.topk(top, 1).indices
    assert ((z.gather(1, best) - z.gather(1, ids)).abs() <= 2 * e).all() and (ids.sort(1).values.diff(dim=1) > 0).all()
    exact = z.gather(1, ids).softmax(1)
    assert ((weight - exact).abs() <= exact * (4 * e + 2.0 ** -19)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("B", [1, 5, 40])
@pytest.mark.parametrize("R,dv", [(64, 64), (248, 72), (512, 136)])
def test_latent_values(R, dv, B):
    from vyomai_amd import ops
    h, dh, keys = 5, 64, 150
    g = torch.Generator(device=DEV).manual_seed(R + B)
    q, wk, wv = (torch.randn(*n, generator=g, device=DEV).to(BF) for n in ((B, h * dh), (h, R, dh), (h, dv, R)))
    cache, gate = torch.randn(B, keys, R, generator=g, device=DEV).to(BF), torch.randn(B, h * dv, generator=g, device=DEV).to(BF)
    start = torch.full((B,), keys - 1, dtype=torch.int32, device=DEV)
    run = lambda w: ops.latent_decode(q, wk * 0.1, w, cache, start, keys, 0.05, gate=gate).double()
    want, got = run(wv), run(moved(wv))
    # the same mean latents (as two bf16 halves, 2^-16 of them, where lines are multiplied), sums over R columns and a rounding to bf16
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -9 * want.abs().mean()).all()


@pytest.mark.parametrize("place", ["rows", "weights"])
def test_text_decode_products_refuse(place):
    """On the host, ahead of any launch: as the products of prompts do."""
    from vyomai_amd import _lib
    lib = _lib.load()
    p, i, l, f = C.c_void_p, C.c_int, C.c_int64, C.c_float
    x, w, to = (0x1000 + 2 * (place == "rows")), (0x2000 + 2 * (place == "weights")), 0x3000
    calls = [("_Z13vy_dec_linearPKviS0_S0_PviiiiiP12ihipStream_t", [p, i, p, p, p, i, i, i, i, i, p], (x, 768, w, None, to, 768, 8, 768, 768, 0, None)),
             ("_Z16vy_dec_linear_exPKviS0_S0_S0_iS0_S0_fPviiiiiP12ihipStream_t", [p, i, p, p, p, i, p, p, f, p, i, i, i, i, i, p],
              (x, 768, w, None, None, 0, None, None, 0.0, to, 768, 8, 768, 768, 0, None)),
             ("_Z20vy_dec_linear_res_lnPKviS0_S0_S0_iS0_S0_fPviPfiiiiP12ihipStream_t", [p, i, p, p, p, i, p, p, f, p, i, p, i, i, i, i, p],
              (x, 768, w, None, None, 0, to, to, 0.0, to, 768, to, 8, 768, 768, 0, None)),
             ("_Z10vy_dec_qkvPKvS0_S0_PKfS2_lPKiPvS5_S5_llliiiiP12ihipStream_t", [p, p, p, p, p, l, p, p, p, p, l, l, l, i, i, i, i, p],
              (x, w, None, None, None, 0, None, to, to, to, 0, 0, 0, 8, 768, 12, 12, None))]
    for name, types, args in calls:
        fn = getattr(lib, name)
        fn.argtypes, fn.restype = types, C.c_int
        assert fn(*args) == -1 and b"16-byte aligned" in lib.vy_last_error(), name
