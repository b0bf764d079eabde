"""Which kernel a product of more than 32 rows takes (pick_tiling of vyomai_amd/csrc/vy_gemm.hip), without a GPU."""
import ctypes as C

import pytest

KINDS = ["256x256", "256x192", "256x128", "128x128", "64", "64 twice", "64 many", "128 split", "320 split"]


def tiling(M, N, K, ws=64 << 20, gated=False):
    """gated: of M x N / 2 outputs, whose factors meet in a pass of their own where K is spread over workgroups"""
    from vyomai_amd import _lib
    f = _lib.load().vy_debug_tiling
    f.argtypes, f.restype = [C.c_int64] * 4 + [C.c_double], C.c_int
    t = f(M, N, K, ws, 3 if gated else 0)
    return KINDS[t % 16], t // 16


#: rows, columns, K; slices of K; kernels within 5 % of the fastest (two builds of it on one box, weights out of the Infinity Cache)
@pytest.mark.parametrize("M,N,K,slices,fastest", [
    (257, 2048, 6144, 16, {"320 split"}), (290, 2048, 6144, 16, {"320 split"}), (320, 2048, 6144, 16, {"320 split"}),
    (512, 1152, 4304, 8, {"128 split"}), (400, 1152, 4304, 8, {"128 split"}), (640, 1152, 4304, 8, {"128 split"}),
    (1300, 1152, 4304, 4, {"128 split"}), (1024, 1152, 4304, 4, {"128 split"}), (33, 512, 1536, 8, {"128 split"}),
    (100, 512, 1536, 8, {"128 split"}), (800, 1024, 6144, 8, {"128 split"}), (40, 3456, 3584, 14, {"128 split"}),
    (39, 256, 1664, 7, {"128 split"}), (4096, 768, 2304, 2, {"64"}), (4096, 768, 3072, 2, {"64", "128 split"}),
    (512, 768, 768, 4, {"64 twice"}), (512, 768, 3072, 16, {"64 many"}), (1000, 768, 3072, 8, {"64 many"}), (700, 1024, 1024, 8, {"64 many"}),
    (700, 1152, 4304, 8, {"128 split"})])
def test_kernel_is_a_fast_one(M, N, K, slices, fastest):
    kind, S = tiling(M, N, K)
    assert S == slices and kind in fastest


#: all of K in one workgroup, few stages of it: kernels within 8 % of the fastest
@pytest.mark.parametrize("M,N,K,fastest", [
    (530, 2432, 128, {"64"}), (430, 4224, 192, {"64"}), (1167, 1856, 192, {"64"}), (139, 8192, 64, {"64"}), (4181, 280, 64, {"64"}), (1019, 2056, 88, {"64"}),
    (29760, 64, 192, {"64"}), (23937, 128, 384, {"64"}), (30506, 72, 1792, {"64", "128x128"}), (1825, 5120, 224, {"256x256"}), (13215, 384, 816, {"128x128", "256x128"})])
def test_short_and_ragged_k(M, N, K, fastest):
    kind, S = tiling(M, N, K)
    assert S == 1 and kind in fastest


@pytest.mark.parametrize("M,N,K", [(32237, 1920, 432), (16988, 3968, 1064), (6307, 11648, 1856), (6632, 8800, 256), (9084, 13056, 512)])
def test_a_gelu_takes_tiles_with_a_table(M, N, K):
    """256 x 192 tiles have none: fastest without an activation, 12 to 32 % slower than 256 x 256 with a GELU."""
    from vyomai_amd import _lib
    f = _lib.load().vy_debug_tiling_gelu
    f.argtypes, f.restype = [C.c_int64] * 4, C.c_int
    assert tiling(M, N, K) == ("256x192", 1) and KINDS[f(M, N, K, 64 << 20) % 16] == "256x256"


@pytest.mark.parametrize("M,I,K,fastest", [(264, 8192, 2048, {"64"}), (129, 1024, 4096, {"64 many"}), (200, 1024, 4096, {"64 many"}),
                                           (129, 512, 2048, {"64 many"}), (129, 768, 3072, {"64 many"}), (264, 16384, 2048, {"256x256"})])
def test_gated_products_stay_in_one_launch(M, I, K, fastest):
    assert tiling(M, 2 * I, K, gated=True)[0] in fastest


def test_every_kernel_is_reached():
    """Kernels that no shape takes are not built for every epilogue."""
    seen = {tiling(M, N, K)[0] for M in (40, 256, 300, 700, 1500, 4200, 9000) for N in (512, 768, 2048, 8192) for K in (768, 2048, 6144, 16384)}
    assert seen == set(KINDS)
