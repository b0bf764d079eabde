"""Products of 5 to 32 rows whose operands come line by line through LDS: no line for some waves, as many as a ring holds, one more, a short
last one; every number of weight rows a workgroup takes.  Against fp64, element by element."""
import pytest
import torch

from tests.test_decode_products_gpu import BF, DEV, NAN, entry, f32, i32, i64, p, ptr, rnd, stream, sums, within

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [5, 16, 17, 32])
@pytest.mark.parametrize("K", [8, 64, 72, 256, 264, 512, 760, 1024, 1032, 1288, 2048, 2120])
@pytest.mark.parametrize("N", [16, 40, 1001, 4100, 8200, 12300])       # (4 or 8 waves; 16, 24, 32, 48 rows; wider ones: test_rows_of_wide_products)
def test_stored(M, K, N):
    x, w, bias = rnd(M, K, seed=N), rnd(N, K, seed=12, scale=K ** -0.5), rnd(N, seed=13, scale=0.5)
    ldy = (N + 7) // 8 * 8 + 8
    y = torch.full((M, ldy), NAN, dtype=BF, device=DEV)
    go = entry("_Z14vy_rows_linearPKvS0_S0_ifPvllllP12ihipStream_t", p, p, p, i32, f32, p, i64, i64, i64, i64, p)
    assert go(ptr(x), ptr(w), ptr(bias), 0, 0.0, ptr(y), ldy, M, N, K, stream()) == 0
    torch.cuda.synchronize()
    assert torch.isnan(y[:, N:]).all()
    want, e = sums(x, w)
    within(y[:, :N], want + bias.double(), e + 2.0 ** -23 * want.abs())


@pytest.mark.parametrize("M", [17, 32])
@pytest.mark.parametrize("K", [8, 64, 248, 256, 264])
def test_wide_products_of_few_columns(M, K):
    """16400 weight rows are more than a round of 64 a workgroup: one line a wave, the last one short or not there, and more."""
    test_stored(M, K, 16400)


@pytest.mark.parametrize("M", [5, 32])
@pytest.mark.parametrize("N", [40, 4100, 12300])
def test_biases_that_start_anywhere(N, M):
    x, w, bias = rnd(M, 512, seed=N), rnd(N, 512, seed=12, scale=512 ** -0.5), rnd(N + 3, seed=13, scale=0.5)
    go = entry("_Z14vy_rows_linearPKvS0_S0_ifPvllllP12ihipStream_t", p, p, p, i32, f32, p, i64, i64, i64, i64, p)
    ldy = (N + 7) // 8 * 8
    y = torch.empty(4, M, ldy, dtype=BF, device=DEV)
    for at in range(4):
        same = torch.cat([bias[:0], bias[at:at + N]])          # (the same numbers at an aligned place)
        assert go(ptr(x), ptr(w), bias.data_ptr() + 2 * at, 0, 0.0, ptr(y[0]), ldy, M, N, 512, stream()) == 0
        assert go(ptr(x), ptr(w), ptr(same), 0, 0.0, ptr(y[1]), ldy, M, N, 512, stream()) == 0
        torch.cuda.synchronize()
        assert torch.equal(y[0, :, :N], y[1, :, :N]), at
