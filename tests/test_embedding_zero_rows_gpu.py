"""Token-embedding backward over rows without a gradient: zeros are skipped, everything else (NaN and infinities too) is added."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,width", [(1, 8), (5, 376), (700, 392), (300, 768), (9, 1000)])
def test_rows_of_zeros(rows, width, dtype):
    from vyomai_amd import ops
    g = torch.Generator().manual_seed(rows)
    vocab = 37
    ids = torch.randint(0, vocab, (rows,), generator=g)
    # whole numbers of one binade, so that sums in any order are exact
    dout = torch.randint(-4, 5, (rows, width), generator=g).to(dtype)
    ids[rows // 2:] = 1
    dout[rows // 2:] = 0
    dout[rows // 2:, 3] = -0.0
    if rows > 4:
        dout[rows - 1, 5], dout[rows - 2, 6], dout[rows - 3, width - 1] = float("nan"), float("inf"), 2.0
    start = torch.randint(-4, 5, (vocab, width), generator=g).float()
    dw = start.clone().cuda()
    ops.embedding_bwd_(dout.cuda(), ids.cuda(), dw, 2)
    keep = ids != 2
    want = start.double().index_add(0, ids[keep], dout[keep].double())
    assert torch.equal(dw.cpu().double().nan_to_num(nan=1e9), want.nan_to_num(nan=1e9))
