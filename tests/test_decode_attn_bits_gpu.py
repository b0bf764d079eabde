"""Decode attention's bits: one softmax over all keys of a row, whatever their number, summed in one order.  Generated texts and the logits behind
them follow these bits, so another order of the same sums is another result.  Digests of outputs from whole-number inputs, the same on any host."""
import hashlib
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"


def numbers(shape, seed):
    """Sixty-fourths from -127 to 127, which bf16 holds."""
    return (torch.randint(-127, 128, shape, generator=torch.Generator().manual_seed(seed)).float() / 64).to(BF).to(DEV)


def digest(t):
    return hashlib.sha256(t.contiguous().view(torch.uint8).cpu().numpy().tobytes()).hexdigest()[:16]


def attention(B, h, hk, S, dh):
    from vyomai_amd import ops
    return digest(ops.attention_decode(numbers((B, h, 1, dh), 1), numbers((B, hk, S, dh), 2), numbers((B, hk, S, dh), 3), S))


def shares(B, h, hk, S):
    """Few sequences: the heads' shares of the output projection."""
    from tests.test_decode_products_gpu import entry, f32, i32, i64, p, ptr, stream
    d = 64 * h
    q, k, v = numbers((B, d), 1), numbers((B, hk, S, 64), 2), numbers((B, hk, S, 64), 3)
    wo = (numbers((d, d), 4).float() / 32).to(BF)
    together = h // hk if B > 1 and 2 <= h // hk <= 4 else 1
    part = torch.zeros((h // together, B, d), device=DEV)
    go = entry("_Z15vy_dec_attn_outPKvS0_S0_lllS0_PfliiillPKifP12ihipStream_t", p, p, p, i64, i64, i64, p, p, i64, i32, i32, i32, i64, i64, p, f32, p)
    assert go(ptr(q), ptr(k), ptr(v), hk * S * 64, S * 64, 64, ptr(wo), ptr(part), part.numel() * 4, B, h, hk, S, S, None, 0.125, stream()) == h // together
    torch.cuda.synchronize()
    return digest(part)


# keys for each number of passes (3, 5, 7, 10, 12 of 64, or of 32 with heads of 256), kept and streamed, 1 to 4 heads of a key head
ATTENTION = [(1, 12, 12, 60, 64), (1, 12, 12, 200, 64), (1, 12, 12, 700, 64), (32, 12, 12, 84, 64), (32, 12, 12, 320, 64), (32, 12, 12, 400, 64),
             (32, 12, 12, 524, 64), (20, 12, 12, 768, 64), (24, 8, 4, 130, 64), (24, 8, 4, 700, 64), (16, 12, 4, 300, 64), (16, 12, 4, 448, 64),
             (9, 16, 4, 190, 64), (9, 16, 4, 641, 64), (1, 8, 1, 60, 256), (1, 8, 1, 300, 256), (12, 8, 2, 161, 256), (12, 8, 2, 384, 256)]
SHARES = [(1, 12, 12, 61), (1, 12, 12, 330), (1, 12, 4, 600), (1, 12, 12, 768), (2, 8, 8, 250), (2, 8, 4, 61), (2, 8, 4, 500), (3, 12, 4, 100), (3, 12, 4, 768),
          (4, 16, 4, 300), (4, 16, 4, 640)]
WANT = dict(zip(itertools.chain(ATTENTION, SHARES), """
4e02703ce131d00f d21793b02e6b7d47 85872d59bd179564 39ef105271860bf3 bee693e122474577 a91023c97d919f8a accadd1678d44c9e 57480d298443e270
8c0491f7fe79999c b66b60ab17f7e627 01e566f565450eca 8aed95bea42940e7 8464333c0d3362f0 c4626c5c336b62c0 4a6517ab89713483 d2d768729037d5bf
f73bad2e9df27180 d06155c23aae1dff 48a41667ae7bd796 709ab833a0739067 245804a76fe23d54 0b0db3b5c6caa468 53adde4ea22e71bf 11025c881af0d9bb
16cb718bfe2fe999 b09cdac33320b007 d793e8b674fbf86d f4ee1f559c6f4ab6 26f6e43a9f48fecd
""".split()))


@pytest.mark.parametrize("case", ATTENTION + SHARES, ids=str)
def test_bits(case):
    assert (attention if len(case) == 5 else shares)(*case) == WANT[case]
