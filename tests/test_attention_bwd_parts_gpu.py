"""Attention backward over few workgroups: two or four waves share a tile's rows.  The sums keep their order, so the gradients of a
batch are those of the same sequences in a batch that is large enough for whole tiles a wave, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda", torch.bfloat16

# B, heads, kv heads, queries, keys, causal, first position, hidden keys, rotation
CASES = [
    (1, 2, 2, 1, 1, True, 0, None, True), (1, 2, 1, 31, 31, False, 0, "end", True), (2, 2, 1, 64, 64, True, 0, None, True),
    (1, 4, 2, 65, 65, True, 0, "start", True), (2, 2, 2, 65, 129, True, 64, "end", False), (2, 4, 2, 33, 200, False, 0, "start", False),
    (1, 3, 1, 127, 96, False, 0, None, False), (1, 4, 2, 128, 128, True, 0, "end", True), (1, 6, 2, 129, 129, True, 0, "start", True),
    (2, 6, 2, 200, 200, True, 0, "end", True), (1, 2, 1, 256, 257, True, 1, None, False), (1, 2, 2, 333, 333, False, 0, "end", True),
    (1, 12, 4, 700, 700, True, 0, "all", True), (2, 12, 12, 512, 512, True, 0, None, False),   # (the last: 384 workgroups of 32 keys)
    (10, 12, 12, 128, 128, False, 0, "end", True), (11, 12, 12, 128, 128, False, 0, "end", True),   # (up to and past half of the CUs)
]


@pytest.mark.parametrize("case", CASES)
def test_shared_tiles_equal_whole_tiles(case):
    from vyomai_amd import ops
    B, h, hk, L, S, causal, start, hidden, rotate = case
    g = torch.Generator().manual_seed(S + L)
    draw = lambda *s: torch.randn(*s, generator=g).to(BF).to(DEV)
    q, k, v, do = draw(B, h, L, 64), draw(B, hk, S, 64), draw(B, hk, S, 64), draw(B, L, h * 64)
    seen = None
    if hidden:
        seen = torch.ones(B, S, dtype=torch.uint8)
        for b in range(B):
            n = (b + 1) * S // (B + 1)
            seen[b, {"end": slice(S - n, S), "start": slice(0, n), "all": slice(0, S)}[hidden]] = 0
        seen = seen.to(DEV)
    kw = dict(causal=causal, start_pos=start)
    tables = dict(zip(("cos", "sin"), ops.rope_tables(64, L + 8, DEV)), rope_pos0=3) if rotate else {}

    def run(times):
        q_, k_, v_, do_ = (t.repeat(times, 1, 1, 1) if t.dim() == 4 else t.repeat(times, 1, 1) for t in (q, k, v, do))
        seen_ = seen.repeat(times, 1) if seen is not None else None
        lse = torch.zeros(B * times, h, L, dtype=torch.float32, device=DEV)
        out = ops.attention(q_, k_, v_, keypad=seen_, lse=lse, **kw)
        grads = [torch.full_like(t, 7.0) for t in (q_, k_, v_)]
        ops.attention_bwd(q_, k_, v_, out, do_, lse, *grads, keypad=seen_, **kw, **tables)
        return [t[-B:] for t in grads]

    tiles = lambda n: (n + 127) // 128
    times = 256 // (B * min(h * tiles(L), hk * tiles(S))) + 1   # (both kernels past 256 workgroups of whole tiles)
    for name, few, many in zip(("dq", "dk", "dv"), run(1), run(times)):
        assert torch.equal(few, many), name
