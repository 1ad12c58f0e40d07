"""Score products so large that their results go through the L2 instead of being streamed: rows that are no whole 128-byte
lines, 16-byte aligned (from 12 * 2^20 results on), at any even address (from 42 * 2^20 on) and 32-byte aligned, masked and
not, by themselves and as views with a pitch.  Inputs are multiples of 2^-3 up to 1/2 in size: every sum of 128 products is a multiple of 2^-6
below 2^5, exact in 32 bits in any order, and so is its one rounding to fp16."""
import pytest
import torch

from gpu_common import raw_matmul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,d,m,n,pitch,causal", [
    (13, 128, 984, 1000, 1000, False),     # 16-byte aligned rows, ragged last tiles
    (13, 64, 1000, 1000, 1000, True),      # (under 2^25 results: hidden tiles are staged)
    (9, 128, 2304, 2200, 2200, True),      # (over: written directly)
    (8, 64, 2350, 2350, 2350, False),      # rows at every fourth, eighth, twelfth and sixteenth byte
    (8, 128, 2347, 2347, 2347, True),      # at any even address
    (8, 64, 2347, 2351, 2353, False),      # with a pitch: what lies between the rows stays
    (15, 128, 2304, 2200, 2200, True),     # as the third, from 70 * 2^20 on, where masked results are not streamed either
    (11, 128, 2347, 2347, 2347, True),     # as the fifth, from 56 * 2^20 on
    (13, 64, 2400, 2352, 2352, False),     # 32-byte aligned rows: from 18 * 2^20 on
    (16, 128, 2400, 2352, 2352, True),     # (masked: from 84 * 2^20 on)
    (8, 128, 2400, 2336, 2336, True),      # rows of whole half lines: streamed
    (9, 64, 2300, 2312, 2336, False),      # (with a pitch)
])
def test_large_scores(heads, d, m, n, pitch, causal):
    gen = torch.Generator(device="cuda").manual_seed(heads * n + d)
    q = (torch.randint(-4, 5, (m, heads * d), generator=gen, device="cuda").float() / 8).half()
    k = (torch.randint(-4, 5, (n, heads * d), generator=gen, device="cuda").float() / 8).half()
    out = torch.full((heads, m, pitch), 7.0, dtype=torch.float16, device="cuda")
    assert heads * m * n >= (12 if pitch % 8 == 0 else 42) * 2 ** 20
    assert raw_matmul("adr_matmul_f16", out, q, k, heads, m, d, n, (1, pitch, m * pitch), (1, heads * d, d),
                      (heads * d, 1, d), scale=0.5, store=4, mask=1 if causal else 0) == 0
    hidden = torch.ones(m, n, device="cuda").triu(1).bool() if causal else None
    for h in range(heads):
        want = ((q[:, h * d:(h + 1) * d].float() @ k[:, h * d:(h + 1) * d].float().t()).half() * 0.5)
        if causal:
            want.masked_fill_(hidden, -float("inf"))
        assert torch.equal(out[h, :, :n].view(torch.int16), want.view(torch.int16)), h
        assert torch.all(out[h, :, n:] == 7.0)
