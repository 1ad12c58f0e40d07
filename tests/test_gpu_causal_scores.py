"""Causal score products on the persistent kernel (K = 64, 128): hidden tiles take their turn with the others, staged or (large
results whose rows are no whole 128-byte lines) in aligned pieces whatever the rows' alignment, and the mask is applied where results are staged (Identity, and Scale with a positive factor) or where they are written (every
other operator and factor).  Against the step-for-step kernel on the same device, bit for bit: the inputs are
dyadic and the sums exact."""
import pytest
import torch

import oracle
from gpu_common import plan
from adrastea_amd import _ffi

pytestmark = pytest.mark.gpu


def call(name, out, q, k, args, bias, beta, scale, store, load):
    rc = getattr(_ffi.lib(), name)(torch.cuda.current_stream().cuda_stream, out.data_ptr(), q.data_ptr(), k.data_ptr(),
                                   *args, bias.data_ptr(), beta, scale, store, load, oracle.MASK_CAUSAL)
    assert rc == 0


# (heads, rows, keys, pad): tile rows that end inside a tile, fewer and more keys than rows, units whose tiles are
# all hidden, result rows aligned to 16, 8, 4 and 2 bytes
SHAPES = [(64, 300, 300, 4), (32, 513, 513, 0), (40, 257, 640, 0), (70, 400, 260, 2), (16, 1024, 1024, 0), (26, 520, 521, 0)]


@pytest.mark.parametrize("k", [64, 128])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "h%d_m%d_n%d_pad%d" % s)
def test_causal_scores_match_the_step_for_step_kernel(shape, k):
    heads, m, n, pad = shape
    width = n + pad
    args = (heads, m, k, n, 1, width, m * width, 1, heads * k, k, heads * k, 1, k)
    gen = torch.Generator(device="cuda").manual_seed(m + k)

    def dyadic(*size):
        return (torch.randint(-8, 9, size, generator=gen, device="cuda") / 8.0).half()
    q, keys, bias = dyadic(m, heads * k), dyadic(n, heads * k), dyadic(n)
    prev = dyadic(heads, m, width)
    for store, scale, load in [(0, 1.0, 0), (4, 0.125, 0), (4, -0.25, 0), (4, 0.0, 0), (0, 0.5, 1), (4, 0.5, 1), (5, 1.0, 0), (3, 1.0, 0)]:
        assert plan(args[0], m, k, n, args[4:7], args[7:10], args[10:], store=store, load=load,
                    mask=oracle.MASK_CAUSAL).startswith("gemm_nt_mfma_persistent")
        got, want = prev.clone(), prev.clone()
        call("adr_matmul_f16", got, q, keys, args, bias, 0.5, scale, store, load)
        call("adr_matmul_f16_slow", want, q, keys, args, bias, 0.5, scale, store, load)
        same = got.view(torch.int16) == want.view(torch.int16)
        # (a product of +-0 with the scale may differ in its sign bit only where both are zero)
        same |= (got == 0) & (want == 0)
        bad = (~same).nonzero()
        assert bad.numel() == 0, (store, scale, load, bad[:4].tolist())
        rows, cols = torch.arange(m, device="cuda")[:, None], torch.arange(n, device="cuda")[None, :]
        assert bool((got[:, :, :n][:, cols > rows] == float("-inf")).all())


# 2^25 results and more (direct): rows of every remainder of 8, several hidden tiles in a row, keys that end in the last
# piece of a tile, one behind it and inside a tile, a last tile row of one row; and smaller ones (staged)
HIDDEN = [(109, 300, 1031 + i, i) for i in range(8)] + [(376, 140, 640, 3), (502, 129, 519, 1), (502, 129, 520, 1),
          (64, 128, 4097, 2), (64, 129, 4096, 64), (63, 128, 4097, 2), (65, 128, 4080, 3)]


@pytest.mark.parametrize("k", [64, 128])
@pytest.mark.parametrize("shape", HIDDEN, ids=lambda s: "h%d_m%d_n%d_pad%d" % s)
def test_hidden_tiles_are_written_to_the_last_element_and_no_further(shape, k):
    """Results at every offset from a 16-byte boundary: the whole buffer against the step-for-step kernel's, and what
    is no element of the result (the pad of the rows, the space before and behind it) as it was."""
    heads, m, n, pad = shape
    width = n + pad
    size = heads * m * width
    args = (heads, m, k, n, 1, width, m * width, 1, heads * k, k, heads * k, 1, k)
    gen = torch.Generator(device="cuda").manual_seed(n + k)

    def dyadic(*shape_):
        return (torch.randint(-8, 9, shape_, generator=gen, device="cuda") / 8.0).half()
    q, keys, bias = dyadic(m, heads * k), dyadic(n, heads * k), dyadic(n)
    for offset in range(8):   # (of the buffer; with whole lines in a row the first one is staged)
        prev = torch.full((size + 80,), 5.0, dtype=torch.float16, device="cuda")
        assert prev.data_ptr() % 128 == 0
        got, want = prev.clone(), prev.clone()
        store, scale, beta = [(0, 1.0, 0.0), (4, 0.125, 0.0), (4, -0.5, 0.0), (3, 1.0, 0.5)][offset % 4]
        call("adr_matmul_f16", got[64 + offset:], q, keys, args, bias, beta, scale, store, 0)
        call("adr_matmul_f16_slow", want[64 + offset:], q, keys, args, bias, beta, scale, store, 0)
        same = (got.view(torch.int16) == want.view(torch.int16)) | ((got == 0) & (want == 0))
        bad = (~same).nonzero()
        assert bad.numel() == 0, (offset, bad[:4].tolist())
        inside = got[64 + offset:64 + offset + size].view(heads, m, width)
        assert bool((inside[:, :, n:] == 5.0).all()) and bool((got[:64 + offset] == 5.0).all())
        assert bool((got[64 + offset + size:] == 5.0).all())
