"""Causal score products on the persistent kernel (K = 64, 128): hidden tiles take their turn with the others, and the
mask is applied where results are staged (Identity, and Scale with a positive factor) or where they are written (every
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
