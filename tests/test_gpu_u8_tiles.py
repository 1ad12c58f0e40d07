"""Every tile of the u8 kernel, forced, at the edges of tiles and with every kind of block: blocks of 8 weights (a scale per
chunk of eight), of 16 (one per pair of chunks) and larger.  All tiles without wavefront groups sum the same products in
the same order, so they are compared bit for bit with one of them, and that one with the fp32 product of the dequantised
weights (fp16 results: half a step is 2^-11 of the value, the sums' own error is far below)."""
import pytest
import torch

from adrastea_amd import GpuKernels, _ffi

pytestmark = pytest.mark.gpu

FORCED = {1: (256, 192), 2: (256, 128), 3: (128, 128), 4: (128, 64), 10: (192, 192), 11: (192, 128), 12: (96, 96)}  # 5: 64 x 64, what they are compared with


def _run(kern, tile, x, q, s, block):
    out = torch.full((x.shape[0], q.shape[0]), 3.0, dtype=torch.float16, device="cuda")
    lib = _ffi.lib()
    try:
        assert lib.adr_debug_knob(1, tile) == 0
        kern.matmul_nt_fp16u8(out, x, q, s, block)
    finally:
        lib.adr_debug_knob(1, 0)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("block", [8, 16, 32, 64, 128])
def test_tiles_give_one_result(block):
    kern = GpuKernels()
    gen = torch.Generator(device="cuda").manual_seed(block)
    for tile, (bm, bn) in FORCED.items():
        for m, n, k in ((bm + 1, bn + 1, 384), (2 * bm - 1, bn - 8, 640), (70, 3 * bn + 5, 256), (bm, 2 * bn, 1152)):
            q = torch.randint(0, 256, (n, k), dtype=torch.uint8, device="cuda", generator=gen)
            s = (torch.rand(n, k // block, device="cuda", generator=gen) * 0.019 + 0.001).half()
            x = torch.randn(m, k, device="cuda", generator=gen).half()
            want, got = _run(kern, 5, x, q, s, block), _run(kern, tile, x, q, s, block)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (tile, m, n, k)
            w = torch.zeros(n, k, dtype=torch.float16, device="cuda")
            kern.dequantize_absmax_uint8(w, s, q)
            ref = x.double() @ w.double().t()
            rms = ref.pow(2).mean().sqrt()
            assert ((want.double() - ref).abs() / torch.maximum(ref.abs(), rms)).max() <= 2.0 ** -11 + 1e-5


@pytest.mark.parametrize("beta", [0.5, 1.0])
def test_tiles_add_to_the_result(beta):
    """beta times the previous result, added to the 32-bit sum before its one rounding: the same bits from every tile, rows of
    16-byte pieces and at any even address."""
    gen = torch.Generator(device="cuda").manual_seed(7)
    lib, k = _ffi.lib(), 640
    for tile, (bm, bn) in FORCED.items():
        for m, n in ((bm + 1, 2 * bn + 8), (2 * bm - 5, bn + 13)):
            q = torch.randint(0, 256, (n, k), dtype=torch.uint8, device="cuda", generator=gen)
            s = (torch.rand(n, k // 32, device="cuda", generator=gen) * 0.019 + 0.001).half()
            x, prev = (torch.randn(*shape, device="cuda", generator=gen).half() for shape in ((m, k), (m, n)))
            outs = []
            for knob in (5, tile):
                outs.append(prev.clone())
                try:
                    assert lib.adr_debug_knob(1, knob) == 0
                    assert lib.adr_matmul_nt_fp16u8(torch.cuda.current_stream().cuda_stream, outs[-1].data_ptr(),
                                                    x.data_ptr(), q.data_ptr(), s.data_ptr(), m, k, n, 32, beta) == 0
                finally:
                    lib.adr_debug_knob(1, 0)
            assert torch.equal(outs[1].view(torch.int16), outs[0].view(torch.int16)), (tile, m, n)
            w = torch.zeros(n, k, dtype=torch.float16, device="cuda")
            GpuKernels().dequantize_absmax_uint8(w, s, q)
            ref = x.double() @ w.double().t() + beta * prev.double()
            rms = ref.pow(2).mean().sqrt()
            assert ((outs[0].double() - ref).abs() / torch.maximum(ref.abs(), rms)).max() <= 2.0 ** -11 + 1e-5
