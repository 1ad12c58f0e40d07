"""The tiled u8-weight kernel addresses the rows of a tile with 32-bit byte offsets: rows of up to 2^22 weights, longer
ones go to the register-staged kernels.  Checked at that edge on every tile, with rows and columns that end inside
a tile: activations are zero but for the first and the last 64 of a row, so every result is a sum of at most 128 known
products (fp32 sum and one rounding to fp16: 2^-11 of the result, plus 128 * 2^-24 of the sum of the magnitudes)."""
import ctypes as C

import pytest
import torch

from adrastea_amd import _ffi

EDGE = 1 << 22


def plan(m, p, n):
    buf = C.create_string_buffer(96)
    assert _ffi.lib().adr_matmul_nt_fp16u8_plan(buf, 96, m, p, n, 32) == 0
    return buf.value.decode()


@pytest.mark.parametrize("m", [257, 300, 511])
def test_longer_rows_are_staged_through_registers(m):
    assert plan(m, EDGE, 200).startswith("gemm_nt_u8_mfma_")
    assert plan(m, EDGE + 64, 200).startswith("gemm_nt_u8_stage_")


@pytest.mark.gpu
@pytest.mark.parametrize("tile,p", [(tile, EDGE) for tile in (*range(8), 10, 11, 12)] + [(0, EDGE + 64), (1, EDGE + 64)])
def test_products_over_the_longest_rows(tile, p):
    """(a forced tile is no tile for longer rows: they have the staged kernels only)"""
    m, n = 257, 200
    gen = torch.Generator(device="cuda").manual_seed(p + tile)
    ends = torch.cat([torch.arange(64), torch.arange(p - 64, p)]).cuda()
    q = torch.randint(0, 256, (n, p), generator=gen, device="cuda", dtype=torch.uint8)
    s = torch.rand(n, p // 32, generator=gen, device="cuda", dtype=torch.float16) * 0.019 + 0.001
    a = torch.zeros(m, p, dtype=torch.float16, device="cuda")
    a[:, ends] = torch.randn(m, 128, generator=gen, device="cuda").half()
    out = torch.full((m, n), 1000.0, dtype=torch.float16, device="cuda")
    lib = _ffi.lib()
    lib.adr_debug_knob(1, tile)
    try:
        assert lib.adr_matmul_nt_fp16u8(torch.cuda.current_stream().cuda_stream, out.data_ptr(), a.data_ptr(),
                                        q.data_ptr(), s.data_ptr(), m, p, n, 32, 0.0) == 0
    finally:
        lib.adr_debug_knob(1, 0)
    w = ((q[:, ends].float() - 127.5) * s[:, ends // 32].float()).half().float()
    x = a[:, ends].float()
    want = (x.double() @ w.double().t())
    bound = want.abs() * 2.0 ** -11 + (x.abs().double() @ w.abs().double().t()) * 128 * 2.0 ** -24 + 2.0 ** -25
    assert ((out.double() - want).abs() <= bound).all()
