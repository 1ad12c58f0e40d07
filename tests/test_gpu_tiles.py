"""The tiles of the fp16 kernel that fill rounds the power-of-two tiles leave partly empty (256 x 224, 192 x 192,
192 x 128, 128 x 96, 96 x 96), forced, at the edges of tiles, at every remainder of their stage periods and over batches
with padded rows; and row pitches that their 32-bit row offsets do not hold.

Inputs are multiples of 2^-6 up to 2^-4 in size: every product is a multiple of 2^-12 and every sum of up to 1088 of
them below 2^2.1, exact in 32 bits in any order, so results are compared bit for bit."""
import pytest
import torch

from adrastea_amd import _ffi

pytestmark = pytest.mark.gpu

TILES = {9: (256, 224), 10: (192, 192), 11: (192, 128), 12: (128, 96), 13: (96, 96)}


def _draw(gen, shape):
    return (torch.randint(-4, 5, shape, generator=gen, device="cuda").float() / 64).half()


def _product(lib, B, M, K, N, ly, rx, oy, gen, tile):
    lz, rz, oz = M * ly + 64, N * rx + 24, M * oy + 16
    l, r = _draw(gen, (B * lz,)), _draw(gen, (B * rz,))
    out = torch.full((B * oz,), 5.0, dtype=torch.float16, device="cuda")
    want = out.clone()
    for b in range(B):
        x = torch.as_strided(l, (M, K), (ly, 1), b * lz).double()
        w = torch.as_strided(r, (N, K), (rx, 1), b * rz).double()
        torch.as_strided(want, (M, N), (oy, 1), b * oz).copy_((x @ w.t()).half())
    try:
        assert lib.adr_debug_knob(0, tile) == 0
        assert lib.adr_matmul_f16(torch.cuda.current_stream().cuda_stream, out.data_ptr(), l.data_ptr(), r.data_ptr(),
                                  B, M, K, N, 1, oy, oz, 1, ly, lz, rx, 1, rz, None, 0.0, 1.0, 0, 0, 0) == 0
    finally:
        lib.adr_debug_knob(0, 0)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16)), (tile, B, M, K, N)


@pytest.mark.parametrize("tile", TILES)
def test_edges_of_tiles_and_every_remainder_of_the_stages(tile):
    lib, gen = _ffi.lib(), torch.Generator(device="cuda").manual_seed(tile)
    bm, bn = TILES[tile]
    for slices in list(range(5, 18)):  # (fewer go to other kernels; periods of 4, 5, 6 and 12 slices)
        _product(lib, 1, bm, 64 * slices, bn, 64 * slices, 64 * slices, bn, gen, tile)
    for m in (1, 15, 17, bm - 1, bm + 1, 2 * bm + 31):
        for n in (8, bn - 8, bn + 8, 2 * bn + 40, 3 * bn - 3):
            _product(lib, 1, m, 384, n, 384, 384, n, gen, tile)
    _product(lib, 2, bm + 37, 448, 2 * bn + 24, 456, 464, 2 * bn + 32, gen, tile)


@pytest.mark.parametrize("store", [0, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("tile", TILES)
def test_every_store_with_and_without_the_mask(tile, store):
    """The epilogues of the tiles' sub-tile widths against the step-for-step kernel, whose sums are the same bits: result
    rows of 16-byte pieces, with a last column tile that ends inside the matrix, and rows at any even address.  The GELU
    stores evaluate their function to 2e-6 of its value, here at most 4, and either side rounds once to fp16."""
    lib, gen = _ffi.lib(), torch.Generator(device="cuda").manual_seed(100 * tile + store)
    bm, bn = TILES[tile]
    K, stream = 384, torch.cuda.current_stream().cuda_stream
    for M, N, oy in ((2 * bm + 31, 2 * bn + 40, 2 * bn + 40), (bm + 17, 2 * bn, 2 * bn + 8), (bm + 33, bn + 13, bn + 13),
                     (2 * bm, 2 * bn, 2 * bn + 5)):
        l, r = _draw(gen, (M, K)), _draw(gen, (N, K))
        bias, prev = (torch.randint(-8, 9, shape, generator=gen, device="cuda").div(4).half() for shape in ((N,), (M, oy)))
        for mask in (0, 1):
            got, want = prev.clone(), prev.clone()
            for fn, out, knob in ((lib.adr_matmul_f16, got, tile), (lib.adr_matmul_f16_slow, want, 0)):
                try:
                    assert lib.adr_debug_knob(0, knob) == 0
                    assert fn(stream, out.data_ptr(), l.data_ptr(), r.data_ptr(), 1, M, K, N, 1, oy, 0, 1, K, 0, K, 1, 0,
                              bias.data_ptr(), 0.5, 0.25, store, 0, mask) == 0
                finally:
                    lib.adr_debug_knob(0, 0)
            torch.cuda.synchronize()
            if store in (2, 6):
                shown = want.isfinite()
                assert torch.equal(got[~shown].view(torch.int16), want[~shown].view(torch.int16)), (M, N, mask)
                assert shown.all() == (mask == 0)
                g, w = got[shown].double(), want[shown].double()
                assert ((g - w).abs() <= w.abs() * 2.0 ** -10 + 8e-6 + 2.0 ** -24).all(), (M, N, mask)
            else:
                assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (M, N, mask)


@pytest.mark.parametrize("M,K,N,tile", [(577, 4096, 4096, "128x96"), (1100, 4096, 4096, "192x128"),
                                        (130, 4096, 12288, "96x96"), (514, 5120, 13824, "192x192"),
                                        (1100, 4096, 11008, "256x224"), (2048, 4096, 12288, "256x192"),
                                        (64, 4096, 17920, "128x128")])
def test_the_choice_is_by_rounds(M, K, N, tile):
    import ctypes as C
    buf = C.create_string_buffer(96)
    assert _ffi.lib().adr_matmul_f16_plan(buf, 96, 1, M, K, N, 1, N, 0, 1, K, 0, K, 1, 0, 0, 0, 0) == 0
    assert buf.value.decode() == f"gemm_nt_mfma_dma_{tile}x64"


@pytest.mark.parametrize("M,N", [(3, 200), (200, 5)])
def test_row_pitches_beyond_32_bit_offsets(M, N):
    """A pitch of 2^22 halves and more: 256 such rows are 2^31 bytes.  K 192 goes to the small tiles, 1088 to any."""
    lib = _ffi.lib()
    pitch = (1 << 22) + 8
    for K in (192, 1088):
        gen = torch.Generator(device="cuda").manual_seed(K)
        rows = min(M, N)
        big, small = _draw(gen, (rows * pitch,)), _draw(gen, (max(M, N), K))
        wide = torch.as_strided(big, (rows, K), (pitch, 1))
        out = torch.zeros(M, N, dtype=torch.float16, device="cuda")
        l, r, ly, rx = (big, small, pitch, K) if M < N else (small, big, K, pitch)
        assert lib.adr_matmul_f16(torch.cuda.current_stream().cuda_stream, out.data_ptr(), l.data_ptr(), r.data_ptr(),
                                  1, M, K, N, 1, N, 0, 1, ly, 0, rx, 1, 0, None, 0.0, 1.0, 0, 0, 0) == 0
        x, w = (wide, small) if M < N else (small, wide)
        assert torch.equal(out, (x.double() @ w.double().t()).half())


@pytest.mark.parametrize("side", ["left", "right"])
@pytest.mark.parametrize("sign", [1, -1])
def test_rows_gigabytes_apart(side, sign):
    """Three rows a little under 2^30 halves apart: their byte offsets need all 32 bits.  On the 64 x 64 tile, on every
    one of TILES, and with K split (K 8256; the view in the middle of its buffer, gigabytes from either end)."""
    lib, R, O = _ffi.lib(), 3, 200
    pitch, front = (1 << 30) - 16384, 1 << 30
    big = torch.empty(front + 2 * pitch + 8256 + front, dtype=torch.float16, device="cuda")
    first = front if sign > 0 else front + 2 * pitch  # of row 0
    gen = torch.Generator(device="cuda").manual_seed(3)
    out = torch.empty(R * O, dtype=torch.float16, device="cuda")
    for K, tiles in ((192, [0]), (1088, [0, *TILES]), (8256, [0])):
        wide, small = _draw(gen, (R, K)), _draw(gen, (O, K))
        if K > 1088:  # (so that sums of 8256 products stay exact)
            wide[:, 1088:] = 0
        for r in range(R):
            big[first + r * sign * pitch:first + r * sign * pitch + K] = wide[r]
        M, N = (R, O) if side == "left" else (O, R)
        x, w = (wide, small) if side == "left" else (small, wide)
        want = (x.double() @ w.double().t()).half()
        at = big.data_ptr() + 2 * first
        l, r, ly, rx = (at, small.data_ptr(), sign * pitch, K) if side == "left" else (small.data_ptr(), at, K, sign * pitch)
        for tile in tiles:
            out.fill_(5.0)
            try:
                assert lib.adr_debug_knob(0, tile) == 0
                assert lib.adr_matmul_f16(torch.cuda.current_stream().cuda_stream, out.data_ptr(), l, r,
                                          1, M, K, N, 1, N, 0, 1, ly, 0, rx, 1, 0, None, 0.0, 1.0, 0, 0, 0) == 0
            finally:
                lib.adr_debug_knob(0, 0)
            assert torch.equal(out.view(M, N), want), (K, tile)


@pytest.mark.parametrize("tile", [0, *TILES])
def test_rows_that_overlap(tile):
    """A pitch of 8 halves, the frames of a signal, and of none: the rows that a ragged tile is short of are not read."""
    lib, gen = _ffi.lib(), torch.Generator(device="cuda").manual_seed(5)
    for M, K, N, ly, rx in ((70, 1088, 200, 8, 1088), (200, 1088, 70, 1088, 8), (70, 448, 130, 0, 8), (70, 192, 200, 8, 192),
                            (70, 8256, 200, 8, 8)):
        l, r = _draw(gen, ((M - 1) * ly + K,)), _draw(gen, ((N - 1) * rx + K,))
        if K > 1088:
            l[600:-600] = 0  # (at most 1200 products that are not zero)
        x, w = torch.as_strided(l, (M, K), (ly, 1)), torch.as_strided(r, (N, K), (rx, 1))
        out = torch.full((M, N), 5.0, dtype=torch.float16, device="cuda")
        try:
            assert lib.adr_debug_knob(0, tile) == 0
            assert lib.adr_matmul_f16(torch.cuda.current_stream().cuda_stream, out.data_ptr(), l.data_ptr(), r.data_ptr(),
                                      1, M, K, N, 1, N, 0, 1, ly, 0, rx, 1, 0, None, 0.0, 1.0, 0, 0, 0) == 0
        finally:
            lib.adr_debug_knob(0, 0)
        assert torch.equal(out, (x.double() @ w.double().t()).half()), (M, K, N, ly, rx)


@pytest.mark.parametrize("M,K,N", [(3, 4096, 1100), (16, 4096, 1100), (64, 1024, 4096), (300, 1088, 700), (200, 8192, 520)])
def test_rows_that_go_backwards(M, K, N):
    """A negative pitch on either side, alone and on both: few rows, tiles, and sums that would be split."""
    lib, gen = _ffi.lib(), torch.Generator(device="cuda").manual_seed(M)
    x, w = _draw(gen, (M, K)), _draw(gen, (N, K))
    x[:, 1088:] = 0  # (so that longer sums stay exact)
    for ly, rx in ((-K, K), (K, -K), (-K, -K)):
        l, r = x.data_ptr() + (2 * (M - 1) * K if ly < 0 else 0), w.data_ptr() + (2 * (N - 1) * K if rx < 0 else 0)
        out = torch.full((M, N), 5.0, dtype=torch.float16, device="cuda")
        assert lib.adr_matmul_f16(torch.cuda.current_stream().cuda_stream, out.data_ptr(), l, r,
                                  1, M, K, N, 1, N, 0, 1, ly, 0, rx, 1, 0, None, 0.0, 1.0, 0, 0, 0) == 0
        want = ((x.flip(0) if ly < 0 else x).double() @ (w.flip(0) if rx < 0 else w).double().t()).half()
        assert torch.equal(out, want), (ly, rx)
