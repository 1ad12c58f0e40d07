"""The row pitch of an operand does not change the kernel of an fp16 product: the tiles' 32-bit row offsets reach every row
of a view of fewer than 2^31 elements.  Host only (adr_matmul_f16_plan)."""
import ctypes as C

import pytest

from adrastea_amd import _ffi


def _plan(M, K, N, ly, rx, workspace=None):
    buf = C.create_string_buffer(96)
    args = (1, M, K, N, 1, N, 0, 1, ly, 0, rx, 1, 0, 0, 0, 0)
    lib = _ffi.lib()
    rc = (lib.adr_matmul_f16_plan(buf, 96, *args) if workspace is None
          else lib.adr_matmul_f16_ws_plan(buf, 96, *args, workspace))
    assert rc == 0, (M, K, N, ly, rx)
    return buf.value.decode()


@pytest.mark.parametrize("M,K,N", [
    (128, 8192, 4096), (100, 192, 4096), (130, 4096, 12288), (256, 11008, 4096), (300, 4160, 1280), (2, 1 << 25, 64),
    (3, 1088, 200), (577, 4096, 4096), (1100, 4096, 4096), (514, 5120, 13824), (2000, 1024, 1024)])
def test_the_plan_does_not_depend_on_the_pitch(M, K, N):
    for rows, other in ((M, N), (N, M)):
        farthest = ((1 << 31) - K) // (rows - 1) // 8 * 8  # the view ends at 2^31 elements or just before
        if (rows - 1) * farthest + K == 1 << 31 and rows <= 192:
            farthest -= 8  # (see below)
        for workspace in (None, 0):
            want = {side: _plan(*((rows, K, other) if side else (other, K, rows)), K, K, workspace) for side in (0, 1)}
            for pitch in (8, K + 8, 1 << 22, (1 << 22) + 8, 1 << 24, 1 << 28, farthest):
                if pitch > farthest:
                    continue
                assert _plan(rows, K, other, pitch, K, workspace) == want[1], (rows, K, other, pitch)
                assert _plan(other, K, rows, K, pitch, workspace) == want[0], (other, K, rows, pitch)


def test_a_tile_that_ends_on_the_last_byte_of_32_bits():
    """129 rows that end on exactly the 2^31st element: an unsplit tile of them does not fit and the 256-row tile, whose
    addresses have 64 bits, takes the product; the pieces of a split end before it."""
    M, K, N = 129, 8192, 4096
    pitch = ((1 << 31) - K) // (M - 1)
    assert (M - 1) * pitch + K == 1 << 31
    assert _plan(M, K, N, pitch, K, 0) == "gemm_nt_mfma_dma_256x128x64"
    assert _plan(M, K, N, pitch, K) == _plan(M, K, N, K, K) == "gemm_nt_mfma_dma_128x128x64_splitk4"
    assert _plan(M, K, N, pitch - 8, K, 0) == _plan(M, K, N, K, K, 0)


@pytest.mark.parametrize("K", [192, 1088, 4096, 8192])
def test_rows_that_go_backwards_are_addressed_in_64_bits(K):
    for M, N, ly, rx in ((300, 700, -K, K), (300, 700, K, -K), (300, 700, -(1 << 22), -K)):
        assert _plan(M, K, N, ly, rx) in ("gemm_nt_mfma_dma_256x192x64", "gemm_nt_mfma_dma_256x128x64",
                                          "gemm_nt_mfma_dma_128x256x64")


@pytest.mark.parametrize("M", [3, 16, 33, 64])
def test_few_rows_that_go_backwards_stay_off_the_unsigned_offsets(M):
    """The kernel for up to 64 rows adds a row's unsigned 32-bit offset to the operand's address: a negative pitch would read
    4 GiB further on."""
    K, N = 4096, 4096
    assert _plan(M, K, N, K, K) == "skinny_f16_mfma16_regstream"
    for ly, rx in ((-K, K), (K, -K)):
        assert not _plan(M, K, N, ly, rx).startswith("skinny")
