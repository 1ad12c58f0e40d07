"""Which fp16 products split K, where the unsplit tiles for partly empty rounds and the pieces are close.  Host only."""
import ctypes as C

import pytest

from adrastea_amd import _ffi


@pytest.mark.parametrize("M,K,N,kernel", [
    (513, 28672, 8192, "128x256x64_splitk3"), (576, 28672, 8192, "128x256x64_splitk3"),  # us: 278 / 291, on 192x128 316 / 321
    (1024, 28672, 8192, "256x128x64"),         # 403, in two pieces 434
    (2048, 14336, 4096, "256x128x64"),         # 185, in two pieces 212
    (1025, 11008, 4096, "192x128x64"), (1152, 11008, 4096, "192x128x64"),  # 101 and 120, in three pieces 118 and 120
    (1280, 11008, 4096, "192x128x64"),         # 118, in three pieces 125
    (2056, 11008, 2048, "192x128x64"),         # 119 (resident weights 91), in three pieces 111 (108)
    (1728, 5120, 1280, "256x128x64_splitk3")])
def test_pieces_against_whole_products(M, K, N, kernel):
    buf = C.create_string_buffer(96)
    assert _ffi.lib().adr_matmul_f16_plan(buf, 96, 1, M, K, N, 1, N, 0, 1, K, 0, K, 1, 0, 0, 0, 0) == 0
    assert buf.value.decode() == f"gemm_nt_mfma_dma_{kernel}"
