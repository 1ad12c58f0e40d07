"""P.V on left rows of an even length, which start at 4-byte aligned addresses: every even remainder of a slice of 64, with the
operand ending where its allocation's last element is, on each tile of the kernel; and the same product one half further on,
whose rows are not so aligned; and rows of an even pitch with NaN behind their elements.  Inputs are multiples of 2^-6 up to 2^-4
and of 2^-4 up to 2^-2: sums of up to 1031 products are multiples of 2^-12 below 2^5, exact in 32 bits in any order."""
import pytest
import torch

from gpu_common import plan, raw_matmul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,m,n,kernel", [(16, 1100, 128, "128x128"), (40, 500, 64, "128x64"), (2, 40, 64, "32x64"),
                                              (20, 448, 64, "64x64")])
def test_every_even_remainder(heads, m, n, kernel):
    gen = torch.Generator(device="cuda").manual_seed(heads * m)
    for k in list(range(258, 322, 2)) + [386, 450, 514, 598]:
        so, sl, sr = (1, n, m * n), (1, k, m * k), (1, n, k * n)
        assert plan(heads, m, k, n, so, sl, sr).startswith(f"gemm_nn_mfma_anyrow_{kernel}") or k % 64 == 0
        p = (torch.randint(-4, 5, (heads * m * k + 1,), generator=gen, device="cuda").float() / 64).half()
        v = (torch.randint(-4, 5, (heads, k, n), generator=gen, device="cuda").float() / 64).half()
        for offset in (0, 1):
            x = p[offset:offset + heads * m * k].view(heads, m, k)
            want = torch.stack([(x[h].double() @ v[h].double()).half() for h in range(heads)])
            out = torch.full((heads, m, n), 7.0, dtype=torch.float16, device="cuda")
            assert raw_matmul("adr_matmul_f16", out, p, v, heads, m, k, n, so, sl, sr, offsets=(0, offset, 0)) == 0
            assert torch.equal(out.view(torch.int16), want.view(torch.int16)), (k, offset)


@pytest.mark.parametrize("heads,m,k,n,pitch,kernel", [
    (2, 140, 70, 64, 76, "128x64x64"), (2, 140, 71, 64, 76, "128x64x64"),
    (2, 140, 326, 64, 332, "32x64x64_k4"), (2, 140, 327, 64, 332, "32x64x64_k4"),
    (40, 330, 1030, 64, 1034, "64x64x64_k4"), (40, 330, 1031, 64, 1034, "64x64x64_k4"),
    (16, 1100, 326, 128, 332, "128x128x64"), (16, 1100, 327, 128, 334, "128x128x64")])
@pytest.mark.parametrize("odd_heads", [0, 1])
def test_what_follows_k_stays_out(heads, m, k, n, pitch, kernel, odd_heads):
    """Rows of an even pitch with NaN behind their K elements, to the end of the allocation: even lengths, and odd ones, whose
    last dword is half theirs.  With heads an odd number of elements apart every second one starts 2 bytes off."""
    gen = torch.Generator(device="cuda").manual_seed(pitch + k)
    lz = m * pitch + odd_heads
    buf = torch.full((heads * lz,), float("nan"), dtype=torch.float16, device="cuda")
    p = (torch.randint(0, 5, (heads, m, k), generator=gen, device="cuda").float() / 64).half()
    torch.as_strided(buf, (heads, m, k), (lz, pitch, 1)).copy_(p)
    v = (torch.randint(-4, 5, (heads, k, n), generator=gen, device="cuda").float() / 16).half()
    so, sl, sr = (1, n, m * n), (1, pitch, lz), (1, n, k * n)
    assert plan(heads, m, k, n, so, sl, sr) == "gemm_nn_mfma_anyrow_" + kernel
    out = torch.full((heads, m, n), 7.0, dtype=torch.float16, device="cuda")
    assert raw_matmul("adr_matmul_f16", out, buf, v, heads, m, k, n, so, sl, sr) == 0
    want = torch.stack([(p[h].double() @ v[h].double()).half() for h in range(heads)])
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
