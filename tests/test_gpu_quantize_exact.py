"""adr_quantize_absmax_u8 where its quotient could go wrong: bytes and scales bit for bit against the oracle
(which divides) for every finite fp16 absmax, and for blocks with infinities and NaN; rows without
gaps, which the kernel takes as one long row, and rows with gaps."""
import numpy as np
import pytest
import torch

import oracle
from adrastea_amd import GpuKernels, TensorLayout, TensorView, _ffi
from adrastea_amd import kernels as K

pytestmark = pytest.mark.gpu


def blocks_of_every_absmax(seed):
    """[31744, 32]: the first value of block b is the fp16 number of bit pattern b, the others are no larger."""
    g = np.random.default_rng(seed)
    top = np.arange(0x7C00, dtype=np.uint32)[:, None]
    bits = (g.random((0x7C00, 32)) * (top + 1)).astype(np.uint16)   # below it, denormals and zeros among them
    bits[:, 0] = top[:, 0]
    near = g.random((0x7C00, 32)) < 0.5                             # half of them at the block's own magnitude
    bits = np.where(near, np.maximum(top - g.integers(0, 2048, bits.shape), 0), bits).astype(np.uint16)
    bits[:, 0] = top[:, 0]
    return (bits | (g.integers(0, 2, bits.shape) << 15)).astype(np.uint16).view(np.float16)


@pytest.mark.parametrize("rows,cols", [(31744, 32), (992, 1024), (1, 31744 * 32)])
def test_every_absmax(rows, cols):
    x = blocks_of_every_absmax(rows).reshape(rows, cols)
    want_q, want_s = oracle.quantize_absmax_u8(x, 32)
    q = torch.zeros(rows, cols, dtype=torch.uint8, device="cuda")
    s = torch.zeros(rows, cols // 32, dtype=torch.float16, device="cuda")
    GpuKernels().quantize_absmax_uint8(q, s, torch.from_numpy(x).cuda())
    assert np.array_equal(s.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(q.cpu().numpy(), want_q)


def test_infinities_and_nan():
    g = np.random.default_rng(5)
    x = g.standard_normal((64, 256)).astype(np.float16)
    for value in (0x7C00, 0xFC00, 0x7E00, 0xFE00):
        x.view(np.uint16)[g.integers(0, 64, 40), g.integers(0, 256, 40)] = value
    want_q, want_s = oracle.quantize_absmax_u8(x, 32)
    q = torch.zeros(64, 256, dtype=torch.uint8, device="cuda")
    s = torch.zeros(64, 8, dtype=torch.float16, device="cuda")
    GpuKernels().quantize_absmax_uint8(q, s, torch.from_numpy(x).cuda())
    assert np.array_equal(s.cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(q.cpu().numpy(), want_q)


@pytest.mark.parametrize("gap_in,gap_q,gap_s", [(8, 0, 0), (0, 8, 0), (0, 0, 1), (16, 24, 3)])
@pytest.mark.parametrize("cols,bs", [(96, 32), (4096, 32), (4104, 8), (8704, 512)])
def test_rows_with_gaps(cols, bs, gap_in, gap_q, gap_s):
    rows = 9
    g = np.random.default_rng(cols + gap_in)
    x = torch.from_numpy(g.standard_normal((rows, cols + gap_in)).astype(np.float16)).cuda()
    q = torch.full((rows, cols + gap_q), 7, dtype=torch.uint8, device="cuda")
    s = torch.full((rows, cols // bs + gap_s), 7.0, dtype=torch.float16, device="cuda")

    def desc(t, width):
        return K.descriptor(TensorView(t, TensorLayout((rows, width), (t.shape[1], 1))))
    assert _ffi.lib().adr_quantize_absmax_uint8(torch.cuda.current_stream().cuda_stream, desc(q, cols),
                                                desc(s, cols // bs), desc(x, cols)) == 0
    want_q, want_s = oracle.quantize_absmax_u8(np.ascontiguousarray(x[:, :cols].cpu().numpy()), bs)
    assert np.array_equal(s[:, :cols // bs].cpu().numpy().view(np.uint16), want_s.view(np.uint16))
    assert np.array_equal(q[:, :cols].cpu().numpy(), want_q)
    assert (q[:, cols:] == 7).all() and (s[:, cols // bs:] == 7).all()


def test_more_values_than_one_launch_counts_along_x():
    """2^36 values: as one long row they would be 2^24 workgroups of 256 lanes, one lane more than a launch takes."""
    rows, cols = 1 << 20, 1 << 16
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    need = rows * cols * 3 + rows * (cols // 32) * 2
    if torch.cuda.mem_get_info()[0] < need + (8 << 30):
        pytest.skip("less than 219 GB of device memory free")
    x = torch.ones(rows, cols, dtype=torch.float16, device="cuda")
    ends = [0, 1, 2, 3, rows - 2, rows - 1]
    x[ends] = torch.randn(len(ends), cols, dtype=torch.float16, device="cuda")
    q = torch.zeros(rows, cols, dtype=torch.uint8, device="cuda")
    s = torch.zeros(rows, cols // 32, dtype=torch.float16, device="cuda")
    try:
        GpuKernels().quantize_absmax_uint8(q, s, x)
        want_q, want_s = oracle.quantize_absmax_u8(x[ends].cpu().numpy(), 32)
        assert np.array_equal(q[ends].cpu().numpy(), want_q)
        assert np.array_equal(s[ends].cpu().numpy().view(np.uint16), want_s.view(np.uint16))
        one_q, one_s = oracle.quantize_absmax_u8(np.ones((1, 32), np.float16), 32)
        assert all((q[r:r + 65536] == int(one_q[0, 0])).all() for r in range(65536, rows - 65536, 65536))
        assert all((s[r:r + 65536] == float(one_s[0, 0])).all() for r in range(65536, rows - 65536, 65536))
    finally:
        del x, q, s
        torch.cuda.empty_cache()
