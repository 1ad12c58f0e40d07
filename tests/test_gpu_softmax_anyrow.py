"""Rows that are not 16-byte aligned: the row lengths at which one more chunk per lane is needed, and
every place a tensor can start at, in place and into a buffer that lies differently, against the CPU
oracle.  One fp16 step: the oracle's exponentials and sums are fp32 in another order, far below it."""
import numpy as np
import pytest
import torch

import oracle
from adrastea_amd import _ffi
from gpu_common import to_dev, to_np
from helpers import rng, ulp_diff_f16

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 7, 9, 505, 506, 512, 513, 1017, 1018, 1024, 1500, 1529, 1530, 2041, 2042, 2043, 2047, 2048, 3065, 3066,
          4082, 4089, 4095, 4096]


@pytest.mark.parametrize("w", WIDTHS)
def test_edges_of_rows_and_chunks(w):
    heads, h, pad = 1, 6, 16
    g = rng(9000 + w)
    n = heads * h * w
    for start_in, start_out, temp in ((1, 1, 1.0), (3, 3, 0.7), (4, 4, 1.0), (7, 7, 1.0), (0, 5, 1.0), (6, 1, 1.0),
                                      (8, 0, 1.0), (2, 10, 0.7)):
        x = (g.standard_normal((heads, h, w)) * 4).astype(np.float16)
        if w > 4:
            x[0, 1, w // 2:] = -np.inf
            x[0, 2, :w // 2] = np.float16(-65504)
        want = oracle.softmax_rows(x, temp, 0)
        # the neighbours of the tensor are infinities: nothing of them may reach a row
        buf = torch.full((pad + n + pad,), float("inf"), dtype=torch.float16, device="cuda")
        buf[start_in:start_in + n] = to_dev(x).flatten()
        out = torch.full((pad + n + pad,), 9.0, dtype=torch.float16, device="cuda")
        s, lib = torch.cuda.current_stream().cuda_stream, _ffi.lib()
        assert lib.adr_softmax_rows(s, out.data_ptr() + 2 * start_out, buf.data_ptr() + 2 * start_in, heads, h, w,
                                    temp) == 0
        got = to_np(out)
        assert np.max(ulp_diff_f16(got[start_out:start_out + n].reshape(x.shape), want)) <= 1, (w, start_in, start_out)
        assert np.all(got[:start_out] == 9.0) and np.all(got[start_out + n:] == 9.0)
        assert lib.adr_softmax_rows(s, buf.data_ptr() + 2 * start_in, buf.data_ptr() + 2 * start_in, heads, h, w,
                                    temp) == 0
        inplace = to_np(buf)
        assert np.array_equal(inplace[start_in:start_in + n], got[start_out:start_out + n])
        assert np.all(np.isinf(inplace[:start_in])) and np.all(np.isinf(inplace[start_in + n:]))


@pytest.mark.parametrize("rows", [12288, 12289])
@pytest.mark.parametrize("w", [2043, 2046, 2047])
def test_one_more_piece_per_lane_in_few_rows_and_in_many(w, rows):
    g = torch.Generator(device="cuda").manual_seed(w + rows)
    x = torch.randn(1, rows, w, dtype=torch.float16, device="cuda", generator=g) * 4
    want = torch.softmax(x.double(), -1).half()
    s = torch.cuda.current_stream().cuda_stream
    assert _ffi.lib().adr_softmax_rows(s, x.data_ptr(), x.data_ptr(), 1, rows, w, 1.0) == 0
    steps = (x.view(torch.int16).int() - want.view(torch.int16).int()).abs().max()   # (no signs: all are >= 0)
    assert int(steps) <= 1
