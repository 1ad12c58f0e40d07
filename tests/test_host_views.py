"""The views a forward pass makes at each call are built past the checking constructor: over ranks,
orders, inferred dims and permuted or gapped bases they are the layouts that constructor builds, and
what it refuses stays refused."""
import itertools

import pytest
import torch

from adrastea_amd import TensorLayout, TensorView, MatmulMask, MatmulOptions, MatmulStore, MatmulLoad
from adrastea_amd.kernels import lower_matmul


def same(layout, dims, strides):
    want = TensorLayout(tuple(dims), tuple(strides))
    assert layout == want and hash(layout) == hash(want) and repr(layout) == repr(want)
    assert all(type(v) is int for v in layout.dims + layout.strides)


@pytest.mark.parametrize("dims", [(1,), (7,), (3, 5), (1, 1), (4, 1, 6), (2, 3, 4, 5)])
def test_views_are_the_checked_layouts(dims):
    base = torch.zeros(dims, dtype=torch.float16)
    for order in itertools.permutations(range(len(dims))):
        t = base.permute(order)
        same(TensorView.of(t).layout, t.shape, t.stride())
        p = TensorView.of(base).permute(list(order)).layout
        same(p, t.shape, t.stride())
        # a cast keeps the volume and forgets the order
        for new in ([-1], [base.numel()], [1, -1], [dims[0], -1], [base.numel(), 1, 1]):
            want = torch.zeros(base.numel(), dtype=torch.float16).reshape(new)
            same(p.shape_cast(new), want.shape, want.stride())


def test_gapped_rows_and_offsets():
    t = torch.zeros(6, 16, dtype=torch.float16)[1:5, 4:12]
    v = TensorView.of(t)
    same(v.layout, (4, 8), (16, 1))
    assert v.data_ptr() == t.data_ptr()
    assert v.skip([2, 3]).data_ptr() == t[2:, 3:].data_ptr()
    assert v.skip([1, 0]).permute([1, 0]).data_ptr() == t[1:].data_ptr()


def test_what_was_refused_stays_refused():
    with pytest.raises(ValueError):
        TensorView.of(torch.zeros(0, 4))
    with pytest.raises(ValueError):
        TensorView.of(torch.zeros(1, 4).expand(3, 4))      # stride 0
    with pytest.raises(ValueError):
        TensorView.of(torch.zeros(()))
    t = TensorLayout.row_major([4, 6])
    for dims in ([], [-1, -1], [5, -1], [4, 5], [0, 24]):
        with pytest.raises(ValueError):
            t.shape_cast(dims)
    with pytest.raises(ZeroDivisionError):
        t.shape_cast([0, -1])
    for order in ([0], [0, 1, 1]):
        with pytest.raises(ValueError):
            t.permute(order)
    with pytest.raises(IndexError):
        t.permute([0, 2])


@pytest.mark.parametrize("rank", [2, 3])
def test_lowering_names_the_mismatch(rank):
    lead = [2] * (rank - 2)
    out, left, right = (TensorLayout.row_major(lead + d) for d in ([4, 5], [4, 3], [3, 5]))
    low = lower_matmul(out, left, right, MatmulOptions.new().load(MatmulLoad.Scale(0.5))
                       .store(MatmulStore.Scale(0.25)).mask(MatmulMask.CAUSAL))
    z = 1 if rank == 3 else 0
    assert low.scalars() == (2 if z else 1, 4, 3, 5, 1, 5, 20 * z, 1, 3, 12 * z, 1, 5, 15 * z)
    assert (low.beta, low.scale, low.store, low.load, low.mask) == (0.0, 0.125, 4, 1, 1)
    for bad, what in (((out, TensorLayout.row_major(lead + [4, 2]), right), "K"),
                      ((out, TensorLayout.row_major(lead + [6, 3]), right), "M"),
                      ((out, left, TensorLayout.row_major(lead + [3, 6])), "N")):
        with pytest.raises(AssertionError, match=what + " mismatch"):
            lower_matmul(*bad, MatmulOptions.new())
