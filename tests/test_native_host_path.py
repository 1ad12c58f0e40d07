"""The native host path (host/native.cpp) against the definitions in tensor.py and kernels.py, on the CPU: views
over ranks, orders and casts, what those refuse, and the argument tuples that reach the C ABI, through callbacks
in the place of the library's functions."""
import ctypes as C
import itertools
import os
import shutil
import sysconfig
import warnings

import pytest
import torch

from adrastea_amd import GpuKernels, MatmulLoad, MatmulMask, MatmulOptions, MatmulStore, TensorLayout, TensorView, _ffi
from adrastea_amd import kernels
from adrastea_amd.kernels import _NATIVE_CALLS, _bind_native, descriptor, _lower
from adrastea_amd.tensor import _native

ABI = _ffi.lib().adr_abi_version()
built = pytest.mark.skipif(_native is None, reason="the native module is not built (test_the_module_is_built)")


def test_the_module_is_built():
    """Where it can be: the tests below say nothing of a module that is not there."""
    if shutil.which("g++") is None or not os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h")):
        pytest.skip("no C++ compiler or no headers of the interpreter")
    assert _native is not None


class Heads(TensorView):
    pass


@built
@pytest.mark.parametrize("dims", [(1,), (6,), (3, 4), (1, 5, 1), (2, 3, 4), (2, 1, 3, 2, 2, 1, 2)])
def test_views(dims):
    t = torch.zeros(dims, dtype=torch.float16)
    v = TensorView.of(t)
    assert type(v) is TensorView and v.storage is t and v.offset == 0 and TensorView.of(t=t).layout == v.layout
    assert v.layout == TensorLayout(tuple(dims), t.stride()) and type(v.layout.dims) is tuple
    shifted = Heads(t, v.layout, 3)
    for order in itertools.islice(itertools.permutations(range(len(dims))), 30):
        order = [i - len(dims) if i % 2 else i for i in order]   # (negative indices too)
        for o in (order, tuple(order)):
            p = shifted.permute(o)
            assert p.layout == v.layout.permute(o) and p.offset == 3 and p.storage is t and type(p) is TensorView
        assert shifted.permute(order=order).layout == p.layout
        for cast in ([-1], (t.numel(),), [1, -1, 1], [dims[0], -1], [t.numel(), 1]):
            assert p.shape_cast(cast).layout == p.layout.shape_cast(cast) and p.shape_cast(cast).offset == 3
        assert p.shape_cast(dims=[-1]).layout == p.layout.shape_cast([-1])
    with pytest.raises(AttributeError):
        v.layout.dims = (1,)                                      # (still frozen)
    eight = TensorView.of(torch.zeros((1,) * 8))                  # past the native path's ranks
    assert eight.permute(list(range(8))).layout == eight.layout


@built
@pytest.mark.parametrize("method,args", [
    ("permute", ([0],)), ("permute", ([0, 2],)), ("permute", ([0, 1, 1],)), ("permute", ("01",)), ("permute", (None,)),
    ("permute", ()), ("permute", ([0, 1], 2)), ("permute", ([0.0, 1],)), ("permute", ([True, False],)),
    ("shape_cast", ([],)), ("shape_cast", ([-1, -1],)), ("shape_cast", ([5, -1],)), ("shape_cast", ([0, -1],)),
    ("shape_cast", ([4, 7],)), ("shape_cast", ([0, 24],)), ("shape_cast", ([1 << 70, -1],)), ("shape_cast", (24,)),
    ("shape_cast", ([4.0, 6.0],)), ("shape_cast", ())])
def test_unusual_arguments_do_what_the_definition_does(method, args):
    view = TensorView.of(torch.zeros(4, 6))

    def outcome(f):
        try:
            return getattr(f(*args), "layout", None)
        except Exception as e:
            return type(e)
    want = outcome(lambda *a: TensorView(view.storage, getattr(view.layout, method)(*a), 0))
    assert outcome(getattr(view, method)) == want


@built
def test_tensors_without_a_layout():
    for t in (torch.zeros(0, 4), torch.zeros(()), torch.zeros(1, 4).expand(3, 4)):
        with pytest.raises(ValueError):
            TensorView.of(t)
    with pytest.raises(AttributeError):
        TensorView.of(3)


@pytest.fixture
def calls():
    """Callbacks in the place of the library's functions: the tuples they were called with, as ctypes sees them."""
    lib, seen, keep = _ffi.lib(), [], []
    for name in _NATIVE_CALLS:
        types = getattr(lib, name).argtypes
        if _ffi.TensorDesc in types:   # (callbacks take no structures by value that large)
            keep.append(None)
            continue
        keep.append(C.CFUNCTYPE(C.c_int, *types)(lambda *a, name=name: seen.append((name, a)) or 7))
    _native.bind(ABI, *(C.cast(f, C.c_void_p).value if f else 0 for f in keep), lambda: 3, lambda dev: 0x1000 + dev)
    yield seen
    _bind_native()   # (what every GpuKernels of this process is bound to)


def as_ctypes(name, args):
    """What ctypes makes of a call's arguments."""
    out = []
    for t, a in zip(getattr(_ffi.lib(), name).argtypes, args):
        out.append(t(a).value)
    return tuple(out)


STORES = [MatmulStore.Identity(), MatmulStore.Add(), MatmulStore.Scale(0.3),
          MatmulStore.BetaBias(0.7, TensorView.of(torch.zeros(5, dtype=torch.float16))),
          MatmulStore.QuickGeluBias(TensorView(torch.zeros(9, dtype=torch.float16), TensorLayout((5,), (1,)), 2)),
          MatmulStore.BetaGeluBias(1, TensorView.of(torch.zeros(5, dtype=torch.float16)))]


@built
@pytest.mark.parametrize("store", STORES, ids=lambda s: str(s.op))
@pytest.mark.parametrize("rank_o,rank_l,rank_r", [(2, 2, 2), (3, 3, 3), (3, 3, 2), (3, 2, 3), (4, 4, 2)])
def test_matmul_arguments(calls, store, rank_o, rank_l, rank_r):
    def view(rank, a, b, turn=False):
        t = torch.zeros(*[2] * (rank - 2), a, b, dtype=torch.float16)
        v = TensorView.of(t)
        return TensorView.of(t.transpose(-1, -2).contiguous()).permute([*range(rank - 2), -1, -2]) if turn else v
    out, left, right = view(rank_o, 4, 5), view(rank_l, 4, 3).skip([0] * rank_l), view(rank_r, 3, 5, turn=True)
    options = MatmulOptions.new().store(store).load(MatmulLoad.Scale(0.1)).mask(MatmulMask.CAUSAL)
    assert _native.matmul_f16(out, left, right, options) == 7
    scalars, tail = _lower(out.layout, left.layout, right.layout, options)
    want = as_ctypes("adr_matmul_f16", (0x1003, out.data_ptr(), left.data_ptr(), right.data_ptr(), *scalars,
                                       store.bias.data_ptr() if store.bias is not None else None, *tail))
    assert calls == [("adr_matmul_f16", want)]
    for bad in ((view(rank_o, 4, 6), left, right), (out, view(rank_l, 4, 2), right), (view(rank_o, 3, 5), left, right),
                (TensorView.of(torch.zeros(4)), left, right), (out, object(), right)):
        assert _native.matmul_f16(*bad, options) is None
    assert len(calls) == 1


@built
@pytest.mark.parametrize("rank", [2, 3])
def test_attention_and_softmax_arguments(calls, rank):
    def view(rows, d=64, heads=3):
        v = TensorView.of(torch.zeros(rows, heads * d, dtype=torch.float16))
        return v.shape_cast([rows, heads, d]).permute([1, 0, 2]) if rank == 3 else v
    o, q, k, v = view(5), view(5), view(9), view(9)
    assert _native.attention_f16(o, q, k, v, 0.125, 1, 1) == 7
    strides = [s for t in (o, q, k, v) for s in (t.stride(-1), t.stride(-2), t.stride(0) if rank == 3 else 0)]
    want = as_ctypes("adr_attention_f16", (0x1003, *(t.data_ptr() for t in (o, q, k, v)), 3 if rank == 3 else 1, 5, 9,
                                           64 if rank == 3 else 192, *strides, 0.125, 1.0, 1))
    assert calls == [("adr_attention_f16", want)]
    for bad in ((o, q, k, view(8)), (view(4), q, k, v), (o, q, view(9, 32), v), (o, view(5, heads=2), k, v)):
        assert _native.attention_f16(*bad, 0.125, 1.0, 0) is None
    assert _native.attention_f16(o, q, k, v, torch.tensor(0.1), 1.0, 0) is None   # (the general path converts it)
    del calls[:]
    s = TensorView.of(torch.zeros(*[2] * (rank - 2), 5, 7, dtype=torch.float16))
    assert _native.softmax_rows_inplace(s, 0.5) == 7
    assert calls == [("adr_softmax_rows", as_ctypes("adr_softmax_rows", (0x1003, s.data_ptr(), s.data_ptr(),
                                                                        2 if rank == 3 else 1, 5, 7, 0.5)))]
    assert _native.softmax_rows_inplace(s.permute([*range(rank - 2), -1, -2]), 0.5) is None
    assert _native.softmax_rows_inplace(TensorView.of(torch.zeros(7)), 0.5) is None


@built
def test_u8_and_quantisation_arguments(calls):
    m, p, n, bs = 3, 64, 5, 32
    out, x = torch.zeros(m, n, dtype=torch.float16), torch.zeros(m, p, dtype=torch.float16)
    q, s = torch.zeros(n, p, dtype=torch.uint8), torch.zeros(n, p // bs, dtype=torch.float16)
    assert _native.matmul_nt_fp16u8(out, x, q, s, bs, 0.5) == 7
    assert _native.quantize_absmax_uint8(q, s, torch.zeros(n, p, dtype=torch.float16)) == 7
    w = torch.zeros(n, p, dtype=torch.float16)
    assert _native.dequantize_absmax_uint8(w, s, q) == 7
    ptr = [t.data_ptr() for t in (out, x, q, s, w)]
    assert calls[0] == ("adr_matmul_nt_fp16u8", as_ctypes("adr_matmul_nt_fp16u8", (0x1003, *ptr[:4], m, p, n, bs, 0.5)))
    assert calls[1][1][:3] == (0x1003, ptr[2], ptr[3]) and calls[1][1][4:] == (n, p, bs)
    assert calls[2][1] == (0x1003, ptr[4], ptr[2], ptr[3], n, p, bs)
    for bad in ((out, x, q, s, 16, 0.0), (out, x, q[:, :32], s, bs, 0.0), (out, x.t(), q, s, bs, 0.0), (out, x, q, s, 0, 0.0),
                (torch.zeros(n, m).t(), x, q, s, bs, 0.0)):
        assert _native.matmul_nt_fp16u8(*bad) is None
    assert _native.quantize_absmax_uint8(q, torch.zeros(n, 0), w) is None
    assert len(calls) == 3


@built
def test_error_stats_descriptors():
    """Callbacks take no structures by value that large: the descriptors are compared through the results
    (test_gpu_error_stats.py); here, what the native path hands back."""
    out, a = TensorView.of(torch.zeros(3)), TensorView.of(torch.zeros(4, 6, dtype=torch.float16))
    assert descriptor(a.shape_cast([-1])).shape[0] == 24
    _native.bind(ABI, *([0] * len(_NATIVE_CALLS)), lambda: 0, lambda dev: 0)
    try:
        assert _native.error_stats(out, a, a, 0) is None
        assert _native.error_stats(out, a, a, 2) is None
    finally:
        _bind_native()


class Interrupted:
    """A tensor whose attributes and methods report what they are given."""
    def __init__(self, what):
        self.what = what

    def raised(self, *_):
        raise self.what
    shape = property(raised)
    stride = data_ptr = is_contiguous = raised


@built
@pytest.mark.parametrize("what", [KeyboardInterrupt, SystemExit])
def test_an_interrupt_is_not_taken_for_an_unusual_argument(calls, what):
    """A signal's handler runs inside the functions that the native path calls: an interrupt goes on to the caller,
    and nothing is launched; an Exception goes back to the definitions, which raise it themselves."""
    x = TensorView.of(torch.zeros(4, 4, dtype=torch.float16))
    for error in (what, RuntimeError):
        inside = Interrupted(error)
        with pytest.raises(error):
            TensorView.of(inside)
        view = TensorView(inside, x.layout, 0)
        attempts = [lambda: _native.matmul_f16(x, view, x, MatmulOptions()), lambda: _native.matmul_f16(x, x, x, inside),
                    lambda: _native.softmax_rows_inplace(view, 1.0),
                    lambda: _native.quantize_absmax_uint8(inside, x.storage, x.storage),
                    lambda: _native.matmul_nt_fp16u8(inside, inside, inside, inside, 32, 0.0)]
        Interrupted.load_ = Interrupted.shape
        try:
            for attempt in attempts:
                if error is RuntimeError:
                    assert attempt() is None
                else:
                    with pytest.raises(what):
                        attempt()
        finally:
            del Interrupted.load_

        def device():
            raise error
        _native.bind(ABI, *([0x1000] * len(_NATIVE_CALLS)), device, lambda dev: 0)   # (never called: the stream comes first)
        if error is RuntimeError:
            assert _native.softmax_rows_inplace(x, 1.0) is None
        else:
            with pytest.raises(what):
                _native.softmax_rows_inplace(x, 1.0)
    assert calls == []


@built
def test_a_tensor_without_a_shape_is_asked_no_further():
    class Strange:
        asked = 0

        def stride(self):
            Strange.asked += 1
            return (1,)
    with pytest.raises(AttributeError, match="shape"):
        TensorView.of(Strange())
    assert Strange.asked == 0   # (the definition reads the shape first as well)


@built
def test_a_library_of_another_abi_is_refused():
    for abi in (ABI - 1, ABI + 1):
        with pytest.raises(RuntimeError, match="ABI version"):
            _native.bind(abi, *([0] * len(_NATIVE_CALLS)), lambda: 0, lambda dev: 0)


def test_the_library_is_built_without_a_compiler_for_the_native_module(monkeypatch, capsys):
    from adrastea_amd import build
    done = []
    for name in ("build_library", "build_stamps_library", "build_legacy_modules", "build_host_test"):
        monkeypatch.setattr(build, name, lambda force, name=name: done.append(name))
    for error in (RuntimeError("no Python.h"), FileNotFoundError("g++")):
        def native(force):
            raise error
        monkeypatch.setattr(build, "build_native_module", native)
        build.main()
        assert str(error) in capsys.readouterr().err
    assert done == 2 * ["build_library", "build_stamps_library", "build_legacy_modules", "build_host_test"]


def test_a_module_that_does_not_load_is_reported(tmp_path, monkeypatch):
    from importlib.machinery import EXTENSION_SUFFIXES
    from adrastea_amd import tensor
    assert tensor._load_native("adrastea_amd.no_such_module") is None
    (tmp_path / ("broken_native" + EXTENSION_SUFFIXES[0])).write_bytes(b"no shared object")
    monkeypatch.syspath_prepend(tmp_path)
    with pytest.raises(ImportError):
        tensor._load_native("broken_native")
    # without the module the kernels say so; with it they say nothing
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        GpuKernels()
        monkeypatch.setattr(kernels, "_native", None)
        with pytest.raises(RuntimeWarning, match="_native"):
            GpuKernels()


@built
@pytest.mark.gpu
def test_both_paths_give_the_same_results(monkeypatch):
    """Every call the native path lowers, against the definitions in kernels.py, end to end."""
    gen = torch.Generator(device="cuda").manual_seed(12)

    def normal(*shape):
        return torch.randn(*shape, dtype=torch.float16, device="cuda", generator=gen)

    def heads(t):
        return TensorView.of(t).shape_cast([t.shape[0], 3, 64]).permute([1, 0, 2])
    x, w, bias, q, kv = normal(70, 192), normal(80, 192), normal(80), normal(33, 192), normal(50, 192)
    options = MatmulOptions.new().store(MatmulStore.BetaBias(0.5, TensorView.of(bias)))
    masked = MatmulOptions.new().store(MatmulStore.Scale(0.125)).load(MatmulLoad.Scale(0.5)).mask(MatmulMask.CAUSAL)

    def results():
        k, view = GpuKernels(), TensorView.of
        product, scores, fused = torch.ones_like(normal(70, 80)), torch.ones_like(normal(3, 33, 50)), torch.ones_like(q)
        k.matmul_f16(view(product), view(x), view(w).permute([1, 0]), options)
        k.matmul_f16(view(scores), heads(q), heads(kv).permute([0, 2, 1]), masked)
        k.softmax_rows_inplace(view(scores), 0.7)
        k.attention_f16(heads(fused), heads(q), heads(kv), heads(kv), 0.125, 0.9, MatmulMask.CAUSAL)
        u8, scales = torch.zeros(80, 192, dtype=torch.uint8, device="cuda"), torch.zeros_like(w[:, :6]).contiguous()
        k.quantize_absmax_uint8(u8, scales, w)
        back, by_u8 = torch.zeros_like(w), torch.ones_like(product)
        k.dequantize_absmax_uint8(back, scales, u8)
        k.matmul_nt_fp16u8(by_u8, x, u8, scales, 32, 0.25)
        stats, stats32 = torch.zeros(3, device="cuda"), torch.zeros(3, device="cuda")
        k.error_stats_f16(view(stats), view(back), view(w))
        k.error_stats_f32(view(stats32), view(back.float()), view(w.float()))
        return product, scores, fused, u8, scales, back, by_u8, stats, stats32
    native = results()
    monkeypatch.setattr(kernels, "_native", None)
    with pytest.warns(RuntimeWarning):
        general = results()
    for got, want in zip(native[:-2], general[:-2]):
        assert torch.equal(got, want)
    for got, want in zip(native[-2:], general[-2:]):   # (sums of atomics: the order is not fixed)
        assert torch.allclose(got, want, rtol=1e-5, atol=0)


@built
def test_the_binding_is_looked_up_once(monkeypatch):
    """A program that makes its kernels for each state pays for the addresses once."""
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    kernels._native_binding.cache_clear()
    for _ in range(3):
        GpuKernels()
    assert kernels._native_binding.cache_info().misses == 1
