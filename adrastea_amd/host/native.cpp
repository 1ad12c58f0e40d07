// The host path of the calls a forward pass makes once per layer, as native code: the views of
// activations (TensorView.of / permute / shape_cast) and the lowering of views and options to the
// argument tuples of the C ABI.  tensor.py and kernels.py define what these do; here is the same for
// the forms that occur in earnest (tuples and lists of plain ints, views of this package), and
// everything else -- wrong ranks, sizes that do not match, zero strides, other types -- goes back to
// those definitions, which raise what they always raised.
//
// What bounds the small calls is this path: a launch takes the host 2-2.5 us, and the interpreter took
// 1.9 us for a view of a tensor, 5 for a head view and 6 for a matmul around its launch.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "../../include/adrastea_kernels.h"

namespace {

constexpr int MAX_RANK = 7;  // of a descriptor; views of higher rank take the general path

PyObject *layout_type, *view_type;                      // the classes of tensor.py
PyObject *of_general, *permute_general, *cast_general;  // their definitions of the methods below
PyObject *current_device, *raw_stream;                  // torch's functions
PyObject *s_shape, *s_stride, *s_dims, *s_strides, *s_storage, *s_layout, *s_offset, *s_data_ptr, *s_load, *s_store,
    *s_mask, *s_op, *s_scale, *s_beta, *s_bias, *s_is_contiguous;

decltype(&adr_matmul_f16) matmul_fn;
decltype(&adr_attention_f16) attention_fn;
decltype(&adr_softmax_rows) softmax_fn;
decltype(&adr_matmul_nt_fp16u8) matmul_u8_fn;
decltype(&adr_quantize_absmax_u8) quantize_fn;
decltype(&adr_dequantize_absmax_u8) dequantize_fn;
decltype(&adr_error_stats_f16) error_stats_fn[2];

// A reference that is given back at the end of its scope.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* q) : p(q) {}
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  operator PyObject*() const { return p; }
  PyObject* release() {
    PyObject* q = p;
    p = nullptr;
    return q;
  }
};

// Clears what an Exception reports (the general path raises it again, if it is one of the call's own); false: an
// interrupt or an exit came by on its way through torch's functions, which is the caller's to see.
bool cleared() {
  if (!PyErr_Occurred()) return true;
  if (!PyErr_ExceptionMatches(PyExc_Exception)) return false;
  PyErr_Clear();
  return true;
}

// None to the caller: "take the general path" (which raises if there is something to raise).
PyObject* general() {
  if (!cleared()) return nullptr;
  Py_RETURN_NONE;
}

// An attribute, unless the object is missing or an exception is on its way already.
PyObject* attr(PyObject* o, PyObject* name) { return o && !PyErr_Occurred() ? PyObject_GetAttr(o, name) : nullptr; }
PyObject* call(PyObject* o, PyObject* method) { return o && !PyErr_Occurred() ? PyObject_CallMethodNoArgs(o, method) : nullptr; }

// A plain int that fits 64 bits.
bool as_int(PyObject* o, int64_t& v) {
  if (!o || !PyLong_CheckExact(o)) return false;
  int overflow;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && !(v == -1 && PyErr_Occurred());
}

struct Layout {
  int rank;
  int64_t dims[MAX_RANK], strides[MAX_RANK];
};

// `t` a tuple or a list of `rank` plain ints (rank < 0: any number up to MAX_RANK)
bool read_ints(PyObject* t, int64_t* out, int& rank) {
  if (!t || !(PyTuple_Check(t) || PyList_CheckExact(t))) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(t);
  if (n < 1 || n > MAX_RANK || (rank >= 0 && n != rank)) return false;
  rank = (int)n;
  for (int i = 0; i < rank; i++)
    if (!as_int(PySequence_Fast_GET_ITEM(t, i), out[i])) return false;
  return true;
}

bool read_layout(PyObject* view, Layout& l) {
  const Ref lay(attr(view, s_layout));
  if (!lay.p || (PyObject*)Py_TYPE(lay.p) != layout_type) return false;
  const Ref dims(attr(lay, s_dims)), strides(attr(lay, s_strides));
  l.rank = -1;
  return read_ints(dims, l.dims, l.rank) && read_ints(strides, l.strides, l.rank);
}

bool call_int(PyObject* o, PyObject* method, int64_t& v) {
  const Ref r(call(o, method));
  return as_int(r, v);
}

// data_ptr() of a view or a tensor
bool read_ptr(PyObject* o, void*& p) {
  int64_t v;
  if ((PyObject*)Py_TYPE(o) == view_type) {
    const Ref offset(attr(o, s_offset));
    int64_t at;
    if (!as_int(offset, at)) return false;
    if (at == 0) {
      const Ref storage(attr(o, s_storage));
      if (!storage.p || !call_int(storage, s_data_ptr, v)) return false;
      p = (void*)(uintptr_t)v;
      return true;
    }
  }
  if (!call_int(o, s_data_ptr, v)) return false;
  p = (void*)(uintptr_t)v;
  return true;
}

bool read_double(PyObject* o, double& v) {
  if (!o || !(PyFloat_CheckExact(o) || PyLong_CheckExact(o))) return false;
  v = PyFloat_AsDouble(o);
  return !(v == -1.0 && PyErr_Occurred());
}

// torch's current stream on its current device
bool read_stream(adr_stream_t& s) {
  const Ref dev(PyObject_CallNoArgs(current_device));
  if (!dev.p) return false;
  const Ref raw(PyObject_CallOneArg(raw_stream, dev));
  int64_t v;
  if (!as_int(raw, v)) return false;
  s = (adr_stream_t)(uintptr_t)v;
  return true;
}

PyObject* ints(const int64_t* v, int n) {
  PyObject* t = PyTuple_New(n);
  for (int i = 0; t && i < n; i++) {
    PyObject* x = PyLong_FromLongLong(v[i]);
    if (!x) Py_CLEAR(t);
    else PyTuple_SET_ITEM(t, i, x);
  }
  return t;
}

// A layout of dims and strides that satisfy its constructor, and a view with it; both references of the
// tuples are taken over.
PyObject* make_view(PyObject* storage, PyObject* dims, PyObject* strides, PyObject* offset) {
  const Ref d(dims), s(strides);
  if (!d.p || !s.p) return nullptr;
  const Ref lay(PyType_GenericAlloc((PyTypeObject*)layout_type, 0));
  if (!lay.p || PyObject_GenericSetAttr(lay, s_dims, d) || PyObject_GenericSetAttr(lay, s_strides, s)) return nullptr;
  Ref view(PyType_GenericAlloc((PyTypeObject*)view_type, 0));
  if (!view.p || PyObject_GenericSetAttr(view, s_storage, storage) || PyObject_GenericSetAttr(view, s_layout, lay) ||
      PyObject_GenericSetAttr(view, s_offset, offset))
    return nullptr;
  return view.release();
}

PyObject* view_of(PyObject*, PyObject* const* a, Py_ssize_t n, PyObject* names) {
  if (n == 1 && !names) {
    PyObject* const t = a[0];
    const Ref shape(attr(t, s_shape)), stride(call(t, s_stride));
    int64_t d[MAX_RANK], s[MAX_RANK];
    int rank = -1;
    if (shape.p && stride.p && PyTuple_Check(shape) && PyTuple_CheckExact(stride) && read_ints(shape, d, rank) &&
        read_ints(stride, s, rank)) {
      bool zero = false;
      for (int i = 0; i < rank; i++) zero |= d[i] == 0 || s[i] == 0;
      if (!zero) {
        const Ref none(PyLong_FromLong(0));
        Py_INCREF(stride.p);
        return make_view(t, ints(d, rank), stride, none);
      }
    }
  }
  return cleared() ? PyObject_Vectorcall(of_general, a, n, names) : nullptr;
}

// A method's general definition, with `self` in front of its arguments.
PyObject* call_general(PyObject* method, PyObject* self, PyObject* const* a, Py_ssize_t n, PyObject* names) {
  if (!cleared()) return nullptr;
  const Ref bound(PyMethod_New(method, self));
  return bound.p ? PyObject_Vectorcall(bound, a, n, names) : nullptr;
}

PyObject* view_permute(PyObject* self, PyObject* const* a, Py_ssize_t n, PyObject* names) {
  Layout l;
  int64_t o[MAX_RANK], d[MAX_RANK], s[MAX_RANK];
  if (n == 1 && !names && read_layout(self, l) && read_ints(a[0], o, l.rank)) {
    bool inside = true;
    for (int i = 0; i < l.rank; i++) {
      if (o[i] < 0) o[i] += l.rank;  // (as a Python index)
      inside = inside && o[i] >= 0 && o[i] < l.rank;
      if (inside) d[i] = l.dims[o[i]], s[i] = l.strides[o[i]];
    }
    const Ref storage(attr(self, s_storage)), offset(attr(self, s_offset));
    if (inside && storage.p && offset.p && PyLong_CheckExact(offset))
      return make_view(storage, ints(d, l.rank), ints(s, l.rank), offset);
  }
  return call_general(permute_general, self, a, n, names);
}

PyObject* view_shape_cast(PyObject* self, PyObject* const* a, Py_ssize_t nargs, PyObject* names) {
  Layout l;
  int64_t d[MAX_RANK], s[MAX_RANK], vol = 1, known = 1;
  int n = -1, inferred = 0, at = 0;
  bool ok = nargs == 1 && !names && read_layout(self, l) && read_ints(a[0], d, n);
  for (int i = 0; ok && i < l.rank; i++) ok = l.dims[i] > 0 && !__builtin_mul_overflow(vol, l.dims[i], &vol);
  for (int i = 0; ok && i < n; i++) {
    if (d[i] < 0) inferred++, at = i;
    else ok = d[i] > 0 && !__builtin_mul_overflow(known, d[i], &known);
  }
  if (ok && inferred == 1) ok = vol % known == 0, d[at] = vol / known;
  else ok = ok && inferred == 0 && known == vol;
  if (ok) {
    int64_t step = 1;
    for (int i = n - 1; i >= 0; i--) s[i] = step, step *= d[i];
    const Ref storage(attr(self, s_storage)), offset(attr(self, s_offset));
    if (storage.p && offset.p && PyLong_CheckExact(offset)) return make_view(storage, ints(d, n), ints(s, n), offset);
  }
  return call_general(cast_general, self, a, nargs, names);
}

// One dimension or stride as the 32-bit argument it becomes (as ctypes converts it).
int32_t i32(int64_t v) { return (int32_t)(uint32_t)(uint64_t)v; }
int64_t last(const int64_t* v, const Layout& l, int from_end) { return v[l.rank - from_end]; }
// the batch stride: 0 for rank 2
int32_t z(const Layout& l) { return l.rank > 2 ? i32(last(l.strides, l, 3)) : 0; }

// matmul_f16(output, left, right, options) -> the C call's result, or None
PyObject* matmul_f16(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Layout o, l, r;
  if (n != 4 || !matmul_fn || !read_layout(a[0], o) || !read_layout(a[1], l) || !read_layout(a[2], r) || o.rank < 2 ||
      l.rank < 2 || r.rank < 2)
    return general();
  const int64_t M = last(l.dims, l, 2), K = last(l.dims, l, 1), N = last(r.dims, r, 1);
  if (K != last(r.dims, r, 2) || last(o.dims, o, 2) != M || last(o.dims, o, 1) != N) return general();
  const Ref load(attr(a[3], s_load)), store(attr(a[3], s_store)), mask(attr(a[3], s_mask));
  if (!load.p || !store.p) return general();
  const Ref load_op(attr(load, s_op)), store_op(attr(store, s_op)), bias(attr(store, s_bias));
  int64_t lop, sop, msk;
  if (!as_int(load_op, lop) || !as_int(store_op, sop) || !as_int(mask, msk) || !bias.p) return general();
  double scale = 1.0, beta = 0.0, v;
  if (lop == 1) {
    const Ref f(attr(load, s_scale));
    if (!read_double(f, scale)) return general();
  }
  if (sop == 4) {
    const Ref f(attr(store, s_scale));
    if (!read_double(f, v)) return general();
    scale *= v;
  }
  if (sop == 2 || sop == 3) {
    const Ref f(attr(store, s_beta));
    if (!read_double(f, beta)) return general();
  }
  adr_stream_t stream;
  void *po, *pl, *pr, *pb = nullptr;
  if (!read_stream(stream) || !read_ptr(a[0], po) || !read_ptr(a[1], pl) || !read_ptr(a[2], pr) ||
      (bias != Py_None && !read_ptr(bias, pb)))
    return general();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = matmul_fn(stream, (uint16_t*)po, (const uint16_t*)pl, (const uint16_t*)pr, o.rank > 2 ? i32(last(o.dims, o, 3)) : 1,
                 i32(M), i32(K), i32(N), i32(last(o.strides, o, 1)), i32(last(o.strides, o, 2)), z(o),
                 i32(last(l.strides, l, 1)), i32(last(l.strides, l, 2)), z(l), i32(last(r.strides, r, 1)),
                 i32(last(r.strides, r, 2)), z(r), (const uint16_t*)pb, (float)beta, (float)scale, (uint32_t)sop,
                 (uint32_t)lop, (uint32_t)msk);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// attention_f16(output, query, key, value, scale, temperature, mask)
PyObject* attention_f16(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Layout o, q, k, v;
  if (n != 7 || !attention_fn || !read_layout(a[0], o) || !read_layout(a[1], q) || !read_layout(a[2], k) ||
      !read_layout(a[3], v))
    return general();
  const int rank = q.rank;
  if ((rank != 2 && rank != 3) || o.rank != rank || k.rank != rank || v.rank != rank) return general();
  const int64_t m = last(q.dims, q, 2), d = last(q.dims, q, 1), keys = last(k.dims, k, 2);
  if (last(k.dims, k, 1) != d || last(v.dims, v, 1) != d || last(v.dims, v, 2) != keys || last(o.dims, o, 2) != m ||
      last(o.dims, o, 1) != d)
    return general();
  const int64_t heads = rank == 3 ? q.dims[0] : 1;
  if (rank == 3 && (o.dims[0] != heads || k.dims[0] != heads || v.dims[0] != heads)) return general();
  double scale, temp;
  int64_t mask;
  adr_stream_t stream;
  void *po, *pq, *pk, *pv;
  if (!read_double(a[4], scale) || !read_double(a[5], temp) || !as_int(a[6], mask) || !read_stream(stream) ||
      !read_ptr(a[0], po) || !read_ptr(a[1], pq) || !read_ptr(a[2], pk) || !read_ptr(a[3], pv))
    return general();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  auto x = [](const Layout& t) { return i32(last(t.strides, t, 1)); };
  auto y = [](const Layout& t) { return i32(last(t.strides, t, 2)); };
  rc = attention_fn(stream, (uint16_t*)po, (const uint16_t*)pq, (const uint16_t*)pk, (const uint16_t*)pv, i32(heads), i32(m),
                    i32(keys), i32(d), x(o), y(o), z(o), x(q), y(q), z(q), x(k), y(k), z(k), x(v), y(v), z(v), (float)scale,
                    (float)temp, (uint32_t)mask);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// softmax_rows_inplace(output, temperature)
PyObject* softmax_rows_inplace(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Layout l;
  double temp;
  if (n != 2 || !softmax_fn || !read_layout(a[0], l) || l.rank < 2 || !read_double(a[1], temp)) return general();
  int64_t step = 1;
  for (int i = l.rank - 1; i >= 0; i--)
    if (l.strides[i] != step || __builtin_mul_overflow(step, l.dims[i], &step)) return general();
  adr_stream_t stream;
  void* p;
  if (!read_stream(stream) || !read_ptr(a[0], p)) return general();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = softmax_fn(stream, (uint16_t*)p, (const uint16_t*)p, l.rank > 2 ? i32(last(l.dims, l, 3)) : 1, i32(last(l.dims, l, 2)),
                  i32(last(l.dims, l, 1)), (float)temp);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

bool read_shape(PyObject* t, int64_t (&d)[MAX_RANK], int rank) {
  const Ref shape(attr(t, s_shape));
  return shape.p && PyTuple_Check(shape) && read_ints(shape, d, rank);
}

bool is_contiguous(PyObject* t) {
  const Ref r(call(t, s_is_contiguous));
  return r == Py_True;
}

// matmul_nt_fp16u8(output, lhs, rhs_q, scales, block_size, beta)
PyObject* matmul_nt_fp16u8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t o[MAX_RANK], l[MAX_RANK], r[MAX_RANK], s[MAX_RANK], block;
  double beta;
  if (n != 6 || !matmul_u8_fn || !read_shape(a[0], o, 2) || !read_shape(a[1], l, 2) || !read_shape(a[2], r, 2) ||
      !read_shape(a[3], s, 2) || !as_int(a[4], block) || block < 1 || !read_double(a[5], beta) || r[1] != l[1] ||
      o[0] != l[0] || o[1] != r[0] || s[0] != r[0] || s[1] != l[1] / block)
    return general();
  adr_stream_t stream;
  void* p[4];
  for (int i = 0; i < 4; i++)
    if (!is_contiguous(a[i]) || !read_ptr(a[i], p[i])) return general();
  if (!read_stream(stream)) return general();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = matmul_u8_fn(stream, (uint16_t*)p[0], (const uint16_t*)p[1], (const uint8_t*)p[2], (const uint16_t*)p[3], i32(l[0]),
                    i32(l[1]), i32(r[0]), i32(block), (float)beta);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// (wide, scales, other): the tensor whose shape counts, its scales, and the third of the call
bool read_quant(PyObject* wide, PyObject* scales, PyObject* other, int64_t (&d)[MAX_RANK], int64_t& block, void* (&p)[3],
                adr_stream_t& stream) {
  int64_t s[MAX_RANK];
  if (!read_shape(wide, d, 2) || !read_shape(scales, s, 2) || s[1] < 1) return false;
  block = d[1] / s[1];
  return read_stream(stream) && read_ptr(wide, p[0]) && read_ptr(scales, p[1]) && read_ptr(other, p[2]);
}

// quantize_absmax_uint8(q, scales, x)
PyObject* quantize_absmax_uint8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t d[MAX_RANK], block;
  void* p[3];
  adr_stream_t stream;
  if (n != 3 || !quantize_fn || !read_quant(a[2], a[1], a[0], d, block, p, stream)) return general();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = quantize_fn(stream, (uint8_t*)p[2], (uint16_t*)p[1], (const uint16_t*)p[0], i32(d[0]), i32(d[1]), i32(block));
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// dequantize_absmax_uint8(output, scales, q)
PyObject* dequantize_absmax_uint8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t d[MAX_RANK], block;
  void* p[3];
  adr_stream_t stream;
  if (n != 3 || !dequantize_fn || !read_quant(a[2], a[1], a[0], d, block, p, stream)) return general();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = dequantize_fn(stream, (uint16_t*)p[2], (const uint8_t*)p[0], (const uint16_t*)p[1], i32(d[0]), i32(d[1]), i32(block));
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// error_stats(output, lhs, rhs, 0 or 1): fp16 or fp32 operands, flattened
PyObject* error_stats(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Layout o;
  int64_t which, count[2];
  adr_tensor_desc desc[3] = {};
  if (n != 4 || !as_int(a[3], which) || which < 0 || which > 1 || !error_stats_fn[which] || !read_layout(a[0], o)) return general();
  desc[0].dims = (uint32_t)o.rank;
  for (int i = 0; i < o.rank; i++) {
    desc[0].shape[i] = (uint32_t)o.dims[o.rank - 1 - i];
    desc[0].strides[i] = (uint32_t)o.strides[o.rank - 1 - i];
  }
  for (int t = 0; t < 2; t++) {
    Layout l;
    if (!read_layout(a[1 + t], l)) return general();
    count[t] = 1;
    for (int i = 0; i < l.rank; i++)
      if (l.dims[i] < 1 || __builtin_mul_overflow(count[t], l.dims[i], &count[t])) return general();
    desc[1 + t].dims = 1;
    desc[1 + t].shape[0] = (uint32_t)count[t];
    desc[1 + t].strides[0] = 1;
  }
  adr_stream_t stream;
  if (count[0] != count[1] || !read_stream(stream)) return general();
  for (int t = 0; t < 3; t++)
    if (!read_ptr(a[t], desc[t].ptr)) return general();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = error_stats_fn[which](stream, desc[0], desc[1], desc[2]);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

#define ADR_METHOD(f) (PyCFunction)(void (*)(void))f, METH_FASTCALL | METH_KEYWORDS
PyMethodDef of_def = {"of", ADR_METHOD(view_of), "View of a torch tensor with its own sizes and strides."};
PyMethodDef permute_def = {"permute", ADR_METHOD(view_permute), nullptr};
PyMethodDef cast_def = {"shape_cast", ADR_METHOD(view_shape_cast), nullptr};

// install(TensorLayout, TensorView): the view's three methods become the ones above, with the classes'
// own definitions behind them
PyObject* install(PyObject*, PyObject* args) {
  PyObject *layout, *view;
  if (!PyArg_ParseTuple(args, "O!O!", &PyType_Type, &layout, &PyType_Type, &view)) return nullptr;
  const Ref of(PyObject_GetAttrString(view, "of")), permute(PyObject_GetAttrString(view, "permute")),
      cast(PyObject_GetAttrString(view, "shape_cast"));
  if (!of.p || !permute.p || !cast.p) return nullptr;
  Py_INCREF(layout), Py_INCREF(view), Py_INCREF(of.p), Py_INCREF(permute.p), Py_INCREF(cast.p);
  layout_type = layout, view_type = view, of_general = of, permute_general = permute, cast_general = cast;
  const Ref f(PyCFunction_New(&of_def, nullptr)), p(PyDescr_NewMethod((PyTypeObject*)view, &permute_def)),
      c(PyDescr_NewMethod((PyTypeObject*)view, &cast_def));
  if (!f.p || !p.p || !c.p) return nullptr;
  const Ref s(PyStaticMethod_New(f));
  if (!s.p || PyObject_SetAttrString(view, "of", s) || PyObject_SetAttrString(view, "permute", p) ||
      PyObject_SetAttrString(view, "shape_cast", c))
    return nullptr;
  Py_RETURN_NONE;
}

// bind(the library's ABI version, addresses of its functions ..., torch.cuda.current_device, torch's raw stream of a
// device).  The signatures above are those of the header at this module's own build.
PyObject* bind(PyObject*, PyObject* args) {
  int abi;
  unsigned long long p[8];
  PyObject *dev, *raw;
  if (!PyArg_ParseTuple(args, "iKKKKKKKKOO", &abi, p, p + 1, p + 2, p + 3, p + 4, p + 5, p + 6, p + 7, &dev, &raw)) return nullptr;
  if (abi != ADR_ABI_VERSION)
    return PyErr_Format(PyExc_RuntimeError,
                        "adrastea_amd._native was built for ABI version %d, the library has %d: build both "
                        "with `python -m adrastea_amd.build`", ADR_ABI_VERSION, abi);
  matmul_fn = (decltype(matmul_fn))p[0];
  attention_fn = (decltype(attention_fn))p[1];
  softmax_fn = (decltype(softmax_fn))p[2];
  matmul_u8_fn = (decltype(matmul_u8_fn))p[3];
  quantize_fn = (decltype(quantize_fn))p[4];
  dequantize_fn = (decltype(dequantize_fn))p[5];
  error_stats_fn[0] = (decltype(&adr_error_stats_f16))p[6];
  error_stats_fn[1] = (decltype(&adr_error_stats_f16))p[7];
  Py_INCREF(dev), Py_INCREF(raw);
  Py_XSETREF(current_device, dev);
  Py_XSETREF(raw_stream, raw);
  Py_RETURN_NONE;
}

#define ADR_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"install", install, METH_VARARGS, nullptr},
                         {"bind", bind, METH_VARARGS, nullptr},
                         ADR_FAST(matmul_f16),
                         ADR_FAST(attention_f16),
                         ADR_FAST(softmax_rows_inplace),
                         ADR_FAST(matmul_nt_fp16u8),
                         ADR_FAST(quantize_absmax_uint8),
                         ADR_FAST(dequantize_absmax_uint8),
                         ADR_FAST(error_stats),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  const struct { PyObject** at; const char* name; } names[] = {
      {&s_shape, "shape"}, {&s_stride, "stride"}, {&s_dims, "dims"}, {&s_strides, "strides"}, {&s_storage, "storage"},
      {&s_layout, "layout"}, {&s_offset, "offset"}, {&s_data_ptr, "data_ptr"}, {&s_load, "load_"}, {&s_store, "store_"},
      {&s_mask, "mask_"}, {&s_op, "op"}, {&s_scale, "scale"}, {&s_beta, "beta"}, {&s_bias, "bias"},
      {&s_is_contiguous, "is_contiguous"}};
  for (const auto& n : names)
    if (!(*n.at = PyUnicode_InternFromString(n.name))) return nullptr;
  return PyModule_Create(&module);
}
