// Native forms of the hottest launchers of row_kernels.py, as a CPython
// module (_launch), and held_state, a check that a decode step makes.
//
// A launcher called from Python costs more than its kernel at small sizes:
// 7 to 16 us of attribute reads, checks, tensor allocations and a ctypes
// call, against 2 to 8 us of kernel. Here the operands are checked and the
// outputs allocated on at::Tensor, and the library is called directly.
//
// Each launcher takes a well-formed call only: it returns None, with nothing
// launched or changed, as soon as an operand is anything but what
// row_kernels.py would accept as it stands, and the Python launcher then
// handles the call (it raises, converts or allocates as it always did). A
// failed launch raises the RuntimeError of _hip.check. The GIL is released
// around allocation and launch, as torch and ctypes do.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <new>
#include <stdexcept>
#include <vector>

#include "nhs.h"

namespace {

using at::Tensor;

struct Skip {};  // not a call for the native path

void need(bool ok) {
  if (!ok) throw Skip();
}

const Tensor& tensor(PyObject* o) {
  need(THPVariable_Check(o));
  return THPVariable_Unpack(o);
}

int64_t integer(PyObject* o) {
  need(PyLong_CheckExact(o));
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Skip();
  }
  return v;
}

int32_t integer32(PyObject* o) {
  const int64_t v = integer(o);
  need(v >= INT32_MIN && v <= INT32_MAX);
  return (int32_t)v;
}

bool truth(PyObject* o) {
  need(o == Py_True || o == Py_False);
  return o == Py_True;
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return NHS_F32;
    case at::kHalf: return NHS_F16;
    case at::kBFloat16: return NHS_BF16;
    default: throw Skip();
  }
}

bool is_half(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }

// Plain strided GPU tensor with elements, sizes that fit the library's 32-bit arguments.
void on_gpu(const Tensor& t, int64_t dim) {
  need(t.is_cuda() && t.layout() == at::kStrided && t.dim() == dim && t.numel() > 0 && !t.is_neg());
  for (int64_t s : t.sizes()) need(s <= INT32_MAX);
}

void on_gpu(const Tensor& t, int64_t dim, const Tensor& other) {
  on_gpu(t, dim);
  need(t.device() == other.device());
}

bool same_sizes(const Tensor& t, at::IntArrayRef sizes) { return t.sizes() == sizes; }

// Whether dimensions from `first` on are laid out contiguously.
bool contiguous_from(const Tensor& t, int64_t first) {
  int64_t expected = 1;
  for (int64_t d = t.dim() - 1; d >= first; --d) {
    if (t.size(d) != 1 && t.stride(d) != expected) return false;
    expected *= t.size(d);
  }
  return true;
}

Tensor make(at::IntArrayRef sizes, const Tensor& like, at::ScalarType type) {
  return at::empty(sizes, like.options().dtype(type).requires_grad(false));
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// Bytes between the blocks of a pool [blocks, 2, P, Hkv, D].
int64_t pool_block_stride(const Tensor& pool) {
  const int64_t P = pool.size(2), H = pool.size(3), D = pool.size(4);
  need(pool.size(1) == 2 && pool.stride(1) == P * H * D && pool.stride(2) == H * D && pool.stride(3) == D &&
       pool.stride(4) == 1 && pool.stride(0) >= 2 * P * H * D);
  return pool.stride(0) * pool.element_size();
}

// lengths as row_kernels._lengths_arg would pass them on unchanged
struct Lengths {
  const int64_t* per_item = nullptr;
  int64_t all = 0;
};
Lengths lengths_of(PyObject* o, int64_t batch, const Tensor& other) {
  Lengths l;
  if (PyLong_CheckExact(o)) {
    l.all = integer(o);
  } else {
    const Tensor& t = tensor(o);
    on_gpu(t, 1, other);
    need(t.scalar_type() == at::kLong && t.size(0) == batch && t.is_contiguous());
    l.per_item = static_cast<const int64_t*>(t.data_ptr());
  }
  return l;
}

PyObject* failed(const char* what, int status) {
  return PyErr_Format(PyExc_RuntimeError, "%s failed with status %d: %s", what, status, nhs_last_error());
}

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// Runs `body`; Skip and anything torch raises on an odd tensor leave the call to the Python launcher.
template <typename F>
PyObject* native(Py_ssize_t nargs, Py_ssize_t wanted, F body) {
  if (nargs != wanted) {
    PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
    return nullptr;
  }
  try {
    return body();
  } catch (const Skip&) {
  } catch (const std::exception&) {
  }
  Py_RETURN_NONE;
}

// ---- decode linear layers -----------------------------------------------------------------

void check_linear(const Tensor& x, const Tensor& w) {
  on_gpu(x, 2);
  on_gpu(w, 2, x);
  need(is_half(x) && w.scalar_type() == x.scalar_type() && x.size(1) == w.size(1) && x.stride(1) == 1 &&
       w.stride(1) == 1);
}

const void* bias_of(PyObject* o, const Tensor& x, int64_t n) {
  if (o == Py_None) return nullptr;
  const Tensor& b = tensor(o);
  on_gpu(b, 1, x);
  need(b.size(0) == n && b.scalar_type() == x.scalar_type() && b.is_contiguous());
  return b.data_ptr();
}

PyObject* linear_small_m(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 4, [&]() -> PyObject* {
    const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
    check_linear(x, w);
    const int64_t m = x.size(0), k = x.size(1), n = w.size(0);
    const void* bias = bias_of(a[2], x, n);
    Tensor out;
    if (a[3] != Py_None) {
      out = tensor(a[3]);
      on_gpu(out, 2, x);
      need(out.size(0) == m && out.size(1) == n && out.scalar_type() == x.scalar_type() && out.stride(1) == 1);
    }
    int st;
    {
      NoGil free;
      if (!out.defined()) out = make({m, n}, x, x.scalar_type());
      st = nhs_linear_small_m(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), bias, dtype_code(x), (int32_t)m,
                              (int32_t)n, (int32_t)k, out.data_ptr(), out.stride(0), stream_of(x));
    }
    return st ? failed("nhs_linear_small_m", st) : THPVariable_Wrap(out);
  });
}

PyObject* linear_silu_mul(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 2, [&]() -> PyObject* {
    const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
    check_linear(x, w);
    need(w.size(0) % 2 == 0);
    const int64_t m = x.size(0), inter = w.size(0) / 2;
    Tensor out;
    int st;
    {
      NoGil free;
      out = make({m, inter}, x, x.scalar_type());
      st = nhs_linear_silu_mul(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), dtype_code(x), (int32_t)m,
                               (int32_t)inter, (int32_t)x.size(1), out.data_ptr(), out.stride(0), stream_of(x));
    }
    return st ? failed("nhs_linear_silu_mul", st) : THPVariable_Wrap(out);
  });
}

PyObject* linear_rope(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 7, [&]() -> PyObject* {
    const Tensor &x = tensor(a[0]), &w = tensor(a[1]), &cos = tensor(a[5]), &sin = tensor(a[6]);
    check_linear(x, w);
    const int64_t m = x.size(0), n = w.size(0);
    const void* bias = bias_of(a[2], x, n);
    const int32_t heads = integer32(a[3]), dim = integer32(a[4]);
    for (const Tensor* t : {&cos, &sin}) {
      on_gpu(*t, 2, x);
      need(t->size(0) == m && t->size(1) == dim / 2 && t->scalar_type() == x.scalar_type() && t->is_contiguous());
    }
    Tensor out;
    int st;
    {
      NoGil free;
      out = make({m, n}, x, x.scalar_type());
      st = nhs_linear_rope(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), bias, dtype_code(x), (int32_t)m,
                           (int32_t)n, (int32_t)x.size(1), dim, heads, cos.data_ptr(), sin.data_ptr(), out.data_ptr(),
                           out.stride(0), stream_of(x));
    }
    return st ? failed("nhs_linear_rope", st) : THPVariable_Wrap(out);
  });
}

PyObject* add_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 5, [&]() -> PyObject* {
    const Tensor &x = tensor(a[0]), &w = tensor(a[2]);
    on_gpu(x, 2);
    on_gpu(w, 1, x);
    need(x.is_contiguous() && w.size(0) == x.size(1) && w.scalar_type() == x.scalar_type() && w.is_contiguous());
    const void* delta = nullptr;
    if (a[1] != Py_None) {
      const Tensor& d = tensor(a[1]);
      on_gpu(d, 2, x);
      need(same_sizes(d, x.sizes()) && d.scalar_type() == x.scalar_type() && d.is_contiguous());
      delta = d.data_ptr();
    }
    need(PyFloat_CheckExact(a[3]));
    const float eps = (float)PyFloat_AS_DOUBLE(a[3]);
    const bool write_back = truth(a[4]);
    const int code = dtype_code(x);
    Tensor out;
    int st;
    {
      NoGil free;
      out = make(x.sizes(), x, x.scalar_type());
      st = nhs_add_rmsnorm((int32_t)x.size(0), (int32_t)x.size(1), code, x.data_ptr(), delta, write_back,
                           w.data_ptr(), eps, out.data_ptr(), stream_of(x));
    }
    return st ? failed("nhs_add_rmsnorm", st) : THPVariable_Wrap(out);
  });
}

// ---- attention ------------------------------------------------------------------------------

// workspace: a tensor, or the dict (device index, stream) -> tensor of row_kernels.attend_workspace
PyObject* attend_batched(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 6, [&]() -> PyObject* {
    const Tensor &q = tensor(a[0]), &pool = tensor(a[1]), &rows = tensor(a[2]);
    on_gpu(q, 3);
    on_gpu(pool, 5, q);
    need(rows.dim() == 2 || rows.dim() == 3);
    on_gpu(rows, rows.dim(), q);
    const int64_t B = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = pool.size(3), n = rows.size(-1);
    const int32_t P = integer32(a[3]);
    need(rows.scalar_type() == at::kLong && pool.size(4) == D && pool.size(2) == P && Hq % Hkv == 0 &&
         q.stride(2) == 1 && rows.size(0) == B && (rows.dim() == 2 || rows.size(1) == Hq) &&
         pool.size(0) * P < (int64_t(1) << 31));
    const int64_t stride = pool_block_stride(pool);
    const int q_code = dtype_code(q), kv_code = dtype_code(pool);
    void* const stream = stream_of(q);
    const int64_t bytes = nhs_attend_workspace_bytes((int32_t)B, (int32_t)Hq, (int32_t)D, (int32_t)n);
    PyObject* held = a[5];
    if (PyDict_CheckExact(held)) {
      PyObject* key = Py_BuildValue("(iK)", (int)q.device().index(), (unsigned long long)(uintptr_t)stream);
      if (!key) return nullptr;
      held = PyDict_GetItemWithError(a[5], key);  // borrowed; the tensor below shares ownership
      Py_DECREF(key);
      if (!held && PyErr_Occurred()) return nullptr;
      need(held != nullptr);
    }
    const Tensor ws = tensor(held);
    need(ws.device() == q.device() && (int64_t)ws.numel() * (int64_t)ws.element_size() >= bytes);
    Tensor out;
    if (a[4] != Py_None) {
      out = tensor(a[4]);
      on_gpu(out, 3, q);
      need(same_sizes(out, q.sizes()) && out.scalar_type() == q.scalar_type() && out.stride(2) == 1);
    }
    int st;
    {
      NoGil free;
      if (!out.defined()) out = make({B, Hq, D}, q, q.scalar_type());
      st = nhs_attend_rows(q.data_ptr(), q_code, q.stride(0), q.stride(1), pool.data_ptr(), kv_code, stride,
                           static_cast<const int64_t*>(rows.data_ptr()), rows.stride(0),
                           rows.dim() == 3 ? rows.stride(1) : 0, rows.stride(-1), (int32_t)B, (int32_t)n, (int32_t)Hq,
                           (int32_t)Hkv, (int32_t)D, P, out.data_ptr(), out.stride(0), out.stride(1), ws.data_ptr(),
                           (int64_t)ws.numel() * (int64_t)ws.element_size(), stream);
    }
    return st ? failed("nhs_attend_rows", st) : THPVariable_Wrap(out);
  });
}

PyObject* prefill_attention(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 4, [&]() -> PyObject* {
    const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    on_gpu(q, 3);
    on_gpu(k, 3, q);
    on_gpu(v, 3, q);
    need(is_half(q) && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() &&
         same_sizes(v, k.sizes()) && k.size(0) == q.size(0) && k.size(2) == q.size(2) && q.stride(2) == 1 &&
         k.stride(2) == 1 && v.stride(2) == 1);
    Tensor out;
    if (a[3] != Py_None) {
      out = tensor(a[3]);
      on_gpu(out, 3, q);
      need(same_sizes(out, q.sizes()) && out.scalar_type() == q.scalar_type() && out.stride(2) == 1);
    }
    int st;
    {
      NoGil free;
      if (!out.defined()) out = make(q.sizes(), q, q.scalar_type());
      st = nhs_prefill_attention(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1),
                                 v.data_ptr(), v.stride(0), v.stride(1), dtype_code(q), (int32_t)q.size(0),
                                 (int32_t)q.size(1), (int32_t)k.size(1), (int32_t)q.size(2), out.data_ptr(),
                                 out.stride(0), out.stride(1), stream_of(q));
    }
    return st ? failed("nhs_prefill_attention", st) : THPVariable_Wrap(out);
  });
}

// ---- selection --------------------------------------------------------------------------------

struct Selection {
  Tensor pages, positions;
  void allocate(int64_t B, int64_t top, int64_t P, const Tensor& like) {
    pages = make({B, top}, like, at::kInt);
    positions = make({B, top * P}, like, at::kInt);
  }
};

PyObject* tuple_of(std::initializer_list<Tensor> tensors) {
  PyObject* result = PyTuple_New((Py_ssize_t)tensors.size());
  if (!result) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor& t : tensors) {
    PyObject* item;
    if (t.defined()) {
      item = THPVariable_Wrap(t);
    } else {
      item = Py_None;
      Py_INCREF(item);
    }
    if (!item) {
      Py_DECREF(result);
      return nullptr;
    }
    PyTuple_SET_ITEM(result, i++, item);
  }
  return result;
}

PyObject* quest_batched(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 8, [&]() -> PyObject* {
    const Tensor &q = tensor(a[0]), &lo = tensor(a[1]), &hi = tensor(a[2]);
    on_gpu(q, 3);
    on_gpu(lo, 4, q);
    on_gpu(hi, 4, q);
    const int64_t B = q.size(0), Hq = q.size(1), D = q.size(2), n_pages = lo.size(1), Hkv = lo.size(2);
    need(same_sizes(hi, lo.sizes()) && lo.size(0) == B && lo.size(3) == D && hi.scalar_type() == lo.scalar_type() &&
         hi.strides() == lo.strides() && contiguous_from(lo, 1) && q.stride(2) == 1);
    const Lengths len = lengths_of(a[3], B, q);
    const int32_t P = integer32(a[4]), top = integer32(a[5]);
    const bool keep_sink = truth(a[6]), select = truth(a[7]);
    need(P >= 1 && top >= 1 && (int64_t)top * P <= INT32_MAX);
    const int q_code = dtype_code(q), b_code = dtype_code(lo);
    Tensor scores;
    Selection s;
    int st;
    {
      NoGil free;
      scores = make({B, n_pages}, q, at::kFloat);
      if (select) s.allocate(B, top, P, q);
      st = nhs_quest_select((int32_t)B, q.data_ptr(), q_code, q.stride(0), q.stride(1), lo.data_ptr(), hi.data_ptr(),
                            b_code, lo.stride(0), (int32_t)Hq, (int32_t)Hkv, (int32_t)D, len.per_item, len.all, P,
                            (int32_t)n_pages, top, keep_sink, static_cast<float*>(scores.data_ptr()),
                            select ? static_cast<int32_t*>(s.pages.data_ptr()) : nullptr,
                            select ? static_cast<int32_t*>(s.positions.data_ptr()) : nullptr, stream_of(q));
    }
    return st ? failed("nhs_quest_select", st) : tuple_of({s.pages, s.positions, scores});
  });
}

void check_table(const Tensor& t, at::ScalarType type, int64_t B, const Tensor& other) {
  on_gpu(t, 2, other);
  need(t.scalar_type() == type && t.size(0) == B && t.stride(1) == 1);
}

PyObject* select_resolve_batched(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return native(nargs, 12, [&]() -> PyObject* {
    const Tensor &scores = tensor(a[0]), &source = tensor(a[1]), &resident = tensor(a[2]), &hot = tensor(a[3]),
                 &tags = tensor(a[4]), &lru = tensor(a[5]);
    on_gpu(scores, 2);
    need(scores.scalar_type() == at::kFloat && scores.is_contiguous());
    const int64_t B = scores.size(0), max_pages = scores.size(1);
    check_table(source, at::kInt, B, scores);
    check_table(resident, at::kInt, B, scores);
    check_table(hot, at::kInt, B, scores);
    check_table(tags, at::kInt, B, scores);
    check_table(lru, at::kLong, B, scores);
    const Lengths len = lengths_of(a[6], B, scores);
    const int32_t P = integer32(a[7]), top = integer32(a[8]);
    const bool keep_sink = truth(a[9]);
    const int32_t mode = integer32(a[10]);
    need(P >= 1 && top >= 1 && (int64_t)top * P <= INT32_MAX);
    const int64_t H = tags.size(1), K = (int64_t)top * P;
    need(same_sizes(resident, source.sizes()) && resident.stride(0) == source.stride(0) && lru.size(1) == H &&
         hot.size(1) * P >= H);
    int64_t* total = nullptr;
    if (a[11] != Py_None) {
      const Tensor& t = tensor(a[11]);
      on_gpu(t, 1, scores);
      need(t.scalar_type() == at::kLong && t.size(0) == 3 && t.is_contiguous());
      total = static_cast<int64_t*>(t.data_ptr());
    }
    Selection s;
    Tensor physical, miss_host, miss_device, counts;
    int st;
    {
      NoGil free;
      s.allocate(B, top, P, scores);
      physical = make({B, K}, scores, at::kLong);
      miss_host = make({B, K}, scores, at::kLong);
      miss_device = make({B, K}, scores, at::kLong);
      counts = make({B, 3}, scores, at::kLong);
      st = nhs_select_resolve_rows(
          (int32_t)B, static_cast<const float*>(scores.data_ptr()), (int32_t)max_pages, mode, top, keep_sink,
          static_cast<const int32_t*>(source.data_ptr()), static_cast<const int32_t*>(resident.data_ptr()),
          source.stride(0), (int32_t)source.size(1), static_cast<const int32_t*>(hot.data_ptr()), hot.stride(0),
          static_cast<int32_t*>(tags.data_ptr()), tags.stride(0), static_cast<int64_t*>(lru.data_ptr()), lru.stride(0),
          (int32_t)H, len.per_item, len.all, P, static_cast<int32_t*>(s.pages.data_ptr()),
          static_cast<int32_t*>(s.positions.data_ptr()), static_cast<int64_t*>(physical.data_ptr()),
          static_cast<int64_t*>(miss_host.data_ptr()), static_cast<int64_t*>(miss_device.data_ptr()), K,
          static_cast<int64_t*>(counts.data_ptr()), total, stream_of(scores));
    }
    return st ? failed("nhs_select_resolve_rows", st)
              : tuple_of({s.pages, s.positions, physical, miss_host, miss_device, counts});
  });
}

// ---- append ------------------------------------------------------------------------------------

// nhs_append_page with the arguments row_kernels.PageAppender prepared (checked there), as whole numbers of any integer
// type; returns the status.
PyObject* append_page(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 17) {
    PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
    return nullptr;
  }
  int64_t v[17];
  for (int i = 0; i < 17; ++i) {  // negative numbers go to the library, which refuses them
    PyObject* whole = PyNumber_Index(a[i]);
    if (!whole) return nullptr;
    v[i] = (int64_t)PyLong_AsUnsignedLongLongMask(whole);
    Py_DECREF(whole);
    if (PyErr_Occurred()) return nullptr;
  }
  const auto at = [&](int i) { return reinterpret_cast<void*>((uintptr_t)v[i]); };
  int st;
  {
    NoGil free;
    st = nhs_append_page(at(0), at(1), v[2], (int32_t)v[3], (int32_t)v[4], (int32_t)v[5], at(6), v[7], v[8],
                         (int32_t)v[9], (int32_t)v[10], at(11), v[12], static_cast<float*>(at(13)), at(14), at(15),
                         at(16));
  }
  return PyLong_FromLong(st);
}

// ---- parameters --------------------------------------------------------------------------------

// Of a tensor its address, dtype, sizes and strides; of any other object, and of a tensor without them, its identity.
void add_state(std::vector<int64_t>& state, PyObject* value) {
  const size_t before = state.size();
  if (PyObject_TypeCheck(value, reinterpret_cast<PyTypeObject*>(THPVariableClass))) {
    try {
      const Tensor& t = THPVariable_Unpack(value);
      state.push_back((int64_t)(uintptr_t)t.const_data_ptr());
      state.push_back((int64_t)t.scalar_type() << 32 | t.dim());
      for (int64_t s : t.sizes()) state.push_back(s);
      for (int64_t s : t.strides()) state.push_back(s);
      return;
    } catch (const std::bad_alloc&) {
      throw;
    } catch (const std::exception&) {  // a sparse or wrapped tensor
      PyErr_Clear();
      state.resize(before);
    }
  }
  state.push_back((int64_t)(uintptr_t)value);
}

// The bytes that tell whether the dicts (of modules' parameters and child
// modules) hold what they held: each dict's size and its values' states. For
// checks made on every step.
PyObject* held_state(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 1 || !PyList_CheckExact(a[0])) {
    PyErr_SetString(PyExc_TypeError, "held_state takes a list of dicts");
    return nullptr;
  }
  try {
    std::vector<int64_t> state;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); ++i) {
      PyObject* dict = PyList_GET_ITEM(a[0], i);
      if (!PyDict_Check(dict)) {
        PyErr_SetString(PyExc_TypeError, "held_state takes a list of dicts");
        return nullptr;
      }
      state.push_back(PyDict_Size(dict));
      PyObject *key, *value;
      Py_ssize_t at = 0;
      while (PyDict_Next(dict, &at, &key, &value)) add_state(state, value);
    }
    return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(state.data()),
                                     (Py_ssize_t)(state.size() * sizeof(int64_t)));
  } catch (const std::bad_alloc&) {
    return PyErr_NoMemory();
  }
}

#define NHS_METHOD(name) \
  { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr }
PyMethodDef methods[] = {NHS_METHOD(linear_small_m), NHS_METHOD(linear_silu_mul),   NHS_METHOD(linear_rope),
                         NHS_METHOD(add_rmsnorm),    NHS_METHOD(attend_batched),    NHS_METHOD(prefill_attention),
                         NHS_METHOD(quest_batched),  NHS_METHOD(select_resolve_batched),
                         NHS_METHOD(append_page),    NHS_METHOD(held_state),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch() { return PyModule_Create(&module); }
