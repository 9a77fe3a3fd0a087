// The common form of the Python entry points in native code: argument checks, output and workspace
// allocation and the library call, for calls whose operands are used as they are (plain CUDA tensors,
// no copy to make, no option beyond those listed at each function). Anything else -- a wrong type,
// shape, dtype, device, stride or alignment, a tensor subclass other than a parameter, an empty batch --
// returns None, and the Python function goes on with its own checks, which copy or raise.
//
// Why: a call of this package is a few microseconds of GPU time at small sizes, and the Python
// wrappers took 10 to 17 us of checks and argument conversion each, so that small calls were bound by
// the host. Time per call, and a decode layer (two calls) of one sequence of 512 tokens: layer
// 32.5 -> 15.6 us, decode of two sequences of 60 tokens 12.6 -> 6.6 (with the append fused
// 16.9 -> 6.7), append of 32 tokens 9.8 -> 4.3, QK-norm + RoPE + append of 32 tokens 15.0 -> 5.3.
//
// The functions take the library's entry points by address (bind), so the module links to nothing but
// torch. Each returns None (not this form), a nonzero int (the library's return code; the caller turns
// it into an exception) or its result.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>

#include "../../include/tileinfer_amd.h"

namespace {

decltype(&ti_kv_append) p_append = nullptr;
decltype(&ti_gqa_decode_plan) p_plan = nullptr;
decltype(&ti_gqa_decode_paged) p_decode = nullptr;
decltype(&ti_gqa_decode_paged_gated) p_decode_gated = nullptr;
decltype(&ti_gqa_decode_paged_append) p_decode_append = nullptr;
decltype(&ti_gqa_prefill_paged) p_prefill = nullptr;
decltype(&ti_gqa_prefill_paged_gated) p_prefill_gated = nullptr;
decltype(&ti_gqa_prefill_workspace_bytes) p_prefill_ws = nullptr;
decltype(&ti_qknorm_rope_append) p_qknorm_append = nullptr;

// A plain tensor with memory of its own on a GPU, or nullptr.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided || t.is_neg()) {
    return nullptr;
  }
  return &t;
}

uintptr_t address(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()); }

int dtype_code(const at::Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return TI_DTYPE_BF16;
  if (t.scalar_type() == at::kHalf) return TI_DTYPE_F16;
  return -1;
}

// Unit element stride, the other strides and the address multiples of `elems` 16-bit elements.
bool aligned_rows(const at::Tensor& t, int64_t elems) {
  const auto st = t.strides();
  const size_t n = st.size();
  if (n == 0 || st[n - 1] != 1 || address(t) % (2 * elems) != 0) return false;
  for (size_t i = 0; i + 1 < n; ++i) {
    if (st[i] % elems != 0) return false;
  }
  return true;
}

bool int32_vector(const at::Tensor& t, int64_t n, const at::Device& dev) {
  return t.scalar_type() == at::kInt && t.dim() == 1 && t.size(0) == n && t.is_contiguous() &&
         t.device() == dev;
}

bool fits32(int64_t x) { return x >= 0 && x <= INT32_MAX; }

// The operands that decode and prefill share: queries [rows, H_q, D] and one layer's cache pages.
struct Paged {
  const at::Tensor *q, *k, *v, *table;
  int64_t rows_q, hq, hkv, d, rows, page, width, batch;
  int dtype;
};

bool paged(PyObject* const* a, PyObject* page, Paged& o) {
  o.q = plain(a[0]);
  o.k = plain(a[1]);
  o.v = plain(a[2]);
  o.table = plain(a[3]);
  if (!o.q || !o.k || !o.v || !o.table || !PyLong_CheckExact(page)) return false;
  o.page = PyLong_AsLongLong(page);
  if (o.page == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  const at::Tensor &q = *o.q, &k = *o.k, &v = *o.v, &t = *o.table;
  if (q.dim() != 3 || k.dim() != 4 || t.dim() != 2 || k.sizes() != v.sizes()) return false;
  o.rows_q = q.size(0);
  o.hq = q.size(1);
  o.d = q.size(2);
  o.hkv = k.size(2);
  o.rows = k.size(0) * k.size(1);
  o.batch = t.size(0);
  o.width = t.size(1);
  o.dtype = dtype_code(q);
  const at::Device dev = q.device();
  return o.rows_q > 0 && o.batch > 0 && o.width > 0 && o.hkv > 0 && o.hq % o.hkv == 0 &&
         k.size(3) == o.d && o.dtype >= 0 && k.scalar_type() == q.scalar_type() &&
         v.scalar_type() == q.scalar_type() && k.is_contiguous() && v.is_contiguous() &&
         t.scalar_type() == at::kInt && t.stride(1) == 1 && k.device() == dev && v.device() == dev &&
         t.device() == dev && o.page > 0 && o.rows % o.page == 0 && aligned_rows(q, 8) &&
         fits32(o.rows_q) && fits32(o.hq) && fits32(o.d) && fits32(o.page) && fits32(o.width) &&
         fits32(o.batch);
}

// The output gate as contiguous [rows, H_q, D] rows; false where it needs a copy or is wrong.
bool gate_rows(PyObject* o, const Paged& p, const at::Tensor** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* g = plain(o);
  if (!g || g->numel() != p.rows_q * p.hq * p.d || g->scalar_type() != p.q->scalar_type() ||
      g->device() != p.q->device() || !g->is_contiguous() || address(*g) % 16 != 0) {
    return false;
  }
  *out = g;
  return true;
}

at::Tensor bytes_on(const at::Tensor& like, int64_t n) {
  return at::empty({n}, like.options().dtype(at::kByte));
}

void* stream_of(PyObject* o) { return PyLong_AsVoidPtr(o); }

// Lets other Python threads run while the library call and the allocations before it do (an
// allocation may wait for the GPU, a launch for room in its queue). Restored on every way out.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;

 private:
  PyThreadState* state_;
};

PyObject* guarded(PyObject* (*f)(PyObject* const*), PyObject* const* a, Py_ssize_t n, Py_ssize_t want) {
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return nullptr;
  }
  try {
    return f(a);
  } catch (...) {  // as torch's own functions raise it (out of memory among them)
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

// (q, k_cache, v_cache, block_table, seqlen, page_size, gate | None, key | None, value, slots, stream)
PyObject* decode(PyObject* const* a) {
  Paged p;
  const at::Tensor *gate, *seqlen = plain(a[4]);
  if (!seqlen || !paged(a, a[5], p) || !gate_rows(a[6], p, &gate)) Py_RETURN_NONE;
  const at::Device dev = p.q->device();
  if (p.rows_q != p.batch || !int32_vector(*seqlen, p.batch, dev)) Py_RETURN_NONE;
  const at::Tensor *key = nullptr, *value = nullptr, *slots = nullptr;
  const int64_t row = p.hkv * p.d;
  if (a[7] != Py_None) {
    key = plain(a[7]);
    value = plain(a[8]);
    slots = plain(a[9]);
    if (!key || !value || !slots || gate || !int32_vector(*slots, p.batch, dev)) Py_RETURN_NONE;
    for (const at::Tensor* t : {key, value}) {
      if (t->dim() != 3 || t->size(0) != p.batch || t->size(1) != p.hkv || t->size(2) != p.d ||
          t->scalar_type() != p.q->scalar_type() || t->device() != dev || t->stride(2) != 1 ||
          t->stride(1) != p.d || t->stride(0) < row || !aligned_rows(*t, 8)) {
        Py_RETURN_NONE;
      }
    }
  }
  void* stream = stream_of(a[10]);
  at::Tensor out;
  int rc;
  {
    Unlocked unlocked;
    int32_t split = 0, splits = 0;
    int64_t ws_bytes = 0;
    rc = p_plan(int32_t(p.batch), int32_t(p.hq), int32_t(p.hkv), int32_t(p.d), int32_t(p.page),
                int32_t(p.width), 0, &split, &splits, &ws_bytes);
    if (rc == TI_OK) {
      out = at::empty({p.batch, p.hq, p.d}, p.q->options());
      at::Tensor ws;
      if (ws_bytes > 0) ws = bytes_on(*p.q, ws_bytes);
      void* wp = ws_bytes > 0 ? ws.data_ptr() : nullptr;
      const int32_t* table = static_cast<const int32_t*>(p.table->data_ptr());
      const int32_t* lens = static_cast<const int32_t*>(seqlen->data_ptr());
#define TI_DECODE_ARGS                                                                            \
  p.q->data_ptr(), p.q->stride(0), p.q->stride(1), p.k->data_ptr(), p.v->data_ptr(), table,       \
      p.table->stride(0), lens, out.data_ptr(), wp, ws_bytes, int32_t(p.batch), int32_t(p.hq),    \
      int32_t(p.hkv), int32_t(p.d), int32_t(p.page), p.rows / p.page, int32_t(p.width), 0,        \
      TI_DECODE_AUTO, p.dtype
      if (key) {
        rc = p_decode_append(TI_DECODE_ARGS, key->data_ptr(), value->data_ptr(), key->stride(0),
                             value->stride(0), static_cast<const int32_t*>(slots->data_ptr()),
                             p.rows, stream);
      } else if (gate) {
        rc = p_decode_gated(TI_DECODE_ARGS, gate->data_ptr(), p.hq * p.d, p.d, stream);
      } else {
        rc = p_decode(TI_DECODE_ARGS, stream);
      }
#undef TI_DECODE_ARGS
    }
  }
  if (rc != TI_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
}

// (q, k_cache, v_cache, block_table, cu_seqlens_q, seqlen_k, max_seqlen_q, page_size, causal,
//  per_unit, gate | None, stream)
PyObject* prefill(PyObject* const* a) {
  Paged p;
  const at::Tensor *gate, *cu = plain(a[4]), *lens = plain(a[5]);
  if (!cu || !lens || !PyLong_CheckExact(a[6]) || !paged(a, a[7], p) || !gate_rows(a[10], p, &gate)) {
    Py_RETURN_NONE;
  }
  const at::Device dev = p.q->device();
  const int64_t max_q = PyLong_AsLongLong(a[6]);
  if (max_q == -1 && PyErr_Occurred()) PyErr_Clear();
  if (!fits32(max_q) || !int32_vector(*cu, p.batch + 1, dev) || !int32_vector(*lens, p.batch, dev)) {
    Py_RETURN_NONE;
  }
  const bool causal = a[8] == Py_True, per_unit = a[9] == Py_True;
  void* stream = stream_of(a[11]);
  at::Tensor out;
  int rc = TI_OK;
  {
    Unlocked unlocked;
    int64_t ws_bytes = 0;
    if (!per_unit) {
      rc = p_prefill_ws(int32_t(p.batch), int32_t(p.rows_q), int32_t(p.hq), int32_t(p.hkv),
                        int32_t(p.d), int32_t(p.page), int32_t(p.width), &ws_bytes);
    }
    if (rc == TI_OK) {
      out = at::empty({p.rows_q, p.hq, p.d}, p.q->options());
      at::Tensor ws;
      if (ws_bytes > 0) ws = bytes_on(*p.q, ws_bytes);
      void* wp = ws_bytes > 0 ? ws.data_ptr() : nullptr;
#define TI_PREFILL_ARGS                                                                           \
  p.q->data_ptr(), p.q->stride(0), p.q->stride(1), p.k->data_ptr(), p.v->data_ptr(),              \
      static_cast<const int32_t*>(p.table->data_ptr()), p.table->stride(0),                       \
      static_cast<const int32_t*>(cu->data_ptr()), static_cast<const int32_t*>(lens->data_ptr()), \
      out.data_ptr(), out.stride(0), out.stride(1), wp, ws_bytes, int32_t(p.batch),               \
      int32_t(p.rows_q), int32_t(max_q), int32_t(p.hq), int32_t(p.hkv), int32_t(p.d),             \
      int32_t(p.page), p.rows / p.page, int32_t(p.width), causal ? 1 : 0, p.dtype
      rc = gate ? p_prefill_gated(TI_PREFILL_ARGS, gate->data_ptr(), p.hq * p.d, p.d, stream)
                : p_prefill(TI_PREFILL_ARGS, stream);
#undef TI_PREFILL_ARGS
    }
  }
  if (rc != TI_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
}

// One layer's cache as token rows [num_slots, row], the same strides for K and V.
bool cache_rows(const at::Tensor* k, const at::Tensor* v, int64_t row, const at::Tensor& like) {
  return k->dim() == 2 && k->size(1) == row && k->stride(1) == 1 && k->sizes() == v->sizes() &&
         k->strides() == v->strides() && k->scalar_type() == like.scalar_type() &&
         v->scalar_type() == like.scalar_type() && k->device() == like.device() &&
         v->device() == like.device();
}

// (key, value, k_cache, v_cache, slot_mapping, stream) -> True
PyObject* append(PyObject* const* a) {
  const at::Tensor *key = plain(a[0]), *value = plain(a[1]), *k = plain(a[2]), *v = plain(a[3]),
                   *slots = plain(a[4]);
  if (!key || !value || !k || !v || !slots || key->dim() != 3 || key->sizes() != value->sizes()) {
    Py_RETURN_NONE;
  }
  const int64_t n = key->size(0), h = key->size(1), d = key->size(2);
  const int code = dtype_code(*key);
  if (n <= 0 || h <= 0 || d <= 0 || code < 0 || value->scalar_type() != key->scalar_type() ||
      value->device() != key->device() || !cache_rows(k, v, h * d, *key) ||
      !int32_vector(*slots, n, key->device())) {
    Py_RETURN_NONE;
  }
  for (const at::Tensor* t : {key, value}) {
    if (t->stride(2) != 1 || t->stride(1) != d || t->stride(0) < h * d) Py_RETURN_NONE;
  }
  void* stream = stream_of(a[5]);
  int rc;
  {
    Unlocked unlocked;
    rc = p_append(key->data_ptr(), value->data_ptr(), key->stride(0), value->stride(0),
                  k->data_ptr(), v->data_ptr(), k->stride(0),
                  static_cast<const int32_t*>(slots->data_ptr()), n, h * d, k->size(0), code, stream);
  }
  if (rc != TI_OK) return PyLong_FromLong(rc);
  Py_RETURN_TRUE;
}

// (q, k, v, q_weight, k_weight, cos, sin, k_cache, v_cache, slot_mapping, eps, stream)
PyObject* qknorm_append(PyObject* const* a) {
  const at::Tensor* t[10];
  for (int i = 0; i < 10; ++i) {
    t[i] = plain(a[i]);
    if (!t[i]) Py_RETURN_NONE;
  }
  const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &qw = *t[3], &kw = *t[4], &cos = *t[5],
                   &sin = *t[6], &slots = *t[9];
  if (!PyFloat_CheckExact(a[10]) || q.dim() != 3 || k.dim() != 3 || v.sizes() != k.sizes()) {
    Py_RETURN_NONE;
  }
  const int64_t n = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(1);
  const int code = dtype_code(q);
  if (code < 0 || n <= 0 || hq <= 0 || hkv <= 0 || k.size(0) != n || k.size(2) != d ||
      cos.dim() != 2 || cos.size(0) != n || cos.sizes() != sin.sizes() ||
      cos.strides() != sin.strides() || cos.stride(1) != 1) {
    Py_RETURN_NONE;
  }
  const int64_t rd = cos.size(1);
  for (int i = 0; i < 7; ++i) {
    if (t[i]->scalar_type() != q.scalar_type() || t[i]->device() != q.device()) Py_RETURN_NONE;
  }
  for (const at::Tensor* x : {&q, &k, &v}) {
    if (!aligned_rows(*x, 2)) Py_RETURN_NONE;
  }
  for (const at::Tensor* x : {&qw, &kw}) {
    if (x->dim() != 1 || x->size(0) != d || x->stride(0) != 1) Py_RETURN_NONE;
  }
  if (rd > d || rd % 2 || rd == 0 || !fits32(n) || !fits32(hq) || !fits32(hkv) || !fits32(d) ||
      !cache_rows(t[7], t[8], hkv * d, q) || !int32_vector(slots, n, q.device())) {
    Py_RETURN_NONE;
  }
  const float eps = float(PyFloat_AS_DOUBLE(a[10]));
  void* stream = stream_of(a[11]);
  at::Tensor out;
  int rc;
  {
    Unlocked unlocked;
    out = at::empty({n, hq, d}, q.options());
    rc = p_qknorm_append(
        q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(),
        v.stride(0), v.stride(1), qw.data_ptr(), kw.data_ptr(), cos.data_ptr(), sin.data_ptr(),
        n == 1 ? 0 : cos.stride(0), out.data_ptr(), out.stride(0), out.stride(1), t[7]->data_ptr(),
        t[8]->data_ptr(), t[7]->stride(0), static_cast<const int32_t*>(slots.data_ptr()),
        t[7]->size(0), int32_t(n), int32_t(hq), int32_t(hkv), int32_t(d), int32_t(rd), eps, code,
        stream);
  }
  if (rc != TI_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
}

// The library's entry points by address, in the order of the list below.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  void** slots[] = {(void**)&p_append,        (void**)&p_plan,          (void**)&p_decode,
                    (void**)&p_decode_gated,  (void**)&p_decode_append, (void**)&p_prefill,
                    (void**)&p_prefill_gated, (void**)&p_prefill_ws,    (void**)&p_qknorm_append};
  if (n != Py_ssize_t(sizeof(slots) / sizeof(slots[0]))) {
    PyErr_SetString(PyExc_TypeError, "bind: nine addresses");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    void* f = PyLong_AsVoidPtr(a[i]);
    if (!f) return nullptr;
    *slots[i] = f;
  }
  Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject* const*), Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(F, a, n, N);
}

#define TI_METHOD(name, n) \
  {#name, (PyCFunction)(void (*)(void))entry<name, n>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
                         TI_METHOD(decode, 11),
                         TI_METHOD(prefill, 12),
                         TI_METHOD(append, 6),
                         TI_METHOD(qknorm_append, 12),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycalls", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for (given by the build): the versions whose structures this file was compiled against.
PyMODINIT_FUNC PyInit__pycalls(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", TI_BUILT_FOR) < 0) Py_CLEAR(m);
  return m;
}
