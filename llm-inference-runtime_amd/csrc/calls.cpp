// The Python hot path's checks and argument marshalling in C++: one extension
// function per launch that an engine makes in every layer (the FlashInfer
// calls of src/models/llama.py:188-245).  Each takes the tensors as Python
// holds them, checks that they have the plain form the kernels take, allocates
// the outputs and calls libpagedattn's C entry point on the current stream.
//
// A step of a small batch is bound by this path: 25-30 arguments converted one
// by one through ctypes, with the shape checks and strides read in Python, took
// 12-15 us a call where the attention kernels take 5-10 us on the GPU.
//
// Returns the call's result, or NotImplemented for anything but the plain form
// (another type or device, a tensor subclass, metadata that needs a conversion,
// empty rows, and every bad argument): the caller then takes the general path in
// Python, which converts or raises.  A non-zero status of the C entry point is
// returned as an int for the caller to raise.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/Allocator.h>
#include <c10/core/DeviceGuard.h>
#include <c10/util/Exception.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "pagedattn.h"

namespace {

// C entry points, bound by address so that this module shares the library
// instance (and HIP runtime) the package has loaded.
struct Entries {
  decltype(&pagedattn_plan_scratch_bytes) scratch_bytes;
  decltype(&pagedattn_decode_run_scratch) decode_run;
  decltype(&pagedattn_prefill_run_scratch) prefill_run;
  decltype(&pagedattn_append_paged_kv_cache) append;
  decltype(&pagedattn_rope_append_paged_kv_cache) rope_append;
  decltype(&pagedattn_append_paged_kv_cache_e4m3_amax) append_amax;
};
Entries g_entry;
PyObject* g_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

constexpr int kPageSize = 16;

const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.layout() == at::kStrided ? &t : nullptr;
}

// A 16-bit element type's code, or -1.
int code16(const at::Tensor& t) {
  const auto s = t.scalar_type();
  return s == at::kBFloat16 ? PAGEDATTN_BF16 : s == at::kHalf ? PAGEDATTN_F16 : -1;
}

// One layer's pool: contiguous [P, 2, Hkv, 16, D] on the device, 16-bit or e4m3.
struct Pool {
  const at::Tensor* t = nullptr;
  int code = -1;
  int64_t pages = 0, hkv = 0, d = 0;
  at::Device device = at::kCPU;
  bool get(PyObject* o) {
    t = plain(o);
    if (!t || !t->is_cuda() || t->dim() != 5 || t->size(1) != 2 || t->size(3) != kPageSize ||
        !t->is_contiguous())
      return false;
    code = t->scalar_type() == at::kFloat8_e4m3fn ? PAGEDATTN_E4M3 : code16(*t);
    pages = t->size(0);
    hkv = t->size(2);
    d = t->size(4);
    device = t->device();
    return code >= 0;
  }
  void* ptr() const { return t->data_ptr(); }
};

// Page scales: taken for e4m3 pools only, as the general path does.
bool get_scales(PyObject* o, const Pool& pool, float** out) {
  *out = nullptr;
  if (pool.code != PAGEDATTN_E4M3) return true;
  const at::Tensor* t = plain(o);
  if (!t || !t->is_cuda() || t->scalar_type() != at::kFloat || t->dim() != 3 ||
      t->size(0) != pool.pages || t->size(1) != 2 || t->size(2) != pool.hkv ||
      !t->is_contiguous())
    return false;
  *out = static_cast<float*>(t->data_ptr());
  return true;
}

// [n, heads, d] rows, d contiguous, at least one row.
const at::Tensor* rows(PyObject* o, int64_t heads, int64_t d) {
  const at::Tensor* t = plain(o);
  if (!t || !t->is_cuda() || t->dim() != 3 || t->size(0) < 1 || t->size(2) != d ||
      (heads >= 0 && t->size(1) != heads) || t->stride(2) != 1 || code16(*t) < 0)
    return nullptr;
  return t;
}

// int32 metadata usable in place on `device`; count < 0: any length.
bool meta(PyObject* o, const at::Device& device, int64_t count, const int32_t** out,
          int64_t* numel = nullptr) {
  const at::Tensor* t = plain(o);
  if (!t || t->device() != device || t->scalar_type() != at::kInt || !t->is_contiguous() ||
      (count >= 0 && t->numel() != count))
    return false;
  *out = static_cast<const int32_t*>(t->data_ptr());
  if (numel) *numel = t->numel();
  return true;
}

// Optional int32 counters of at least n entries.
bool get_flag(PyObject* o, int64_t n, int32_t** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = plain(o);
  if (!t || !t->is_cuda() || t->scalar_type() != at::kInt || t->numel() < n ||
      !t->is_contiguous())
    return false;
  *out = static_cast<int32_t*>(t->data_ptr());
  return true;
}

bool raw_stream(const at::Device& device, void** out) {
  PyObject* idx = PyLong_FromLong(device.index());
  if (!idx) return false;
  PyObject* r = PyObject_CallOneArg(g_raw_stream, idx);
  Py_DECREF(idx);
  if (!r) return false;
  *out = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  return !(*out == nullptr && PyErr_Occurred());
}

// Output [n, heads, d] in q's type (or the caller's), and the optional LSE.
struct Outputs {
  at::Tensor out, lse;
  PyObject* out_o = nullptr;  // borrowed: the caller's tensors
  PyObject* lse_o = nullptr;
  void* lse_ptr = nullptr;
  bool want_lse = false;
  bool get(PyObject* o, PyObject* l, int return_lse, const at::Tensor& q, int64_t n,
           int64_t hq, int64_t d) {
    want_lse = return_lse != 0;
    if (o == Py_None) {
      out = at::empty({n, hq, d}, q.options().requires_grad(false));
    } else {
      const at::Tensor* t = plain(o);
      if (!t || t->device() != q.device() || t->scalar_type() != q.scalar_type() ||
          !t->is_contiguous() || t->dim() != 3 || t->size(0) != n || t->size(1) != hq ||
          t->size(2) != d)
        return false;
      out = *t;
      out_o = o;
    }
    if (l != Py_None) {
      const at::Tensor* t = plain(l);
      if (!t || t->device() != q.device() || t->scalar_type() != at::kFloat ||
          !t->is_contiguous() || t->numel() < n * hq)
        return false;
      lse = *t;
      lse_o = l;
      lse_ptr = lse.data_ptr();
    } else if (want_lse) {
      lse = at::empty({n, hq}, q.options().dtype(at::kFloat).requires_grad(false));
      lse_ptr = lse.data_ptr();
    }
    return true;
  }
  static PyObject* wrap(const at::Tensor& t, PyObject* o) {
    if (o) {
      Py_INCREF(o);
      return o;
    }
    return THPVariable_Wrap(t);
  }
  PyObject* result() const {
    PyObject* a = wrap(out, out_o);
    if (!a || !want_lse) return a;
    PyObject* b = wrap(lse, lse_o);
    if (!b) {
      Py_DECREF(a);
      return nullptr;
    }
    PyObject* r = PyTuple_Pack(2, a, b);
    Py_DECREF(a);
    Py_DECREF(b);
    return r;
  }
};

// The scratch of one run of a plan that cuts KV ranges: torch's caching
// allocator hands it out per run and stream (and per captured graph), so runs of
// one plan may overlap; freed when the call returns, it is reused in stream
// order.  Without memory for it the run takes the plan's whole form.
struct Scratch {
  c10::DataPtr mem;
  void* ptr = nullptr;
  size_t bytes = 0;
  void get(const pagedattn_plan* plan, const at::Tensor& q) {
    bytes = g_entry.scratch_bytes(plan, q.size(0));
    if (!bytes) return;
    try {
      const c10::DeviceGuard guard(q.device());
      mem = c10::GetAllocator(c10::DeviceType::CUDA)->allocate(bytes);
      ptr = mem.get();
    } catch (const c10::OutOfMemoryError&) {
      bytes = 0;
    }
  }
};

PyObject* general() { Py_RETURN_NOTIMPLEMENTED; }

bool arg_count(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
  return false;
}

// decode_run(plan, q, pool, indices, indptr, last, batch, hq, hkv, d, scales,
//            out, lse, return_lse, sm_scale, key, value, rope, positions)
PyObject* decode_run(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arg_count(n, 19)) return nullptr;
  auto* plan = static_cast<pagedattn_plan*>(PyLong_AsVoidPtr(a[0]));
  const int64_t bsz = PyLong_AsLongLong(a[6]), hq = PyLong_AsLongLong(a[7]),
                hkv = PyLong_AsLongLong(a[8]), d = PyLong_AsLongLong(a[9]);
  const int return_lse = PyObject_IsTrue(a[13]);
  const double scale = PyFloat_AsDouble(a[14]);
  if (PyErr_Occurred()) return nullptr;
  Pool pool;
  if (!pool.get(a[2]) || pool.hkv != hkv || pool.d != d) return general();
  const at::Tensor* q = rows(a[1], hq, d);
  float* scales;
  if (!q || q->size(0) != bsz || !get_scales(a[10], pool, &scales)) return general();
  const int32_t *indices, *indptr, *last, *pos = nullptr;
  int64_t n_ind = 0;
  if (!meta(a[3], q->device(), -1, &indices, &n_ind) ||
      !meta(a[4], q->device(), bsz + 1, &indptr) || !meta(a[5], q->device(), bsz, &last))
    return general();
  const bool append = a[15] != Py_None;
  const bool rope = a[17] != Py_None;
  const at::Tensor *k = nullptr, *v = nullptr;
  double rope_scale = 1.0, rope_theta = 1.0;
  if (append) {
    k = rows(a[15], hkv, d);
    v = rows(a[16], hkv, d);
    if (!k || !v || k->size(0) != bsz || v->size(0) != bsz ||
        k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type())
      return general();
    if (rope) {
      if (!PyTuple_CheckExact(a[17]) || PyTuple_GET_SIZE(a[17]) != 2) return general();
      rope_scale = PyFloat_AsDouble(PyTuple_GET_ITEM(a[17], 0));
      rope_theta = PyFloat_AsDouble(PyTuple_GET_ITEM(a[17], 1));
      if (PyErr_Occurred()) return nullptr;
      if (a[18] != Py_None && !meta(a[18], q->device(), bsz, &pos)) return general();
    } else if (a[18] != Py_None) {
      return general();
    }
  } else if (a[16] != Py_None) {
    return general();
  }
  Outputs o;
  if (!o.get(a[11], a[12], return_lse, *q, bsz, hq, d)) return general();
  void* stream;
  if (!raw_stream(q->device(), &stream)) return nullptr;
  const void* qp = q->data_ptr();
  const void* kp = append ? k->data_ptr() : nullptr;
  const void* vp = append ? v->data_ptr() : nullptr;
  void* pp = pool.ptr();
  void* op = o.out.data_ptr();
  float* lp = static_cast<float*>(o.lse_ptr);
  const int code = code16(*q);
  const int64_t ks[2] = {append ? k->stride(0) : 0, append ? k->stride(1) : 0};
  const int64_t vs[2] = {append ? v->stride(0) : 0, append ? v->stride(1) : 0};
  Scratch scratch;
  scratch.get(plan, *q);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_entry.decode_run(plan, qp, q->stride(0), q->stride(1), code, kp, vp, ks[0], ks[1], vs[0],
                          vs[1], rope, pos, (float)rope_scale, (float)rope_theta, pp, pool.code,
                          scales, (int32_t)pool.pages, indices, (int32_t)n_ind, indptr, last, op,
                          lp, (float)scale, scratch.ptr, scratch.bytes, stream);
  Py_END_ALLOW_THREADS
  return rc ? PyLong_FromLong(rc) : o.result();
  END_HANDLE_TH_ERRORS
}

// prefill_run(plan, q, pool, qo_indptr, indices, indptr, last, batch, qo_rows,
//             hq, hkv, d, scales, out, lse, return_lse, causal, sm_scale);
// qo_rows < 0: known on the device only
PyObject* prefill_run(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arg_count(n, 18)) return nullptr;
  auto* plan = static_cast<pagedattn_plan*>(PyLong_AsVoidPtr(a[0]));
  const int64_t bsz = PyLong_AsLongLong(a[7]), qo_rows = PyLong_AsLongLong(a[8]),
                hq = PyLong_AsLongLong(a[9]), hkv = PyLong_AsLongLong(a[10]),
                d = PyLong_AsLongLong(a[11]);
  const int return_lse = PyObject_IsTrue(a[15]);
  const int causal = PyObject_IsTrue(a[16]);
  const double scale = PyFloat_AsDouble(a[17]);
  if (PyErr_Occurred()) return nullptr;
  Pool pool;
  if (!pool.get(a[2]) || pool.hkv != hkv || pool.d != d) return general();
  const at::Tensor* q = rows(a[1], hq, d);
  float* scales;
  if (!q || q->size(0) < qo_rows || !get_scales(a[12], pool, &scales)) return general();
  const int32_t *qo, *indices, *indptr, *last;
  int64_t n_ind = 0;
  if (!meta(a[3], q->device(), bsz + 1, &qo) || !meta(a[4], q->device(), -1, &indices, &n_ind) ||
      !meta(a[5], q->device(), bsz + 1, &indptr) || !meta(a[6], q->device(), bsz, &last))
    return general();
  Outputs o;
  if (!o.get(a[13], a[14], return_lse, *q, q->size(0), hq, d)) return general();
  void* stream;
  if (!raw_stream(q->device(), &stream)) return nullptr;
  const void* qp = q->data_ptr();
  void* pp = pool.ptr();
  void* op = o.out.data_ptr();
  Scratch scratch;
  scratch.get(plan, *q);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_entry.prefill_run(plan, qp, q->stride(0), q->stride(1), code16(*q), qo, pp, pool.code,
                           scales, (int32_t)pool.pages, indices, (int32_t)n_ind, indptr, last, op,
                           static_cast<float*>(o.lse_ptr), causal, (float)scale, scratch.ptr,
                           scratch.bytes, stream);
  Py_END_ALLOW_THREADS
  return rc ? PyLong_FromLong(rc) : o.result();
  END_HANDLE_TH_ERRORS
}

// What the three append calls share: rows, pool, metadata, scales, counters.
struct AppendArgs {
  Pool pool;
  const at::Tensor *k = nullptr, *v = nullptr;
  const int32_t *bi, *pos, *ind, *indptr;
  int64_t nnz = 0, n_ind = 0, n_ptr = 0;
  float* scales = nullptr;
  int32_t* flag = nullptr;
  void* stream = nullptr;
  // a: key, value, batch_indices, positions, pool, indices, indptr, scales, flag
  bool get(PyObject* const* a) {
    if (!pool.get(a[4])) return false;
    k = rows(a[0], pool.hkv, pool.d);
    v = rows(a[1], pool.hkv, pool.d);
    if (!k || !v || k->scalar_type() != v->scalar_type() || k->size(0) != v->size(0))
      return false;
    if (pool.code != PAGEDATTN_E4M3 && pool.code != code16(*k)) return false;
    nnz = k->size(0);
    return meta(a[2], pool.device, nnz, &bi) && meta(a[3], pool.device, nnz, &pos) &&
           meta(a[5], pool.device, -1, &ind, &n_ind) &&
           meta(a[6], pool.device, -1, &indptr, &n_ptr) && get_scales(a[7], pool, &scales) &&
           get_flag(a[8], pool.code == PAGEDATTN_E4M3 ? 2 : 1, &flag);
  }
};

PyObject* done(int rc) {
  if (rc) return PyLong_FromLong(rc);
  Py_RETURN_NONE;
}

// append(key, value, batch_indices, positions, pool, indices, indptr, scales, flag, last)
PyObject* append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arg_count(n, 10)) return nullptr;
  AppendArgs x;
  const at::Tensor* last = plain(a[9]);
  if (!last || !x.get(a)) return general();
  if (!raw_stream(x.pool.device, &x.stream)) return nullptr;
  const void *kp = x.k->data_ptr(), *vp = x.v->data_ptr();
  void* pp = x.pool.ptr();
  const auto* lp = static_cast<const int32_t*>(last->data_ptr());
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_entry.append(kp, vp, x.k->stride(0), x.k->stride(1), x.v->stride(0), x.v->stride(1),
                      code16(*x.k), x.bi, x.pos, (int32_t)x.nnz, pp, x.pool.code, x.scales,
                      (int32_t)x.pool.pages, x.ind, (int32_t)x.n_ind, x.indptr, lp,
                      (int32_t)x.n_ptr - 1, (int32_t)x.pool.hkv, (int32_t)x.pool.d, kPageSize,
                      x.flag, x.stream);
  Py_END_ALLOW_THREADS
  return done(rc);
  END_HANDLE_TH_ERRORS
}

// rope_append(key, value, batch_indices, positions, pool, indices, indptr,
//             scales, flag, q, rope_scale, rope_theta)
PyObject* rope_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arg_count(n, 12)) return nullptr;
  const double rope_scale = PyFloat_AsDouble(a[10]), rope_theta = PyFloat_AsDouble(a[11]);
  if (PyErr_Occurred()) return nullptr;
  AppendArgs x;
  if (!x.get(a)) return general();
  const at::Tensor* q = rows(a[9], -1, x.pool.d);
  if (!q || q->size(0) != x.nnz || q->scalar_type() != x.k->scalar_type()) return general();
  if (!raw_stream(x.pool.device, &x.stream)) return nullptr;
  void *qp = q->data_ptr(), *kp = x.k->data_ptr(), *pp = x.pool.ptr();
  const void* vp = x.v->data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_entry.rope_append(qp, q->stride(0), q->stride(1), (int32_t)q->size(1), kp, vp,
                           x.k->stride(0), x.k->stride(1), x.v->stride(0), x.v->stride(1),
                           code16(*q), x.bi, x.pos, (int32_t)x.nnz, (float)rope_scale,
                           (float)rope_theta, pp, x.pool.code, x.scales, (int32_t)x.pool.pages,
                           x.ind, (int32_t)x.n_ind, x.indptr, (int32_t)x.n_ptr - 1,
                           (int32_t)x.pool.hkv, (int32_t)x.pool.d, kPageSize, x.flag, x.stream);
  Py_END_ALLOW_THREADS
  return done(rc);
  END_HANDLE_TH_ERRORS
}

// append_amax(key, value, batch_indices, positions, pool, indices, indptr, scales, flag)
PyObject* append_amax(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arg_count(n, 9)) return nullptr;
  AppendArgs x;
  if (!x.get(a) || x.pool.code != PAGEDATTN_E4M3) return general();
  if (!raw_stream(x.pool.device, &x.stream)) return nullptr;
  const void *kp = x.k->data_ptr(), *vp = x.v->data_ptr();
  void* pp = x.pool.ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_entry.append_amax(kp, vp, x.k->stride(0), x.k->stride(1), x.v->stride(0),
                           x.v->stride(1), code16(*x.k), x.bi, x.pos, (int32_t)x.nnz, pp,
                           x.scales, (int32_t)x.pool.pages, x.ind, (int32_t)x.n_ind, x.indptr,
                           (int32_t)x.n_ptr - 1, (int32_t)x.pool.hkv, (int32_t)x.pool.d,
                           kPageSize, x.flag, x.stream);
  Py_END_ALLOW_THREADS
  return done(rc);
  END_HANDLE_TH_ERRORS
}

// bind(raw_stream, {name: address}): the current-stream function and the C
// entry points, once, before any other call
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arg_count(n, 2)) return nullptr;
  bool ok = true;
  auto at = [&](const char* name) -> void* {
    PyObject* v = PyDict_GetItemString(a[1], name);
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
    if (!p) ok = false;
    return p;
  };
  Entries e;
  e.scratch_bytes =
      reinterpret_cast<decltype(e.scratch_bytes)>(at("pagedattn_plan_scratch_bytes"));
  e.decode_run = reinterpret_cast<decltype(e.decode_run)>(at("pagedattn_decode_run_scratch"));
  e.prefill_run = reinterpret_cast<decltype(e.prefill_run)>(at("pagedattn_prefill_run_scratch"));
  e.append = reinterpret_cast<decltype(e.append)>(at("pagedattn_append_paged_kv_cache"));
  e.rope_append =
      reinterpret_cast<decltype(e.rope_append)>(at("pagedattn_rope_append_paged_kv_cache"));
  e.append_amax = reinterpret_cast<decltype(e.append_amax)>(
      at("pagedattn_append_paged_kv_cache_e4m3_amax"));
  if (!ok) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: missing entry point");
    return nullptr;
  }
  Py_INCREF(a[0]);
  Py_XSETREF(g_raw_stream, a[0]);
  g_entry = e;
  Py_RETURN_NONE;
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef kMethods[] = {
    {"bind", FAST(bind), nullptr},
    {"decode_run", FAST(decode_run), nullptr},
    {"prefill_run", FAST(prefill_run), nullptr},
    {"append", FAST(append), nullptr},
    {"rope_append", FAST(rope_append), nullptr},
    {"append_amax", FAST(append_amax), nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) { return PyModule_Create(&kModule); }
