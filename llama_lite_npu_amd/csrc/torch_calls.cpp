// The per-layer calls of a prefill from PyTorch tensors: the checks of ops.py's wrappers and the
// conversion of their arguments, in native code. A short prompt is bound by the host (two calls per
// layer against 12 us of kernels), and there most of a call was Python: some sixty attribute reads
// on tensors and twenty conversions by ctypes. One prompt of 203 tokens, 28 layers, 16 / 8 heads: 543 -> 359 us. Two
// chunks of 64 rows over up to 1500 cached tokens, 32 / 8 heads of 64, cut along their keys: 638 -> 426 us.
//
// A function takes what it recognises as a plain, well-formed call; anything else (another dtype, a
// shape that does not fit, a tensor subclass) it leaves alone and answers None, and the wrapper goes
// through its own checks, conversions and messages. None says that the library was not called: what it
// answered goes back as it is, since a launch error is reported after the launch (and may be an older
// one of the thread), and the epilogue, which works in place, must not run twice.
#include <Python.h>
#include <stdio.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "litekv.h"

namespace {

// A tensor as torch itself makes them (or an nn.Parameter), on the GPU; else null.
const at::Tensor *gpu_tensor(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

const at::Tensor *half_tensor(PyObject *o) {
  const at::Tensor *t = gpu_tensor(o);
  return t != nullptr && t->scalar_type() == at::kHalf ? t : nullptr;
}

// int32, contiguous, `numel` elements (any number if negative)
const at::Tensor *index_tensor(PyObject *o, int64_t numel) {
  const at::Tensor *t = gpu_tensor(o);
  return t != nullptr && t->scalar_type() == at::kInt && t->is_contiguous() && (numel < 0 || t->numel() == numel)
             ? t
             : nullptr;
}

// [T, heads, d] rows whose [heads, d] block is contiguous: elements between tokens, or -1
int64_t row_stride(const at::Tensor &t, int64_t tokens, int64_t heads, int64_t d) {
  if (t.dim() != 3 || t.size(0) != tokens || t.size(1) != heads || t.size(2) != d) return -1;
  if (t.stride(2) != 1 || t.stride(1) != d) return -1;
  return tokens > 1 ? t.stride(0) : std::max(t.stride(0), heads * d);
}

enum Format { kNone, kF16, kFp8, kInt8 };

// A [slots, 2 * Hkv, D] pool and its scales (codes only); kNone: not a plain one.
struct Pool {
  Format format = kNone;
  const at::Tensor *t = nullptr;
  const void *scales = nullptr;
  int64_t slots = 0, hkv = 0, d = 0;
};

Pool pool_of(PyObject *pool, PyObject *scales) {
  Pool p;
  p.t = gpu_tensor(pool);
  if (p.t == nullptr || p.t->dim() != 3 || !p.t->is_contiguous() || p.t->size(1) % 2 != 0) return p;
  p.slots = p.t->size(0);
  p.hkv = p.t->size(1) / 2;
  p.d = p.t->size(2);
  switch (p.t->scalar_type()) {
    case at::kHalf:
      if (scales == Py_None) p.format = kF16;
      return p;
    case at::kByte:
    case at::kFloat8_e4m3fn:
    case at::kChar: {
      const at::Tensor *s = gpu_tensor(scales);
      if (s == nullptr || s->scalar_type() != at::kFloat || !s->is_contiguous() || s->numel() != 2 * p.hkv) return p;
      p.scales = s->data_ptr();
      p.format = p.t->scalar_type() == at::kChar ? kInt8 : kFp8;
      return p;
    }
    default:
      return p;
  }
}

void *address(const at::Tensor *t) { return t != nullptr ? t->data_ptr() : nullptr; }

// Runs `call` without the interpreter lock, as ctypes does.
template <typename Call>
int unlocked(Call call) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call();
  Py_END_ALLOW_THREADS
  return rc;
}

// (q, k, v, slot_mapping, kv_pool, q_norm_weight, k_norm_weight, cos, sin, eps, kv_scales, stream)
// -> True if launched, the library's status if that is not 0, or None
PyObject *qk_norm_rope_append(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 12) Py_RETURN_NONE;
  try {
    const at::Tensor *q = half_tensor(a[0]), *k = half_tensor(a[1]), *v = half_tensor(a[2]);
    if (q == nullptr || k == nullptr || v == nullptr || q->dim() != 3) Py_RETURN_NONE;
    const Pool pool = pool_of(a[4], a[10]);
    if (pool.format == kNone) Py_RETURN_NONE;
    const int64_t t = q->size(0), hq = q->size(1), d = pool.d;
    const int64_t qs = row_stride(*q, t, hq, d), ks = row_stride(*k, t, pool.hkv, d), vs = row_stride(*v, t, pool.hkv, d);
    const at::Tensor *slots = index_tensor(a[3], t);
    if (qs < 0 || ks < 0 || vs < 0 || slots == nullptr) Py_RETURN_NONE;
    const at::Tensor *qw = nullptr, *kw = nullptr, *cos = nullptr, *sin = nullptr;
    if (a[5] != Py_None || a[6] != Py_None) {
      qw = half_tensor(a[5]);
      kw = half_tensor(a[6]);
      if (qw == nullptr || kw == nullptr || qw->numel() != d || kw->numel() != d || !qw->is_contiguous() ||
          !kw->is_contiguous()) {
        Py_RETURN_NONE;
      }
    }
    int64_t cs = 0;
    if (a[7] != Py_None || a[8] != Py_None) {
      cos = half_tensor(a[7]);
      sin = half_tensor(a[8]);
      if (cos == nullptr || sin == nullptr || cos->dim() != 2 || sin->dim() != 2 || cos->size(0) != t ||
          sin->size(0) != t || cos->size(1) != sin->size(1) || cos->size(1) < d / 2 || cos->stride(1) != 1 ||
          sin->stride(1) != 1 || cos->stride(0) != sin->stride(0)) {
        Py_RETURN_NONE;
      }
      cs = cos->stride(0);
    }
    const double eps = PyFloat_AsDouble(a[9]);
    void *stream = PyLong_AsVoidPtr(a[11]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (t > INT32_MAX || hq > INT32_MAX || pool.hkv > INT32_MAX || d > INT32_MAX) Py_RETURN_NONE;
    void *qp = address(q), *kp = address(k), *vp = address(v), *qwp = address(qw), *kwp = address(kw);
    void *cp = address(cos), *sp = address(sin), *pp = address(pool.t);
    const int32_t *slp = static_cast<const int32_t *>(address(slots));
    const float *scales = static_cast<const float *>(pool.scales);
    const int rc = unlocked([&] {
      switch (pool.format) {
        case kF16:
          return litekv_qk_norm_rope_append(qp, qs, kp, ks, vp, vs, qwp, kwp, cp, sp, cs, slp, pp, (int32_t)t, (int32_t)hq,
                                            (int32_t)pool.hkv, (int32_t)d, pool.slots, (float)eps, stream);
        case kFp8:
          return litekv_qk_norm_rope_append_fp8(qp, qs, kp, ks, vp, vs, qwp, kwp, cp, sp, cs, slp, pp, scales, (int32_t)t,
                                                (int32_t)hq, (int32_t)pool.hkv, (int32_t)d, pool.slots, (float)eps, stream);
        default:
          return litekv_qk_norm_rope_append_int8(qp, qs, kp, ks, vp, vs, qwp, kwp, cp, sp, cs, slp, pp, scales, (int32_t)t,
                                                 (int32_t)hq, (int32_t)pool.hkv, (int32_t)d, pool.slots, (float)eps, stream);
      }
    });
    if (rc != 0) return PyLong_FromLong(rc);
    Py_RETURN_TRUE;
  } catch (...) {  // (a tensor without storage, under a transform: the wrapper meets the same and says so)
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// (q, kv_pool, block_table, cu_q_lens, context_lens, max_q_len, softmax_scale, page_size, kv_scales,
//  max_kv_len or None, stream) -> the output, or the library's status if that is not 0, or None. A launch
// that is to be cut along its keys (one request's chunk over a long history) gets the workspace of its partial rows
// here, which like the wrapper's goes back to the allocator of the current stream behind the launches.
PyObject *paged_prefill(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 11) Py_RETURN_NONE;
  try {
    const at::Tensor *q = half_tensor(a[0]);
    if (q == nullptr || q->dim() != 3) Py_RETURN_NONE;
    const Pool pool = pool_of(a[1], a[8]);
    if (pool.format == kNone) Py_RETURN_NONE;
    const int64_t t = q->size(0), hq = q->size(1), d = pool.d;
    const int64_t qs = row_stride(*q, t, hq, d);
    const at::Tensor *cu = index_tensor(a[3], -1);
    if (qs < 0 || cu == nullptr || cu->numel() < 1) Py_RETURN_NONE;
    const int64_t b = cu->numel() - 1;
    const at::Tensor *table = index_tensor(a[2], -1);
    if (table == nullptr || table->dim() != 2 || table->size(0) != b) Py_RETURN_NONE;
    const at::Tensor *ctx = nullptr;
    if (a[4] != Py_None) {
      ctx = index_tensor(a[4], b);
      if (ctx == nullptr) Py_RETURN_NONE;
    }
    const int64_t max_q = PyLong_AsLongLong(a[5]), page = PyLong_AsLongLong(a[7]);
    const int64_t max_kv = a[9] == Py_None ? -1 : PyLong_AsLongLong(a[9]);
    const double scale = PyFloat_AsDouble(a[6]);
    void *stream = PyLong_AsVoidPtr(a[10]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (page < 1 || page > 65536 || pool.slots % page != 0 || max_q < 0 || max_q > INT32_MAX || t > INT32_MAX || b > INT32_MAX ||
        hq > INT32_MAX || pool.hkv > INT32_MAX || d > INT32_MAX || table->stride(0) > INT32_MAX) {
      Py_RETURN_NONE;
    }
    // (the count's rule and the rows it looks at as in the wrapper)
    int32_t slices = 1;
    if (a[9] != Py_None && t * hq > 0 && t * hq <= 128 * 512) {
      slices = litekv_paged_prefill_key_slices((int32_t)b, (int32_t)hq, (int32_t)pool.hkv, (int32_t)d, (int32_t)max_q, max_kv);
    }
    at::Tensor out = at::empty({t, hq, d}, q->options());
    at::Tensor partials;
    size_t partial_bytes = 0;
    if (slices > 1) {
      partial_bytes = litekv_paged_prefill_split_workspace_bytes(t, (int32_t)hq, (int32_t)d, slices);
      partials = at::empty({(int64_t)(partial_bytes / sizeof(float))}, q->options().dtype(at::kFloat));
    }
    const void *qp = address(q), *pp = address(pool.t);
    const int32_t *tp = static_cast<const int32_t *>(address(table)), *cup = static_cast<const int32_t *>(address(cu));
    const int32_t *ctxp = static_cast<const int32_t *>(address(ctx));
    const float *scales = static_cast<const float *>(pool.scales);
    void *op = address(&out);
    PyObject *result = THPVariable_Wrap(std::move(out));  // (before the launch: it may throw)
    const int32_t ts = (int32_t)table->stride(0);
    const int64_t pages = pool.slots / page;
    void *wp = slices > 1 ? partials.data_ptr() : nullptr;
    const int rc = unlocked([&] {
      if (slices > 1 && pool.format == kF16) {
        return litekv_paged_prefill_split(qp, qs, pp, tp, ts, cup, ctxp, op, hq * d, (int32_t)b, (int32_t)hq, (int32_t)pool.hkv,
                                          (int32_t)d, (int32_t)page, pages, (int32_t)max_q, t, slices, wp, partial_bytes,
                                          (float)scale, stream);
      }
      if (slices > 1) {
        return litekv_paged_prefill_split_q8(qp, qs, pp, scales, pool.format == kInt8, tp, ts, cup, ctxp, op, hq * d, (int32_t)b,
                                             (int32_t)hq, (int32_t)pool.hkv, (int32_t)d, (int32_t)page, pages, (int32_t)max_q, t,
                                             slices, wp, partial_bytes, (float)scale, stream);
      }
      return litekv_paged_prefill_bounded(qp, qs, pp, scales, pool.format == kInt8, tp, ts, cup, ctxp, op, hq * d, (int32_t)b,
                                          (int32_t)hq, (int32_t)pool.hkv, (int32_t)d, (int32_t)page, pages, (int32_t)max_q,
                                          max_kv < 0 ? 0 : max_kv, (float)scale, stream);
    });
    if (rc == 0) return result;
    Py_DECREF(result);
    return PyLong_FromLong(rc);
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

PyMethodDef methods[] = {
    {"qk_norm_rope_append", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(qk_norm_rope_append)), METH_FASTCALL, nullptr},
    {"paged_prefill", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(paged_prefill)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
  PyObject *m = PyModule_Create(&module);
  if (m == nullptr) return nullptr;
  char torch_version[32];
  snprintf(torch_version, sizeof(torch_version), "%d.%d.%d", TORCH_VERSION_MAJOR, TORCH_VERSION_MINOR, TORCH_VERSION_PATCH);
  if (PyModule_AddIntConstant(m, "ABI_VERSION", LITEKV_ABI_VERSION) != 0 ||
      PyModule_AddStringConstant(m, "TORCH_VERSION", torch_version) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
