// The two operators' checks and calls without the interpreter (module _vmi_host, loaded by vllmini_amd/_lib.py).
//
// A decode step of a small batch is bound by what the host does per call: read some thirty sizes, strides, types and devices off eight
// tensors (one attribute of the interpreter each: 5 us), pack twenty arguments (2 us), launch.  Here the same facts are read off the
// tensors directly.  Every function answers None, having done nothing, for whatever is not the plain case below — another type, a
// subclass of Tensor, a shape or stride that does not fit, no workspace yet — and the caller goes through ops.py's own checks, which
// accept it or say what is wrong; else the C-ABI's return code.  Both operators of one sequence, 12 heads of 64, 300 tokens, one call behind
// the other: 17.6 -> 12.4 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "vmi_paged_attention.h"

namespace {

struct Entries {   // of one of the libraries; addresses come from ctypes, the library stays loaded for the process
  decltype(&vmi_paged_attention_v1_f16) v1;
  decltype(&vmi_paged_attention_v1_f16_variant) v1_variant;
  decltype(&vmi_paged_attention_v1_f16_ws) v1_ws;
  decltype(&vmi_paged_attention_v1_fp8) fp8;
  decltype(&vmi_paged_attention_v1_fp8_ws) fp8_ws;
  decltype(&vmi_reshape_and_cache_f16) cache;
  decltype(&vmi_reshape_and_cache_fp8) cache_fp8;
};
constexpr const char* ENTRIES = "vmi_host.entries";

const at::Tensor* tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }
bool whole(PyObject* o, int64_t* v) {
  if (!PyLong_Check(o)) return false;
  *v = PyLong_AsLongLong(o);
  return !PyErr_Occurred();
}
bool real(PyObject* o, float* v) {
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  *v = (float)PyFloat_AsDouble(o);
  return !PyErr_Occurred();
}
// 0: 16-bit pages, 1: fp8 E4M3 pages, -1: something else
int pages(PyObject* o) {
  if (!PyUnicode_Check(o)) return -1;
  if (PyUnicode_CompareWithASCIIString(o, "auto") == 0) return 0;
  return PyUnicode_CompareWithASCIIString(o, "fp8") == 0 || PyUnicode_CompareWithASCIIString(o, "fp8_e4m3") == 0 ? 1 : -1;
}
bool page_type(const at::Tensor& t, int fp8) {
  return fp8 ? t.scalar_type() == at::kByte || t.scalar_type() == at::kFloat8_e4m3fn : t.scalar_type() == at::kHalf;
}
PyObject* other_way() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// (entries, out, query, key_cache, value_cache, num_kv_heads, scale, block_tables, seq_lens, block_size, max_seq_len, kv_cache_dtype, kv_scale,
//  variant, workspaces or None)
PyObject* attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 15) return other_way();
  const auto* fn = static_cast<const Entries*>(PyCapsule_GetPointer(a[0], ENTRIES));
  const at::Tensor *out = tensor(a[1]), *q = tensor(a[2]), *kc = tensor(a[3]), *vc = tensor(a[4]), *tab = tensor(a[7]), *lens = tensor(a[8]);
  int64_t kv_heads, bs, max_len, variant;
  float scale, kv_scale;
  const int fp8 = pages(a[11]);
  if (!fn || !out || !q || !kc || !vc || !tab || !lens || fp8 < 0 || !whole(a[5], &kv_heads) || !real(a[6], &scale) || !whole(a[9], &bs) ||
      !whole(a[10], &max_len) || !real(a[12], &kv_scale) || !whole(a[13], &variant))
    return other_way();
  try {
    if (q->dim() != 3 || kc->dim() != 5 || vc->dim() != 4 || tab->dim() != 2 || lens->dim() != 1 || !q->is_cuda()) return other_way();
    const auto dev = q->device();
    for (const at::Tensor* t : {out, kc, vc, tab, lens})
      if (t->device() != dev) return other_way();
    if (q->scalar_type() != at::kHalf || out->scalar_type() != at::kHalf || !page_type(*kc, fp8) || !page_type(*vc, fp8) ||
        tab->scalar_type() != at::kInt || lens->scalar_type() != at::kInt)
      return other_way();
    const int64_t S = q->size(0), H = q->size(1), D = q->size(2), x = fp8 ? 16 : 8, tile = D * bs;
    if (kc->size(4) != x || kc->size(3) != bs || vc->size(3) != bs || kc->size(2) * x != D || vc->size(2) != D || kc->size(1) != kv_heads ||
        vc->size(1) != kv_heads || q->stride(2) != 1 || q->stride(1) != D)
      return other_way();
    // every (block, head) tile dense (dimensions of size 1 carry no layout), both caches strided alike
    if (kc->stride(4) != 1 || (kc->stride(3) != x && bs != 1) || (kc->stride(2) != bs * x && kc->size(2) != 1) ||
        (kc->stride(1) != tile && kv_heads != 1) || (vc->stride(3) != 1 && bs != 1) || (vc->stride(2) != bs && D != 1) ||
        (vc->stride(1) != tile && kv_heads != 1) || vc->stride(0) != kc->stride(0) || vc->stride(1) != kc->stride(1))
      return other_way();
    if (!out->is_contiguous() || out->numel() != S * H * D || tab->size(0) != S || tab->stride(1) != 1 ||
        (tab->stride(0) != tab->size(1) && S > 1) || lens->size(0) != S || !lens->is_contiguous())
      return other_way();
    if (S > INT32_MAX || H > INT32_MAX || kv_heads > INT32_MAX || max_len > INT32_MAX || max_len < INT32_MIN || tab->size(1) > INT32_MAX ||
        variant > INT32_MAX || variant < INT32_MIN)
      return other_way();
    const int index = dev.index();
    void* const stream = c10::hip::getCurrentHIPStream(index).stream();
    void* ws = nullptr;
    int64_t ws_bytes = 0;
    if (a[14] != Py_None && (D == 64 || D == 128)) {   // the workspace of this device and stream
      PyObject* key = Py_BuildValue("(iK)", index, (unsigned long long)(uintptr_t)stream);
      PyObject* held = key && PyDict_Check(a[14]) ? PyDict_GetItemWithError(a[14], key) : nullptr;   // (borrowed)
      Py_XDECREF(key);
      const at::Tensor* w = held ? tensor(held) : nullptr;
      if (!w) return other_way();
      ws = w->data_ptr();
      ws_bytes = w->numel();
    }
    void *po = out->data_ptr(), *pq = q->data_ptr(), *pk = kc->data_ptr(), *pv = vc->data_ptr();
    const auto* pt = static_cast<const int32_t*>(tab->data_ptr());
    const auto* pl = static_cast<const int32_t*>(lens->data_ptr());
    const int64_t qs = q->stride(0), ks = kc->stride(0), hs = kc->stride(1), MB = tab->size(1);
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    if (fp8 && ws)
      rc = fn->fp8_ws(po, pq, pk, pv, S, H, D, kv_heads, scale, pt, pl, bs, max_len, MB, nullptr, qs, ks, hs, index, stream, kv_scale, ws, ws_bytes, variant);
    else if (fp8)
      rc = fn->fp8(po, pq, pk, pv, S, H, D, kv_heads, scale, pt, pl, bs, max_len, MB, nullptr, qs, ks, hs, index, stream, kv_scale, variant);
    else if (ws)
      rc = fn->v1_ws(po, pq, pk, pv, S, H, D, kv_heads, scale, pt, pl, bs, max_len, MB, nullptr, qs, ks, hs, index, stream, ws, ws_bytes, variant);
    else if (variant)
      rc = fn->v1_variant(po, pq, pk, pv, S, H, D, kv_heads, scale, pt, pl, bs, max_len, MB, nullptr, qs, ks, hs, index, stream, variant);
    else
      rc = fn->v1(po, pq, pk, pv, S, H, D, kv_heads, scale, pt, pl, bs, max_len, MB, nullptr, qs, ks, hs, index, stream);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
  } catch (const std::exception&) {   // (a tensor without storage, say: the other way says so)
    return other_way();
  }
}

// (entries, key, value, key_cache, value_cache, slot_mapping, kv_cache_dtype, kv_scale)
PyObject* cache(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 8) return other_way();
  const auto* fn = static_cast<const Entries*>(PyCapsule_GetPointer(a[0], ENTRIES));
  const at::Tensor *k = tensor(a[1]), *v = tensor(a[2]), *kc = tensor(a[3]), *vc = tensor(a[4]), *slots = tensor(a[5]);
  const int fp8 = pages(a[6]);
  float kv_scale;
  if (!fn || !k || !v || !kc || !vc || !slots || fp8 < 0 || !real(a[7], &kv_scale)) return other_way();
  try {
    if (k->dim() != 3 || v->dim() != 3 || k->sizes() != v->sizes() || kc->dim() != 5 || vc->dim() != 4 || !k->is_cuda()) return other_way();
    const auto dev = k->device();
    for (const at::Tensor* t : {v, kc, vc, slots})
      if (t->device() != dev) return other_way();
    const int64_t T = k->size(0), H = k->size(1), D = k->size(2), bs = kc->size(3), x = kc->size(4);
    if (k->scalar_type() != at::kHalf || v->scalar_type() != at::kHalf || !page_type(*kc, fp8) || !page_type(*vc, fp8) ||
        slots->scalar_type() != at::kLong || !kc->is_contiguous() || !vc->is_contiguous() || kc->size(1) != H || kc->size(2) * x != D ||
        vc->size(1) != H || vc->size(2) != D || vc->size(3) != bs || k->stride(2) != 1 || k->stride(1) != D || v->stride(2) != 1 ||
        v->stride(1) != D || slots->numel() != T || !slots->is_contiguous() || T > INT32_MAX || H > INT32_MAX || bs > INT32_MAX)
      return other_way();
    const int index = dev.index();
    void* const stream = c10::hip::getCurrentHIPStream(index).stream();
    void *pk = k->data_ptr(), *pv = v->data_ptr(), *pkc = kc->data_ptr(), *pvc = vc->data_ptr();
    const auto* ps = static_cast<const int64_t*>(slots->data_ptr());
    const int64_t ks = k->stride(0), vs = v->stride(0);
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = fp8 ? fn->cache_fp8(pk, pv, pkc, pvc, ps, T, H, D, bs, x, ks, vs, kv_scale, index, stream)
             : fn->cache(pk, pv, pkc, pvc, ps, T, H, D, bs, x, ks, vs, index, stream);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
  } catch (const std::exception&) {
    return other_way();
  }
}

// (addresses of the seven entries, in the order of Entries) -> what the other two take first
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  constexpr Py_ssize_t N = sizeof(Entries) / sizeof(void*);
  void* at[N];
  if (n != N) {
    PyErr_SetString(PyExc_TypeError, "bind: seven addresses");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < N; ++i) {
    at[i] = PyLong_AsVoidPtr(a[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  auto* e = new Entries;
  static_assert(sizeof(*e) == sizeof(at), "function pointers only");
  memcpy(static_cast<void*>(e), at, sizeof(at));
  return PyCapsule_New(e, ENTRIES, [](PyObject* c) { delete static_cast<Entries*>(PyCapsule_GetPointer(c, ENTRIES)); });
}

PyMethodDef methods[] = {{"bind", reinterpret_cast<PyCFunction>(bind), METH_FASTCALL, nullptr},
                         {"attend", reinterpret_cast<PyCFunction>(attend), METH_FASTCALL, nullptr},
                         {"cache", reinterpret_cast<PyCFunction>(cache), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_vmi_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__vmi_host(void) { return PyModule_Create(&module); }
