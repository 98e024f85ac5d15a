// binding.cpp -- the per-layer call's launch path from torch tensors, for CPython.
//
// scatter(src, kv, slots, block_size, hnd, shift, k_scale, error_flags) is
// shift_kernels.scatter_shifted's usual call: it reads the tensors through torch's C++
// interface, checks what that function checks and calls mkv_scatter_shifted on the current
// stream.  Through Python methods and ctypes the same call spent 3.6 us of its 6.7 around
// the launch, longer than the kernel of a short span runs (2.4 us for 300 tokens), so a loop
// over layers was bound by it: 28 calls of 301 fp16 tokens 165 -> 79 to 108 us, a process
// settling at one figure or another between these (2.8 to 3.8 us a call).
//
// Returns the library's status, or None wherever the call is not the usual one (tensors
// that need a copy or a conversion, subclasses and wrapped tensors, another current device,
// anything the general path refuses): nothing has been launched then, and the caller takes
// the general path, which also raises the errors.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "marathon_kvshift.h"

namespace {

typedef decltype(&mkv_scatter_shifted) scatter_fn;
scatter_fn g_scatter = nullptr;

PyObject* s_delta;
PyObject* s_cos;
PyObject* s_sgn;
PyObject* s_emb_cos;
PyObject* s_rotary;

struct Ref {  // one owned reference
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {}
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

// The plain tensor behind `o` (no subclass, nothing that wraps another tensor), or null.
const at::Tensor* plain(PyObject* o) {
  if (o == nullptr || !THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.layout() == at::kStrided && t.has_storage() ? &t : nullptr;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16:
      return MKV_BF16;
    case at::kHalf:
      return MKV_F16;
    case at::kFloat:
      return MKV_F32;
    case at::kFloat8_e4m3fn:
      return MKV_FP8_E4M3;
    default:
      return -1;
  }
}

enum { kUsual, kOther, kError };

struct Shift {
  int64_t rotary = 0;
  const float* cos = nullptr;
  const float* sgn = nullptr;
};

// A RopeShift's tables; kOther unless they are plain tensors on `dev` that fit.
int read_shift(PyObject* shift, const at::Device& dev, int64_t head_size, Shift& out) {
  const Ref emb(PyObject_GetAttr(shift, s_emb_cos));
  const Ref delta(emb.p != nullptr ? PyObject_GetAttr(shift, s_delta) : nullptr);
  if (delta.p == nullptr) return kError;
  const at::Tensor* e = plain(emb.p);
  if (e == nullptr || !PyLong_CheckExact(delta.p)) return kOther;
  const Ref declared(PyObject_GetAttr(shift, s_rotary));
  if (declared.p == nullptr) {  // the reference's RopeShift has no such field
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return kError;
    PyErr_Clear();
  } else if (declared.p != Py_None) {
    if (!PyLong_CheckExact(declared.p)) return kOther;
    int over = 0;
    if (PyLong_AsLongLongAndOverflow(declared.p, &over) != e->numel() || over != 0) return kOther;
  }
  const int moved = PyObject_IsTrue(delta.p);
  if (moved == 0 || e->numel() == 0) return kUsual;  // a plain scatter
  const Ref cos_o(PyObject_GetAttr(shift, s_cos));
  const Ref sgn_o(cos_o.p != nullptr ? PyObject_GetAttr(shift, s_sgn) : nullptr);
  if (sgn_o.p == nullptr) return kError;
  const at::Tensor* cos = plain(cos_o.p);
  const at::Tensor* sgn = plain(sgn_o.p);
  if (cos == nullptr || sgn == nullptr || cos->device() != dev || sgn->device() != dev ||
      cos->numel() != head_size || sgn->numel() != head_size || e->numel() > INT32_MAX)
    return kOther;
  out.rotary = e->numel();
  out.cos = static_cast<const float*>(cos->data_ptr());
  out.sgn = static_cast<const float*>(sgn->data_ptr());
  return kUsual;
}

PyObject* scatter(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 8 || g_scatter == nullptr) {
    PyErr_SetString(PyExc_TypeError, "scatter takes 8 arguments, after bind()");
    return nullptr;
  }
  try {
    if (at::impl::PythonTorchFunctionTLS::stack_len() != 0) Py_RETURN_NONE;
    const at::Tensor* src = plain(args[0]);
    const at::Tensor* kv = plain(args[1]);
    const at::Tensor* slots = plain(args[2]);
    if (src == nullptr || kv == nullptr || slots == nullptr || !kv->is_cuda() ||
        src->dim() != 3 || kv->dim() != 4)
      Py_RETURN_NONE;
    const at::Device dev = kv->device();
    const int64_t n = src->size(0), two_d = src->size(2);
    const int code = dtype_code(kv->scalar_type());
    if (n == 0 || two_d % 2 != 0 || kv->size(3) != two_d || code < 0 ||
        src->scalar_type() != kv->scalar_type() || src->device() != dev ||
        slots->device() != dev || src->stride(2) != 1 || kv->stride(3) != 1 ||
        slots->scalar_type() != at::kLong || !slots->is_contiguous() || slots->numel() != n ||
        src->size(1) > INT32_MAX || two_d > INT32_MAX)
      Py_RETURN_NONE;
    if (!PyLong_CheckExact(args[3])) Py_RETURN_NONE;
    int over = 0;
    const long long block_size = PyLong_AsLongLongAndOverflow(args[3], &over);
    if (over != 0 || block_size > INT32_MAX || block_size < INT32_MIN) Py_RETURN_NONE;
    const int hnd = PyObject_IsTrue(args[4]);
    if (hnd < 0) return nullptr;
    Shift sh;
    if (args[5] != Py_None) {
      const int got = read_shift(args[5], dev, two_d / 2, sh);
      if (got == kError) return nullptr;
      if (got == kOther) Py_RETURN_NONE;
    }
    const float* scale = nullptr;
    if (sh.rotary > 0 && code == MKV_FP8_E4M3) {
      const at::Tensor* k = plain(args[6]);
      if (k == nullptr || k->device() != dev || k->scalar_type() != at::kFloat || k->numel() < 1)
        Py_RETURN_NONE;
      scale = static_cast<const float*>(k->data_ptr());
    }
    int32_t* flags = nullptr;
    if (args[7] != Py_None) {
      const at::Tensor* f = plain(args[7]);
      if (f == nullptr) Py_RETURN_NONE;
      flags = static_cast<int32_t*>(f->data_ptr());
    }
    if (c10::hip::current_device() != dev.index()) Py_RETURN_NONE;
    void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
    const int head_dim = hnd ? 1 : 2, off_dim = hnd ? 2 : 1;
    const void* src_p = src->data_ptr();
    void* kv_p = kv->data_ptr();
    const int64_t* slots_p = static_cast<const int64_t*>(slots->data_ptr());
    const int64_t st = src->stride(0), sh_ = src->stride(1), kb = kv->stride(0),
                  kh = kv->stride(head_dim), ko = kv->stride(off_dim), blocks = kv->size(0);
    const int32_t heads = static_cast<int32_t>(src->size(1));
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_scatter(src_p, st, sh_, kv_p, kb, kh, ko, blocks, slots_p, n, heads,
                   static_cast<int32_t>(two_d / 2), static_cast<int32_t>(block_size), code,
                   sh.cos, sh.sgn, static_cast<int32_t>(sh.rotary), scale, flags, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

PyObject* bind(PyObject*, PyObject* address) {
  void* p = PyLong_AsVoidPtr(address);
  if (p == nullptr) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "NULL function");
    return nullptr;
  }
  g_scatter = reinterpret_cast<scatter_fn>(p);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"scatter", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(scatter)), METH_FASTCALL,
     "mkv_scatter_shifted on torch tensors; None: take the general path"},
    {"bind", bind, METH_O, "the address of mkv_scatter_shifted"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "marathon_binding", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_marathon_binding() {
  s_delta = PyUnicode_InternFromString("delta");
  s_cos = PyUnicode_InternFromString("cos");
  s_sgn = PyUnicode_InternFromString("sgn");
  s_emb_cos = PyUnicode_InternFromString("emb_cos");
  s_rotary = PyUnicode_InternFromString("rotary");
  if (!s_delta || !s_cos || !s_sgn || !s_emb_cos || !s_rotary) return nullptr;
  // what it was compiled against; the loader compares them before it calls anything
  PyObject* m = PyModule_Create(&module);
  if (m == nullptr || PyModule_AddIntConstant(m, "abi", MKV_ABI_VERSION) != 0 ||
      PyModule_AddStringConstant(m, "torch", MARATHON_TORCH) != 0) {
    Py_XDECREF(m);
    return nullptr;
  }
  return m;
}
