// Native front of the two calls that every quantized linear makes, quantize() and gemm(): the
// argument checks, the output allocation and the launch of a plain call, without the interpreter.
//
// Each function takes a call only if it can see that the Python front (hip.py) would accept it and
// launch at once: plain CUDA tensors, contiguous, of the right dtypes and shapes, no forced schedule.
// Anything else returns None, and the Python front handles the call and raises what it raises: no error
// is decided here.  The launches are the same C ABI calls, with the interpreter lock released.
//
// Measured on a [1, 256] activation: quantize 7.3 -> 4.6 us of host time, gemm 9.4 -> 4.4 us, of which
// the HIP launch takes about 3 each.
#include <Python.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <mutex>
#include <unordered_map>

#include "m5k.h"

namespace {

PyObject* g_stream_of = nullptr;  // torch's raw stream handle of a device index
PyObject* g_splits = nullptr;     // hip._native_splits(mode, m, n, k, device index) -> K ranges, 0: not here

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return M5K_F32;
    case at::kHalf: return M5K_F16;
    case at::kBFloat16: return M5K_BF16;
    default: return -1;
  }
}

// A tensor whose storage a kernel may read as it is: exactly torch.Tensor (or Parameter), strided and
// contiguous on a GPU, and not a wrapper of a transform (vmap, forward or reverse mode of torch.func).
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  const c10::DispatchKeySet keys = t.key_set();
  if (!t.is_cuda() || t.layout() != at::kStrided ||
      keys.has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                        c10::DispatchKey::Functionalize, c10::DispatchKey::Python,
                                        c10::DispatchKey::Conjugate, c10::DispatchKey::Negative})) ||
      !t.has_storage() || !t.is_contiguous())
    return nullptr;
  return &t;
}

bool vector_of(const at::Tensor* t, int64_t n, at::ScalarType st, c10::Device d) {
  return t && t->dim() == 1 && t->size(0) == n && t->scalar_type() == st && t->device() == d;
}

bool stream_of(c10::Device d, void** out) {
  PyObject* index = PyLong_FromLong(d.index());
  if (!index) return false;
  PyObject* r = PyObject_CallOneArg(g_stream_of, index);
  Py_DECREF(index);
  if (!r) return false;
  *out = reinterpret_cast<void*>(PyLong_AsUnsignedLongLong(r));
  Py_DECREF(r);
  return !PyErr_Occurred();
}

at::Tensor empty(at::IntArrayRef shape, at::ScalarType st, c10::Device d) {
  return at::empty(shape, at::TensorOptions().dtype(st).device(d));
}

PyObject* failed(const char* name, int rc) {
  PyErr_Format(PyExc_RuntimeError, "%s failed (%d): %s", name, rc, m5k_last_error());
  return nullptr;
}

// quantize(x, mode): codes and scales of mode "int8" or "fp8".
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 2 || !PyUnicode_Check(args[1])) Py_RETURN_NONE;
  const bool i8 = PyUnicode_CompareWithASCIIString(args[1], "int8") == 0;
  if (!i8 && PyUnicode_CompareWithASCIIString(args[1], "fp8") != 0) Py_RETURN_NONE;
  const at::Tensor* x = plain(args[0]);
  if (!x || x->dim() != 2 || x->size(0) == 0 || x->size(1) == 0) Py_RETURN_NONE;
  const int code = dtype_code(x->scalar_type());
  if (code < 0) Py_RETURN_NONE;
  void* stream = nullptr;
  if (!stream_of(x->device(), &stream)) return nullptr;
  const int64_t rows = x->size(0), k = x->size(1);
  at::Tensor q = empty({rows, k}, i8 ? at::kChar : at::kByte, x->device());
  at::Tensor s = empty({rows}, at::kFloat, x->device());
  const void* xp = x->data_ptr();
  void* qp = q.data_ptr();
  float* sp = static_cast<float*>(s.data_ptr());
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = m5k_quantize_rows(xp, code, rows, k, i8 ? M5K_QUANT_INT8 : M5K_QUANT_FP8, qp, sp, stream);
  Py_END_ALLOW_THREADS
  if (rc) return failed("m5k_quantize_rows", rc);
  PyObject* qo = THPVariable_Wrap(std::move(q));
  PyObject* so = THPVariable_Wrap(std::move(s));
  PyObject* r = qo && so ? PyTuple_Pack(2, qo, so) : nullptr;
  Py_XDECREF(qo);
  Py_XDECREF(so);
  return r;
  END_HANDLE_TH_ERRORS
}

// K ranges of an aligned INT8 or FP8 product, from hip.py's planner, kept per shape and settings of
// the environment (bounded: emptied when full).
struct Key {
  int mode, device, state;
  int64_t m, n, k;
  bool operator==(const Key& o) const {
    return mode == o.mode && device == o.device && state == o.state && m == o.m && n == o.n && k == o.k;
  }
};
struct Hash {
  size_t operator()(const Key& x) const {
    uint64_t h = 1469598103934665603ull;
    for (uint64_t v : {uint64_t(x.mode), uint64_t(x.device), uint64_t(x.state), uint64_t(x.m), uint64_t(x.n), uint64_t(x.k)})
      h = (h ^ v) * 1099511628211ull, h ^= h >> 29;
    return h;
  }
};
std::mutex g_mutex;
std::unordered_map<Key, int, Hash> g_plans;

int planned_splits(const Key& key, PyObject* mode) {  // -1: a Python error is set
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    const auto it = g_plans.find(key);
    if (it != g_plans.end()) return it->second;
  }
  PyObject* r = PyObject_CallFunction(g_splits, "OLLLi", mode, (long long)key.m, (long long)key.n, (long long)key.k,
                                      key.device);
  if (!r) return -1;
  const long v = PyLong_AsLong(r);
  Py_DECREF(r);
  if (PyErr_Occurred()) return -1;
  std::lock_guard<std::mutex> lock(g_mutex);
  if (g_plans.size() >= 4096) g_plans.clear();
  g_plans[key] = static_cast<int>(v);
  return static_cast<int>(v);
}

// gemm(a, b, mode, a_scales, b_scales, output_dtype, bias, bias_row_map, residual, gate, gate_row_map).
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 11 || !PyUnicode_Check(args[2])) Py_RETURN_NONE;
  enum { INT8, FP8, B16, H16 };
  PyObject* mo = args[2];
  const int mode = PyUnicode_CompareWithASCIIString(mo, "int8") == 0   ? INT8
                   : PyUnicode_CompareWithASCIIString(mo, "bf16") == 0 ? B16
                   : PyUnicode_CompareWithASCIIString(mo, "fp8") == 0  ? FP8
                   : PyUnicode_CompareWithASCIIString(mo, "fp16") == 0 ? H16
                                                                       : -1;
  if (mode < 0) Py_RETURN_NONE;
  const bool quant = mode == INT8 || mode == FP8;
  static const at::ScalarType operand[] = {at::kChar, at::kByte, at::kBFloat16, at::kHalf};
  const at::Tensor *a = plain(args[0]), *b = plain(args[1]);
  if (!a || !b || a->dim() != 2 || b->dim() != 2 || a->scalar_type() != operand[mode] ||
      b->scalar_type() != operand[mode] || a->device() != b->device())
    Py_RETURN_NONE;
  const c10::Device dev = a->device();
  const int64_t m = a->size(0), k = a->size(1), n = b->size(0);
  if (b->size(1) != k || m == 0 || n == 0 || k == 0 || (mode == FP8 && k % 128) || (mode == INT8 && k > 133144))
    Py_RETURN_NONE;
  const float *sa = nullptr, *sb = nullptr;
  if (quant) {
    const at::Tensor *ta = plain(args[3]), *tb = plain(args[4]);
    if (!vector_of(ta, m, at::kFloat, dev) || !vector_of(tb, n, at::kFloat, dev)) Py_RETURN_NONE;
    sa = static_cast<const float*>(ta->data_ptr());
    sb = static_cast<const float*>(tb->data_ptr());
  } else if (args[3] != Py_None || args[4] != Py_None) {
    Py_RETURN_NONE;
  }
  at::ScalarType out = at::kFloat;
  if (args[5] != Py_None) {
    if (!THPDtype_Check(args[5])) Py_RETURN_NONE;
    out = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
  }
  const int out_code = dtype_code(out);
  if (out_code < 0) Py_RETURN_NONE;
  // A table (bias or gate): [n], or [P, n] with an int32 map of the m rows.
  auto table = [&](PyObject* to, PyObject* ro, at::ScalarType st, const void** tp, const int32_t** rp) {
    const at::Tensor* t = plain(to);
    if (!t || t->scalar_type() != st || t->device() != dev) return false;
    if (ro == Py_None) {
      if (t->dim() != 1 || t->size(0) != n) return false;
    } else {
      const at::Tensor* r = plain(ro);
      if (t->dim() != 2 || t->size(0) == 0 || t->size(1) != n || !vector_of(r, m, at::kInt, dev)) return false;
      *rp = static_cast<const int32_t*>(r->data_ptr());
    }
    *tp = t->data_ptr();
    return true;
  };
  const void *bias = nullptr, *residual = nullptr, *gate = nullptr;
  const int32_t *bias_map = nullptr, *gate_map = nullptr;
  if (args[6] != Py_None || args[7] != Py_None) {
    if (mode != INT8 || args[6] == Py_None || args[8] != Py_None || args[9] != Py_None || args[10] != Py_None ||
        !table(args[6], args[7], at::kFloat, &bias, &bias_map))
      Py_RETURN_NONE;
  } else if (args[8] != Py_None || args[9] != Py_None || args[10] != Py_None) {
    const at::Tensor* r = plain(args[8]);
    if ((mode != INT8 && mode != B16) || args[5] == Py_None || out != at::kBFloat16 || !r || r->dim() != 2 ||
        r->size(0) != m || r->size(1) != n || r->scalar_type() != at::kBFloat16 || r->device() != dev ||
        !table(args[9], args[10], at::kBFloat16, &gate, &gate_map))
      Py_RETURN_NONE;
    residual = r->data_ptr();
  }
  const int state = m5k_gemm_schedule_state();
  if (state & 0xF) Py_RETURN_NONE;  // a schedule is forced
  const void *ap = a->data_ptr(), *bp = b->data_ptr();
  int splits = 1;
  if (quant && k % 16 == 0 && ((reinterpret_cast<uintptr_t>(ap) | reinterpret_cast<uintptr_t>(bp)) & 15u) == 0) {
    splits = planned_splits(Key{mode, dev.index(), state, m, n, k}, mo);
    if (splits < 0) return nullptr;
    if (splits == 0) Py_RETURN_NONE;
  }
  void* stream = nullptr;
  if (!stream_of(dev, &stream)) return nullptr;
  at::Tensor c = empty({m, n}, out, dev), workspace;
  if (splits > 1) workspace = empty({splits, m, n}, mode == INT8 ? at::kInt : at::kFloat, dev);
  void* cp = c.data_ptr();
  void* wp = splits > 1 ? workspace.data_ptr() : nullptr;
  const int64_t elems = splits * m * n;
  const char* name = nullptr;
  int rc = 0;
  auto* ai = static_cast<const int8_t*>(ap);
  auto* bi = static_cast<const int8_t*>(bp);
  auto* au = static_cast<const uint8_t*>(ap);
  auto* bu = static_cast<const uint8_t*>(bp);
  auto* fbias = static_cast<const float*>(bias);
  Py_BEGIN_ALLOW_THREADS
  if (mode == INT8 && splits > 1) {
    name = "m5k_gemm_i8_splitk";
    rc = m5k_gemm_i8_splitk(ai, bi, m, n, k, sa, sb, cp, out_code, fbias, bias_map, residual, gate, gate_map, splits,
                            static_cast<int32_t*>(wp), elems, stream);
  } else if (mode == INT8) {
    name = "m5k_gemm_i8";
    rc = m5k_gemm_i8(ai, bi, m, n, k, sa, sb, cp, out_code, fbias, bias_map, residual, gate, gate_map, stream);
  } else if (mode == FP8 && splits > 1) {
    name = "m5k_gemm_f8_splitk";
    rc = m5k_gemm_f8_splitk(au, bu, m, n, k, sa, sb, cp, out_code, splits, static_cast<float*>(wp), elems, stream);
  } else if (mode == FP8) {
    name = "m5k_gemm_f8";
    rc = m5k_gemm_f8(au, bu, m, n, k, sa, sb, cp, out_code, stream);
  } else {
    name = "m5k_gemm_float";
    rc = m5k_gemm_float(ap, bp, mode == B16 ? M5K_BF16 : M5K_F16, m, n, k, cp, out_code, residual, gate, gate_map, stream);
  }
  Py_END_ALLOW_THREADS
  if (rc) return failed(name, rc);
  return THPVariable_Wrap(std::move(c));
  END_HANDLE_TH_ERRORS
}

// bind(stream_of, splits): the Python callables above.
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *s, *p;
  if (!PyArg_ParseTuple(args, "OO", &s, &p)) return nullptr;
  Py_INCREF(s);
  Py_INCREF(p);
  Py_XDECREF(g_stream_of);
  Py_XDECREF(g_splits);
  g_stream_of = s;
  g_splits = p;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"quantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(quantize)), METH_FASTCALL, nullptr},
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gemm)), METH_FASTCALL, nullptr},
    {"bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "m5k_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// abi_version and torch_version: what this file was compiled for, compared before the first call
// (_lib.load_fast).
PyMODINIT_FUNC PyInit_m5k_fast() {
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && (PyModule_AddIntConstant(m, "abi_version", M5K_ABI_VERSION) != 0 ||
                       PyModule_AddStringConstant(m, "torch_version", M5K_TORCH_VERSION) != 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
