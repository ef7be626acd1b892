// Native front of the calls that a projection makes, quantize(), gemm() and the Q/K and Q/K/V
// projections: the argument checks, the output allocation and the launches of a plain call, without the
// interpreter.
//
// Each function takes a call only if it can see that the Python front (hip.py) would accept it and
// launch at once: plain CUDA tensors, contiguous, of the right dtypes and shapes, no forced schedule.
// Anything else returns None, and the Python front handles the call and raises what it raises: no error
// is decided here.  The launches are the same C ABI calls, with the interpreter lock released.
//
// Measured on a [1, 256] activation: quantize 7.3 -> 4.6 us of host time, gemm 9.4 -> 4.4 us, of which
// the HIP launch takes about 3 each.  The projections' staged form, two launches, takes
// 18 to 20 us through Python and 8 to 10 us here; the fused one 10 to 13 and 5 to 6 us.
#include <Python.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <cmath>
#include <mutex>
#include <unordered_map>

#include "m5k.h"

namespace {

PyObject* g_stream_of = nullptr;  // torch's raw stream handle of a device index
PyObject* g_splits = nullptr;     // hip._native_splits(mode, m, n, k, device index) -> K ranges, 0: not here
PyObject* g_staged = nullptr;     // hip._native_staged(mode, m, n, k, device index, aligned, grouped) -> 0 or 1

enum Mode { INT8, FP8, B16, H16 };

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

// What hip.py's planner says of a shape, kept per shape and settings of the environment (bounded:
// emptied when full).  `what`: the mode, and for a projection's route bits 4 (a route), 5 (aligned
// operands) and 6 (grouped layout).
struct Key {
  int what, device, state;
  int64_t m, n, k;
  bool operator==(const Key& o) const {
    return what == o.what && device == o.device && state == o.state && m == o.m && n == o.n && k == o.k;
  }
};
struct Hash {
  size_t operator()(const Key& x) const {
    uint64_t h = 1469598103934665603ull;
    for (uint64_t v : {uint64_t(x.what), uint64_t(x.device), uint64_t(x.state), uint64_t(x.m), uint64_t(x.n), uint64_t(x.k)})
      h = (h ^ v) * 1099511628211ull, h ^= h >> 29;
    return h;
  }
};
std::mutex g_mutex;
std::unordered_map<Key, int, Hash> g_plans;

template <class Ask>
int planned(const Key& key, Ask ask) {  // -1: a Python error is set
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    const auto it = g_plans.find(key);
    if (it != g_plans.end()) return it->second;
  }
  PyObject* r = ask();
  if (!r) return -1;
  const long v = PyLong_AsLong(r);
  Py_DECREF(r);
  if (PyErr_Occurred()) return -1;
  std::lock_guard<std::mutex> lock(g_mutex);
  if (g_plans.size() >= 4096) g_plans.clear();
  g_plans[key] = static_cast<int>(v);
  return static_cast<int>(v);
}

// K ranges of an aligned INT8 or FP8 product.
int planned_splits(const Key& key, PyObject* mode) {
  return planned(key, [&] {
    return PyObject_CallFunction(g_splits, "OLLLi", mode, (long long)key.m, (long long)key.n, (long long)key.k, key.device);
  });
}

// Whether a projection runs as the GEMM and a postprocess.
int planned_staged(const Key& key, PyObject* mode, bool aligned, bool grouped) {
  return planned(key, [&] {
    return PyObject_CallFunction(g_staged, "OLLLiii", mode, (long long)key.m, (long long)key.n, (long long)key.k,
                                 key.device, int(aligned), int(grouped));
  });
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// gemm(a, b, mode, a_scales, b_scales, output_dtype, bias, bias_row_map, residual, gate, gate_row_map).
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 11 || !PyUnicode_Check(args[2])) Py_RETURN_NONE;
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
  if (quant && k % 16 == 0 && aligned16(ap) && aligned16(bp)) {
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

// The Q/K projection (args: a, b, gamma, cos, sin, mode, a_scales, b_scales, epsilon) and the grouped
// Q/K/V one (a, w, q_gamma, k_gamma, cos, sin, mode, a_scales, w_scales, epsilon), by the route that
// hip.projection_staged names.
constexpr int64_t HEAD = 128;

PyObject* project(PyObject* const* args, bool grouped) {
  const int at = grouped ? 4 : 3;  // index of cos
  PyObject* mo = args[at + 2];
  if (!PyUnicode_Check(mo)) Py_RETURN_NONE;
  const bool i8 = PyUnicode_CompareWithASCIIString(mo, "int8") == 0;
  if (!i8 && PyUnicode_CompareWithASCIIString(mo, "bf16") != 0) Py_RETURN_NONE;
  const at::Tensor *a = plain(args[0]), *b = plain(args[1]);
  const at::ScalarType operand = i8 ? at::kChar : at::kBFloat16;
  if (!a || !b || a->dim() != 2 || b->dim() != 2 || a->scalar_type() != operand || b->scalar_type() != operand ||
      a->device() != b->device())
    Py_RETURN_NONE;
  const c10::Device dev = a->device();
  const int64_t m = a->size(0), k = a->size(1), n = b->size(0), block = grouped ? 3 * HEAD : HEAD;
  if (b->size(1) != k || m == 0 || n == 0 || k == 0 || n % block || (i8 && k > 131071)) Py_RETURN_NONE;
  const float *sa = nullptr, *sb = nullptr;
  if (i8) {
    const at::Tensor *ta = plain(args[at + 3]), *tb = plain(args[at + 4]);
    if (!vector_of(ta, m, at::kFloat, dev) || !vector_of(tb, n, at::kFloat, dev)) Py_RETURN_NONE;
    sa = static_cast<const float*>(ta->data_ptr());
    sb = static_cast<const float*>(tb->data_ptr());
  } else if (args[at + 3] != Py_None || args[at + 4] != Py_None) {
    Py_RETURN_NONE;
  }
  const at::Tensor *g = plain(args[2]), *gk = grouped ? plain(args[3]) : g;
  const at::Tensor *cos = plain(args[at]), *sin = plain(args[at + 1]);
  if (!vector_of(g, HEAD, at::kBFloat16, dev) || !vector_of(gk, HEAD, at::kBFloat16, dev) || !aligned16(g->data_ptr()) ||
      !aligned16(gk->data_ptr()))
    Py_RETURN_NONE;
  for (const at::Tensor* t : {cos, sin})
    if (!t || t->dim() != 2 || t->size(0) != m || t->scalar_type() != at::kBFloat16 || t->device() != dev) Py_RETURN_NONE;
  const int64_t half = cos->size(1);
  if (half < 1 || half > HEAD / 2 || sin->size(1) != half) Py_RETURN_NONE;
  if (!PyFloat_CheckExact(args[at + 5])) Py_RETURN_NONE;
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(args[at + 5]));
  if (!(eps > 0.0f) || !std::isfinite(eps)) Py_RETURN_NONE;
  const int state = m5k_gemm_schedule_state();
  if (state & 0xF) Py_RETURN_NONE;  // a schedule is forced
  const void *ap = a->data_ptr(), *bp = b->data_ptr();
  const int64_t row = k * (i8 ? 1 : 2);
  const bool whole = row % 16 == 0 && aligned16(ap) && aligned16(bp), aligned = whole && row <= int64_t(1) << 23;
  const int mode = i8 ? INT8 : B16;
  const int staged = planned_staged(Key{mode | 16 | (aligned ? 32 : 0) | (grouped ? 64 : 0), dev.index(), state, m, n, k},
                                    mo, aligned, grouped);
  if (staged < 0) return nullptr;
  int splits = 1;
  if (staged && i8 && whole) {
    splits = planned_splits(Key{mode, dev.index(), state, m, n, k}, mo);
    if (splits < 0) return nullptr;
    if (splits == 0) Py_RETURN_NONE;
  }
  void* stream = nullptr;
  if (!stream_of(dev, &stream)) return nullptr;
  const int64_t heads = n / block;
  at::Tensor y[3], projected, workspace;
  for (int i = 0; i < (grouped ? 3 : 1); ++i) y[i] = empty({heads, m, HEAD}, at::kBFloat16, dev);
  if (staged) projected = empty({m, n}, at::kBFloat16, dev);
  if (splits > 1) workspace = empty({splits, m, n}, at::kInt, dev);
  void* yp[3] = {y[0].data_ptr(), grouped ? y[1].data_ptr() : nullptr, grouped ? y[2].data_ptr() : nullptr};
  void* pp = staged ? projected.data_ptr() : nullptr;
  auto* wp = splits > 1 ? static_cast<int32_t*>(workspace.data_ptr()) : nullptr;
  const void *gp = g->data_ptr(), *gkp = gk->data_ptr(), *cp = cos->data_ptr(), *sp = sin->data_ptr();
  auto* ai = static_cast<const int8_t*>(ap);
  auto* bi = static_cast<const int8_t*>(bp);
  const int r = static_cast<int>(half), dtype = i8 ? M5K_I8 : M5K_BF16;
  const char* name = nullptr;
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS
  if (staged) {
    if (splits > 1) {
      name = "m5k_gemm_i8_splitk";
      rc = m5k_gemm_i8_splitk(ai, bi, m, n, k, sa, sb, pp, M5K_BF16, nullptr, nullptr, nullptr, nullptr, nullptr, splits,
                              wp, splits * m * n, stream);
    } else if (i8) {
      name = "m5k_gemm_i8";
      rc = m5k_gemm_i8(ai, bi, m, n, k, sa, sb, pp, M5K_BF16, nullptr, nullptr, nullptr, nullptr, nullptr, stream);
    } else {
      name = "m5k_gemm_float";
      rc = m5k_gemm_float(ap, bp, M5K_BF16, m, n, k, pp, M5K_BF16, nullptr, nullptr, nullptr, stream);
    }
    if (rc == 0 && grouped) {
      name = "m5k_qkv_norm_rope";
      rc = m5k_qkv_norm_rope(pp, m, heads, gp, gkp, cp, sp, r, eps, yp[0], yp[1], yp[2], stream);
    } else if (rc == 0) {
      name = "m5k_qk_norm_rope";
      rc = m5k_qk_norm_rope(pp, m, n, gp, cp, sp, r, eps, yp[0], stream);
    }
  } else if (grouped) {
    name = "m5k_projection_qkv_rope";
    rc = m5k_projection_qkv_rope(ap, bp, dtype, m, heads, k, sa, sb, gp, gkp, cp, sp, r, eps, yp[0], yp[1], yp[2], stream);
  } else {
    name = "m5k_projection_qk_rope";
    rc = m5k_projection_qk_rope(ap, bp, dtype, m, n, k, sa, sb, gp, cp, sp, r, eps, yp[0], stream);
  }
  Py_END_ALLOW_THREADS
  if (rc) return failed(name, rc);
  if (!grouped) return THPVariable_Wrap(std::move(y[0]));
  PyObject* out = PyTuple_New(3);
  for (int i = 0; out && i < 3; ++i) {
    PyObject* o = THPVariable_Wrap(std::move(y[i]));
    if (!o) {
      Py_CLEAR(out);
      break;
    }
    PyTuple_SET_ITEM(out, i, o);
  }
  return out;
}

PyObject* qk(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 9) Py_RETURN_NONE;
  return project(args, false);
  END_HANDLE_TH_ERRORS
}

PyObject* qkv(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 10) Py_RETURN_NONE;
  return project(args, true);
  END_HANDLE_TH_ERRORS
}

// bind(stream_of, splits, staged): the Python callables above.
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *s, *p, *q;
  if (!PyArg_ParseTuple(args, "OOO", &s, &p, &q)) return nullptr;
  PyObject** slots[] = {&g_stream_of, &g_splits, &g_staged};
  PyObject* given[] = {s, p, q};
  for (int i = 0; i < 3; ++i) {
    Py_INCREF(given[i]);
    Py_XDECREF(*slots[i]);
    *slots[i] = given[i];
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"quantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(quantize)), METH_FASTCALL, nullptr},
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gemm)), METH_FASTCALL, nullptr},
    {"qk", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(qk)), METH_FASTCALL, nullptr},
    {"qkv", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(qkv)), METH_FASTCALL, nullptr},
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
