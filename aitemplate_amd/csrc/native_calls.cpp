// The common case of the eager calls and of Model.run_with_tensors, without the interpreter.
//
// A call of a few microseconds on the GPU used to spend 12 to 16 us in Python: a dozen tensor attribute reads, their
// comparisons, reshapes and some twenty ctypes argument conversions per launch (linear layer of one row, 768 x 768:
// 14.2 us a call, 3.6 us of it on the GPU; a compiled block of five kernels 71 us, 43 of them on the GPU; 4.0 and 54 us
// with this module).  These
// functions read the same attributes from the C++ tensors, allocate the result and call the same C ABI.
//
// They take ordinary arguments only: plain GPU tensors of one type whose shapes fit and whose rows are contiguous, and
// outside of torch's modes.  For anything else they return NotImplemented without having done anything, and the caller's
// Python path, which handles the remaining cases and words the errors, takes the call.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/headeronly/version.h>

#include <ATen/Context.h>
#include <ATen/core/DimVector.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>

#include <cmath>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "../../include/aitemplate_amd_kernels.h"
#include "../../include/model_interface.h"
#include "native_device.h"

// torch's own version string, pre-release part and all (the Makefile reads it from torch/version.py)
#ifndef AITAMD_TORCH_BUILD
#define AITAMD_TORCH_BUILD TORCH_VERSION
#endif

namespace {

struct OpInfo {
  const char* name;
  int epilogue;
  int residuals;
};
// the reference's op names, as _kernels.EPILOGUE_OF_OP has them
const OpInfo kOps[] = {
    {"gemm_rcr", AITAMD_EPI_NONE, 0},
    {"gemm_rcr_bias", AITAMD_EPI_BIAS, 0},
    {"gemm_rcr_bias_relu", AITAMD_EPI_BIAS_RELU, 0},
    {"gemm_rcr_bias_gelu", AITAMD_EPI_BIAS_GELU, 0},
    {"gemm_rcr_bias_fast_gelu", AITAMD_EPI_BIAS_GELU, 0},
    {"gemm_rcr_bias_add", AITAMD_EPI_BIAS_ADD, 1},
    {"gemm_rcr_bias_add_add", AITAMD_EPI_BIAS_ADD_ADD, 2},
    {"gemm_rcr_bias_add_relu", AITAMD_EPI_BIAS_ADD_RELU, 1},
    {"gemm_rcr_bias_add_add_relu", AITAMD_EPI_BIAS_ADD_ADD_RELU, 2},
    {"gemm_rcr_bias_sigmoid", AITAMD_EPI_BIAS_SIGMOID, 0},
    {"gemm_rcr_bias_tanh", AITAMD_EPI_BIAS_TANH, 0},
    {"gemm_rcr_bias_swish", AITAMD_EPI_BIAS_SWISH, 0},
    {"gemm_rcr_bias_hardswish", AITAMD_EPI_BIAS_HARDSWISH, 0},
    {"gemm_rcr_bias_mul", AITAMD_EPI_BIAS_MUL, 1},
    {"gemm_rcr_bias_mul_add", AITAMD_EPI_BIAS_MUL_ADD, 2},
    {"gemm_rcr_bias_sigmoid_mul", AITAMD_EPI_BIAS_SIGMOID_MUL, 1},
    {"gemm_rcr_bias_sigmoid_mul_tanh", AITAMD_EPI_BIAS_SIGMOID_MUL_TANH, 1},
    {"gemm_rcr_bias_mul_tanh", AITAMD_EPI_BIAS_MUL_TANH, 1},
};

PyObject* not_ordinary() { Py_RETURN_NOTIMPLEMENTED; }

// A plain tensor on the GPU, or null (also for None and for subclasses, which may intercept what is done to them).
// The wrappers of torch.func and of functionalization are of the exact type torch.Tensor and report the device of what
// they wrap, but have no memory of their own.
const at::Tensor* gpu_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet wrappers(
      {c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper});
  return on_device(t) && t.layout() == at::kStrided && t.has_storage() && !t.key_set().has_any(wrappers) ? &t : nullptr;
}

int dtype_id(const at::Tensor& t) {
  const at::ScalarType s = t.scalar_type();
  return s == at::kHalf ? 0 : (s == at::kBFloat16 ? 1 : -1);
}

// The class of the function mode behind `with torch.device(...)` and torch.set_default_device (null where torch has none)
PyTypeObject* device_context_type() {
  // (not an initializer of the static: the import may give up the interpreter lock, and others would wait with it held)
  static PyTypeObject* type = nullptr;
  if (type == nullptr) {
    THPObjectPtr from(PyImport_ImportModule("torch.utils._device"));
    PyObject* found = from ? PyObject_GetAttrString(from, "DeviceContext") : nullptr;
    if (found == nullptr)
      PyErr_Clear();
    else if (type == nullptr && PyType_Check(found))
      type = reinterpret_cast<PyTypeObject*>(found);  // (kept for good)
    else
      Py_DECREF(found);
  }
  return type;
}

// Whether every function mode gives new tensors a default device and no more: what is allocated here names its device
bool device_contexts_only() {
  for (int64_t i = at::impl::PythonTorchFunctionTLS::stack_len(); i-- > 0;)
    if (Py_TYPE(at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter())) != device_context_type()) return false;
  return true;
}

// False under a mode that sees, changes, records or refuses what the Python path does through torch (its allocation,
// reshapes and views): dispatch modes, fake tensors among them, function modes other than those of a default device,
// torch.func transforms, functionalization, tracing.  All but the function modes put a key of theirs into the thread's
// dispatch keys; autocast, no_grad and inference mode put none.
bool ordinary_context() {
  return (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() && device_contexts_only();
}

// results of torch.empty that torch would have to fill are not ordinary
bool plain_allocation() {
  return !(at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory());
}

// Row pitch of a [rows, cols] view with contiguous rows; false where the rows are not contiguous.
bool row_pitch(const at::Tensor& t, int64_t* pitch) {
  const int64_t rows = t.size(0), cols = t.size(1);
  if (cols > 1 && t.stride(1) != 1) return false;
  *pitch = rows > 1 ? t.stride(0) : std::max(cols, t.stride(0));
  return true;
}

// The same for an operand whose leading dims are flattened into `rows`.
bool flat_row_pitch(const at::Tensor& t, int64_t rows, int64_t cols, int64_t* pitch) {
  if (t.dim() == 2 && t.size(0) == rows && t.size(1) == cols) return row_pitch(t, pitch);
  if (!t.is_contiguous() || t.numel() != rows * cols) return false;
  *pitch = cols;
  return true;
}

PyObject* finish(int rc, const char* what, const at::Tensor* made, PyObject* out) {
  if (rc != 0) return PyErr_Format(PyExc_RuntimeError, "%s failed: %s", what, aitamd_last_error());
  if (made != nullptr) return THPVariable_Wrap(*made);
  Py_INCREF(out);
  return out;
}

// torch's own translation of C++ exceptions: the types and texts that its bindings raise
template <class F>
PyObject* guarded(F&& body) {
  HANDLE_TH_ERRORS
  return ordinary_context() ? body() : not_ordinary();
  END_HANDLE_TH_ERRORS
}

// The launch itself runs without the interpreter lock, as it does through ctypes.  What it takes is plain pointers and
// numbers, read beforehand: a tensor's accessors may throw, and the error is raised with the lock held.
struct Unlocked {
  PyThreadState* const save = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(save); }
};
template <class F>
int unlocked(F&& launch) {
  const Unlocked here;
  return launch();
}

const void* pointer(const at::Tensor* t) { return t == nullptr ? nullptr : t->data_ptr(); }

// gemm(op, a, b, bias, d0, d1, out, algo, workspace)
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    if (nargs != 9 || !PyUnicode_Check(args[0]) || !PyLong_CheckExact(args[7])) return not_ordinary();
    const char* op = PyUnicode_AsUTF8(args[0]);
    if (op == nullptr) {  // (a lone surrogate)
      PyErr_Clear();
      return not_ordinary();
    }
    const OpInfo* info = nullptr;
    for (const OpInfo& o : kOps)
      if (strcmp(o.name, op) == 0) info = &o;
    if (info == nullptr) return not_ordinary();
    const at::Tensor *a = gpu_tensor(args[1]), *b = gpu_tensor(args[2]);
    if (a == nullptr || b == nullptr || a->dim() < 1 || b->dim() != 2) return not_ordinary();
    const int dt = dtype_id(*a);
    const int64_t K = a->size(-1), N = b->size(0);
    if (dt < 0 || b->scalar_type() != a->scalar_type() || b->size(1) != K || a->numel() == 0 || N == 0) return not_ordinary();
    const int64_t M = a->numel() / K;
    int64_t lda, ldb, ldc = N, ldd = N;
    if (!flat_row_pitch(*a, M, K, &lda) || !row_pitch(*b, &ldb)) return not_ordinary();
    const at::Tensor* opt[3] = {};  // bias, d0, d1
    for (int i = 0; i < 3; ++i) {
      if (args[3 + i] == Py_None) continue;
      opt[i] = gpu_tensor(args[3 + i]);
      if (opt[i] == nullptr || opt[i]->scalar_type() != a->scalar_type()) return not_ordinary();
    }
    if (info->epilogue != AITAMD_EPI_NONE && (opt[0] == nullptr || opt[0]->numel() != N || !opt[0]->is_contiguous()))
      return not_ordinary();
    for (int i = 0; i < 2; ++i) {
      int64_t pitch;
      if (i >= info->residuals) {
        if (opt[1 + i] != nullptr) return not_ordinary();
        continue;
      }
      if (opt[1 + i] == nullptr || !flat_row_pitch(*opt[1 + i], M, N, &pitch) || (i == 1 && pitch != ldd)) return not_ordinary();
      ldd = pitch;
    }
    void* ws = nullptr;
    int64_t ws_bytes = 0;
    if (args[8] != Py_None) {
      const at::Tensor* w = gpu_tensor(args[8]);
      if (w == nullptr || w->scalar_type() != at::kByte || !w->is_contiguous()) return not_ordinary();
      ws = w->data_ptr();
      ws_bytes = w->numel();
    }
    at::Tensor made;
    void* c;
    if (args[6] == Py_None) {
      if (!plain_allocation()) return not_ordinary();
      c10::SmallVector<int64_t, 6> sizes(a->sizes().begin(), a->sizes().end());
      sizes.back() = N;
      made = empty_like_device(sizes, *a);
      c = made.data_ptr();
    } else {
      const at::Tensor* out = gpu_tensor(args[6]);
      if (out == nullptr || out->scalar_type() != a->scalar_type()) return not_ordinary();
      if (out->dim() == 2 && out->size(0) == M && out->size(1) == N && out->stride(1) == 1 && out->stride(0) >= N) {
        if (!row_pitch(*out, &ldc)) return not_ordinary();
      } else if (!out->is_contiguous() || out->numel() != M * N) {
        return not_ordinary();
      }
      c = out->data_ptr();
    }
    const int algo = (int)PyLong_AsLong(args[7]);
    if (algo == -1 && PyErr_Occurred()) return nullptr;
    const void *pa = pointer(a), *pb = pointer(b), *bias = pointer(opt[0]), *d0 = pointer(opt[1]), *d1 = pointer(opt[2]);
    void* stream = current_stream();
    const int rc = unlocked([&] {
      return aitamd_gemm_rcr_ws(info->epilogue, dt, algo, pa, pb, bias, d0, d1, c, M, N, K, lda, ldb, ldc, ldd, ws, ws_bytes,
                                stream);
    });
    return finish(rc, info->name, made.defined() ? &made : nullptr, args[6]);
  });
}

// bmm(layout, a, b, out, d1, algo, what): layout is the C ABI's operand layout, `what` names the op in errors
PyObject* bmm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    if (nargs != 7 || !PyLong_CheckExact(args[0]) || !PyLong_CheckExact(args[4]) || !PyLong_CheckExact(args[5]))
      return not_ordinary();
    const int layout = (int)PyLong_AsLong(args[0]);
    const int64_t d1 = PyLong_AsLongLong(args[4]);
    const int algo = (int)PyLong_AsLong(args[5]);
    if (PyErr_Occurred()) return nullptr;
    const at::Tensor *a = gpu_tensor(args[1]), *b = gpu_tensor(args[2]);
    if (a == nullptr || b == nullptr || a->dim() < 2 || a->dim() > 3 || b->dim() < 2 || b->dim() > 3) return not_ordinary();
    const int dt = dtype_id(*a);
    if (dt < 0 || b->scalar_type() != a->scalar_type() || !a->is_contiguous() || !b->is_contiguous()) return not_ordinary();
    const int64_t ba = a->dim() == 3 ? a->size(0) : 1, bb = b->dim() == 3 ? b->size(0) : 1;
    const int64_t B = std::max(ba, bb);
    if ((ba != 1 && ba != B) || (bb != 1 && bb != B)) return not_ordinary();
    const int64_t M = a->size((layout & 2) ? -1 : -2), K = a->size((layout & 2) ? -2 : -1);
    const int64_t N = b->size((layout & 1) ? -1 : -2), Kb = b->size((layout & 1) ? -2 : -1);
    if (Kb != K || B * M * N == 0 || d1 < 0 || (d1 > 0 && B % d1 != 0)) return not_ordinary();
    at::Tensor made;
    void* c;
    if (args[3] == Py_None) {
      if (!plain_allocation()) return not_ordinary();
      made = d1 > 0 ? empty_like_device({B / d1, M, d1, N}, *a) : empty_like_device({B, M, N}, *a);
      c = made.data_ptr();
    } else {
      const at::Tensor* out = gpu_tensor(args[3]);
      if (out == nullptr || out->scalar_type() != a->scalar_type() || !out->is_contiguous() || out->numel() != B * M * N)
        return not_ordinary();
      c = out->data_ptr();
    }
    const int64_t sa = ba == 1 && B > 1 ? 0 : M * K, sb = bb == 1 && B > 1 ? 0 : N * K;
    const int64_t lda = a->size(-1), ldb = b->size(-1);
    const void *pa = pointer(a), *pb = pointer(b);
    void* stream = current_stream();
    const int rc = unlocked([&] {
      return aitamd_bmm(layout, dt, algo, pa, pb, c, B, M, N, K, lda, ldb, N, sa, sb, M * N, d1, stream);
    });
    return finish(rc, PyUnicode_AsUTF8(args[6]), made.defined() ? &made : nullptr, args[3]);
  });
}

// operands of an attention call: contiguous, of one type, `dims` dims; the type id or -1
int attention_operands(PyObject* const* args, int64_t dims, const at::Tensor** t) {
  for (int i = 0; i < 3; ++i) {
    t[i] = gpu_tensor(args[i]);
    if (t[i] == nullptr || t[i]->dim() != dims || !t[i]->is_contiguous() || t[i]->numel() == 0) return -1;
    if (t[i]->scalar_type() != t[0]->scalar_type()) return -1;
  }
  return dtype_id(*t[0]);
}

// the result tensor: a new one of `sizes`, or the caller's; null where it is not ordinary
void* attention_out(PyObject* out_arg, at::IntArrayRef sizes, const at::Tensor& like, at::Tensor* made) {
  if (out_arg == Py_None) {
    if (!plain_allocation()) return nullptr;
    *made = empty_like_device(sizes, like);
    return made->data_ptr();
  }
  const at::Tensor* out = gpu_tensor(out_arg);
  if (out == nullptr || out->scalar_type() != like.scalar_type() || !out->is_contiguous() ||
      out->numel() != c10::multiply_integers(sizes))
    return nullptr;
  return out->data_ptr();
}

// bmm_softmax_bmm_permute(q, k, v, heads, scale, causal, out)
PyObject* bmm_softmax_bmm_permute(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    const at::Tensor* t[3];
    if (nargs != 7 || !PyLong_CheckExact(args[3]) || !PyFloat_CheckExact(args[4]) || !PyBool_Check(args[5])) return not_ordinary();
    const int dt = attention_operands(args, 3, t);
    if (dt < 0) return not_ordinary();
    const int64_t B = t[0]->size(0), M = t[0]->size(1), K = t[0]->size(2), N = t[2]->size(1), O = t[2]->size(2);
    const int64_t G = PyLong_AsLongLong(args[3]);
    // (raised here: the Python path would pass on what is left of it in 64 bits)
    if (G == -1 && PyErr_Occurred()) return nullptr;
    if (t[1]->size(0) != B || t[1]->size(1) != N || t[1]->size(2) != K || t[2]->size(0) != B || G <= 0 || B % G != 0)
      return not_ordinary();
    at::Tensor made;
    void* out = attention_out(args[6], {B / G, M, G, O}, *t[0], &made);
    if (out == nullptr) return not_ordinary();
    const float scale = (float)PyFloat_AS_DOUBLE(args[4]);
    const int causal = args[5] == Py_True;
    const void *q = pointer(t[0]), *k = pointer(t[1]), *v = pointer(t[2]);
    void* stream = current_stream();
    const int rc = unlocked([&] {
      return aitamd_bmm_softmax_bmm_permute(dt, q, k, v, out, B, M, N, K, O, G, scale, causal, stream);
    });
    return finish(rc, "bmm_softmax_bmm_permute", made.defined() ? &made : nullptr, args[6]);
  });
}

// mem_eff_attention(q, k, v, causal, lengths_kv, lengths_q, out, scale)
PyObject* mem_eff_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    const at::Tensor* t[3];
    if (nargs != 7 || !PyBool_Check(args[3])) return not_ordinary();
    const int dt = attention_operands(args, 4, t);
    if (dt < 0) return not_ordinary();
    const int64_t B = t[0]->size(0), H = t[0]->size(1), M = t[0]->size(2), K = t[0]->size(3), N = t[2]->size(2), O = t[2]->size(3);
    if (t[1]->size(0) != B || t[1]->size(1) != H || t[1]->size(2) != N || t[1]->size(3) != K || t[2]->size(0) != B ||
        t[2]->size(1) != H)
      return not_ordinary();
    const int32_t* lengths[2] = {};
    for (int i = 0; i < 2; ++i) {
      if (args[4 + i] == Py_None) continue;
      const at::Tensor* l = gpu_tensor(args[4 + i]);
      if (l == nullptr || l->scalar_type() != at::kInt || l->numel() != B || !l->is_contiguous() || l->device() != t[0]->device())
        return not_ordinary();
      lengths[i] = static_cast<const int32_t*>(l->data_ptr());
    }
    at::Tensor made;
    void* out = attention_out(args[6], {B, M, H, O}, *t[0], &made);
    if (out == nullptr) return not_ordinary();
    const float scale = (float)std::pow((double)K, -0.5);
    const int causal = args[3] == Py_True;
    const void *q = pointer(t[0]), *k = pointer(t[1]), *v = pointer(t[2]);
    void* stream = current_stream();
    const int rc = unlocked([&] {
      return aitamd_mem_eff_attention(dt, q, k, v, out, B, H, M, N, K, O, scale, causal, lengths[0], lengths[1], stream);
    });
    return finish(rc, "mem_eff_attention", made.defined() ? &made : nullptr, args[6]);
  });
}

// ---- Model.run_with_tensors -------------------------------------------------------------------------------------

typedef AITemplateError (*ModelRun)(AITemplateModelHandle, const AITData*, size_t, AITData*, size_t, AITemplateStreamHandle, bool,
                                    bool, int64_t**);

bool model_dtype(at::ScalarType s, AITemplateDtype* out) {
  switch (s) {
    case at::kHalf: *out = AITemplateDtype::kHalf; return true;
    case at::kBFloat16: *out = AITemplateDtype::kBFloat16; return true;
    case at::kFloat: *out = AITemplateDtype::kFloat; return true;
    case at::kInt: *out = AITemplateDtype::kInt; return true;
    case at::kLong: *out = AITemplateDtype::kLong; return true;
    case at::kBool: *out = AITemplateDtype::kBool; return true;
    default: return false;
  }
}

typedef std::vector<std::pair<THPObjectPtr, size_t>> Names;

// A Python integer from 0 to 2^63 - 1, or -1, without an error of Python's: such calls are declined
int64_t small_integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1) PyErr_Clear();
  return v < 0 ? -1 : v;
}

// The tensors of a list, or of a dict ordered by `index` (name -> position), and the names in the order of the caller's
// dict (of `index` for a list); false where they are not ordinary.  Both are held, not borrowed: the caller's containers
// may change while the run has given up the interpreter lock.
bool model_tensors(PyObject* params, PyObject* index, std::vector<at::Tensor>* out, Names* names) {
  auto hold = [&](size_t i, PyObject* o) {
    const at::Tensor* t = gpu_tensor(o);
    if (t == nullptr || !t->is_contiguous()) return false;
    (*out)[i] = *t;
    return true;
  };
  const Py_ssize_t n = PyDict_Size(index);
  out->resize((size_t)n);
  const bool by_name = PyDict_CheckExact(params);
  if (by_name) {
    if (PyDict_Size(params) != n) return false;
  } else {
    if ((!PyList_CheckExact(params) && !PyTuple_CheckExact(params)) || PySequence_Fast_GET_SIZE(params) != n) return false;
    for (Py_ssize_t i = 0; i < n; ++i)
      if (!hold((size_t)i, PySequence_Fast_GET_ITEM(params, i))) return false;
  }
  PyObject *name, *value;
  Py_ssize_t pos = 0;
  while (PyDict_Next(by_name ? params : index, &pos, &name, &value)) {
    if (!PyUnicode_CheckExact(name)) return false;
    PyObject* at_index = PyDict_GetItemWithError(index, name);  // (no error: strings have hashes and compare)
    if (at_index == nullptr) return false;
    const size_t i = (size_t)small_integer(at_index);
    if (i >= (size_t)n || (by_name && !hold(i, value))) return false;
    if (names != nullptr) names->emplace_back(THPObjectPtr::dup(name), i);
  }
  return true;
}

// What a run gets of its tensors.  The sizes are copied: a tensor's own move when it is given another shape.
struct ModelData {
  std::vector<AITData> data;
  std::vector<c10::DimVector> sizes;
};
bool model_data(const std::vector<at::Tensor>& tensors, ModelData* out) {
  out->data.resize(tensors.size());
  out->sizes.reserve(tensors.size());
  for (size_t i = 0; i < tensors.size(); ++i) {
    const at::Tensor& t = tensors[i];
    const c10::DimVector& sizes = out->sizes.emplace_back(t.sizes().begin(), t.sizes().end());
    AITData& d = out->data[i];
    d.ptr = t.data_ptr();
    d.shape = AITemplateParamShape(sizes.data(), sizes.size());
    if (!model_dtype(t.scalar_type(), &d.dtype)) return false;
  }
  return true;
}

// model_run(function address, handle, input index, output index, output ranks, inputs, outputs, stream, sync, graph_mode)
PyObject* model_run(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    if (nargs != 10 || !PyDict_CheckExact(args[2]) || !PyDict_CheckExact(args[3]) || !PyList_CheckExact(args[4]) ||
        !PyBool_Check(args[8]) || !PyBool_Check(args[9]))
      return not_ordinary();
    std::vector<at::Tensor> in, out;
    Names names;
    if (!model_tensors(args[5], args[2], &in, nullptr) || !model_tensors(args[6], args[3], &out, &names)) return not_ordinary();
    ModelData in_data, out_data;
    if (!model_data(in, &in_data) || !model_data(out, &out_data)) return not_ordinary();
    const size_t n_out = out.size();
    std::vector<int64_t> dims;
    dims.reserve(8 * n_out);
    std::vector<int64_t*> shapes(n_out);
    if ((size_t)PyList_GET_SIZE(args[4]) != n_out) return not_ordinary();
    for (size_t i = 0; i < n_out; ++i) {
      const int64_t rank = small_integer(PyList_GET_ITEM(args[4], (Py_ssize_t)i));
      if (rank != (int64_t)out_data.sizes[i].size() || dims.size() + (size_t)rank > dims.capacity()) return not_ordinary();
      shapes[i] = dims.data() + dims.size();
      dims.resize(dims.size() + (size_t)rank);
    }
    auto run = reinterpret_cast<ModelRun>(PyLong_AsVoidPtr(args[0]));
    auto handle = reinterpret_cast<AITemplateModelHandle>(PyLong_AsVoidPtr(args[1]));
    void* stream = args[7] == Py_None ? current_stream() : PyLong_AsVoidPtr(args[7]);
    if (PyErr_Occurred()) return nullptr;
    const bool sync = args[8] == Py_True, graph = args[9] == Py_True;
    const int rc = unlocked([&] {
      return (int)run(handle, in_data.data.data(), in.size(), out_data.data.data(), n_out,
                      reinterpret_cast<AITemplateStreamHandle>(stream), sync, graph, shapes.data());
    });
    if (rc != 0) return PyErr_Format(PyExc_RuntimeError, "Error in function: AITemplateModelContainerRun");
    // every output under its name (a caller's dict keeps its order), as a view of the shape of this run
    THPObjectPtr result(PyDict_New());
    if (!result) return nullptr;
    for (const auto& [name, i] : names) {
      const at::Tensor& t = out[i];
      const at::IntArrayRef shape(shapes[i], out_data.sizes[i].size());
      const int64_t numel = c10::multiply_integers(shape);
      THPObjectPtr view(THPVariable_Wrap(numel == t.numel() ? t.view(shape) : t.flatten().narrow(0, 0, numel).view(shape)));
      if (!view || PyDict_SetItem(result.get(), const_cast<PyObject*>(name.get()), view.get()) != 0) return nullptr;
    }
    return result.release();
  });
}

PyMethodDef kMethods[] = {
#define AITAMD_METHOD(f, doc) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL, doc}
    AITAMD_METHOD(gemm, "gemm(op, a, b, bias, d0, d1, out, algo, workspace)"),
    AITAMD_METHOD(bmm, "bmm(layout, a, b, out, d1, algo, what)"),
    AITAMD_METHOD(bmm_softmax_bmm_permute, "bmm_softmax_bmm_permute(q, k, v, heads, scale, causal, out)"),
    AITAMD_METHOD(mem_eff_attention, "mem_eff_attention(q, k, v, causal, lengths_kv, lengths_q, out)"),
    AITAMD_METHOD(model_run,
                  "model_run(function, handle, input_index, output_index, output_ranks, inputs, outputs, stream, sync, graph_mode)"),
#undef AITAMD_METHOD
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Eager calls and model runs on torch tensors (see eager.py, compiler/model.py)",
                       -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  THPObjectPtr module(PyModule_Create(&kModule));
  // (the loader compares it with the torch that is there)
  if (!module || PyModule_AddStringConstant(module.get(), "torch_version", TORCH_VERSION) != 0 ||
      PyModule_AddStringConstant(module.get(), "torch_build", AITAMD_TORCH_BUILD) != 0)
    return nullptr;
  return module.release();
}
