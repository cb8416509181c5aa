// The host side of the layer's calls in native code: checks a call's tensors, allocates its result and
// workspace from torch's allocator and enters the C ABI, in a few microseconds where the same steps in
// Python take tens (a decode step of a few tokens is over on the GPU in less).  Every function answers
// None when the call is anything but the plain case; the Python caller then takes its own path, which
// names what is wrong or serves what is rare.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/Context.h>
#include <ATen/EmptyTensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/moe_gfx950.h"

namespace {

PyObject* g_raw_stream = nullptr;   // torch._C._cuda_getCurrentRawStream

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MOE_F32;
    case at::kHalf: return MOE_F16;
    case at::kBFloat16: return MOE_BF16;
    default: return -1;
  }
}

const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// A GPU tensor, or null.
const at::Tensor* gpu_tensor(PyObject* o) {
  const at::Tensor* t = tensor(o);
  return t && t->is_cuda() ? t : nullptr;
}

// False when `o` is neither None nor a contiguous GPU tensor on `dev` of `type` and `shape`; else `t` is it or null.
bool optional_tensor(PyObject* o, const at::Device& dev, at::ScalarType type, at::IntArrayRef shape, const at::Tensor** t) {
  *t = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* x = gpu_tensor(o);
  if (!x || x->device() != dev || x->scalar_type() != type || !x->is_contiguous() || x->sizes() != shape) return false;
  *t = x;
  return true;
}

// Plain ints, bools and floats, or false, with no Python error set: the Python caller's own path then converts
// what can be converted and names what cannot.
bool int_arg(PyObject* o, int64_t* v) {
  int overflow = 0;
  if (!PyLong_CheckExact(o)) return false;
  *v = PyLong_AsLongAndOverflow(o, &overflow);
  return !overflow;
}
bool flag_arg(PyObject* o, bool* v) {
  if (!PyBool_Check(o)) return false;
  *v = o == Py_True;
  return true;
}
bool float_arg(PyObject* o, float* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = static_cast<float>(PyFloat_AS_DOUBLE(o));
  return true;
}

// Other Python threads run while a call allocates and enqueues (fresh memory and the first launch of a kernel take
// milliseconds, a full queue makes a launch wait).  Nothing of Python is touched meanwhile.
struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  WithoutGil() = default;
  WithoutGil(const WithoutGil&) = delete;
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// Allocations and the library call at their end, made without the GIL; its return code.
template <typename Call>
int enqueue(const Call& call) {
  const WithoutGil nogil;
  return call();
}

void* current_stream(const at::Device& dev) {
  PyObject* idx = PyLong_FromLong(dev.index());
  PyObject* r = idx ? PyObject_CallOneArg(g_raw_stream, idx) : nullptr;
  Py_XDECREF(idx);
  if (!r) throw python_error();
  void* s = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  return s;
}

void check(int rc) {
  if (rc == 0) return;
  PyErr_SetString(PyExc_RuntimeError, moe_last_error());
  throw python_error();
}

// An uninitialised tensor on `dev`, which is the current device.  Where nothing stands between the dispatcher and the
// allocator that could change the tensor (a mode, a transform, memory that is to be filled) it comes from the same allocator
// without a way through the dispatcher: a call of a few microseconds makes up to five.  What only looks on does not count: a
// profiler has the allocator's memory events of these tensors and no `aten::empty`.  Norm and gate of 135 tokens enqueued from
// Python, by the dispatcher and this way: 15.9 and 13.9 us.
at::Tensor empty(at::IntArrayRef shape, at::ScalarType type, const at::Device& dev) {
  const uint64_t included = c10::impl::tls_local_dispatch_key_set().included_.raw_repr();
  const at::Context& context = at::globalContext();
  if ((included & ~c10::default_included_set.raw_repr()) ||
      (context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory()))
    return at::empty(shape, at::TensorOptions().dtype(type).device(dev));
  constexpr c10::DispatchKeySet keys(c10::DispatchKey::CUDA);
  return at::detail::empty_generic(shape, at::detail::getCUDAHooks().getCUDADeviceAllocator(), keys, type, std::nullopt);
}

PyObject* tuple_of(const at::Tensor& a, const at::Tensor& b, const at::Tensor& c) {
  PyObject* t = PyTuple_New(3);
  if (!t) throw python_error();
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(a));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(b));
  PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(c));
  return t;
}

#define MOE_NONE Py_RETURN_NONE

// layer(x, router_logits | None, w13, w2, w13_bias, w2_bias, w13_scale, w2_scale, topk_weights | None,
//       topk_ids | None, top_k, renormalize, activation, weight_on_input, weight_layout, inplace)
// -> result tensor, or None.  Codes as in moe_gfx950.h.
PyObject* layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t K, activation, weight_layout;
  bool renormalize, weight_on_input, inplace;
  if (n != 16 || !int_arg(a[10], &K) || !flag_arg(a[11], &renormalize) || !int_arg(a[12], &activation) ||
      !flag_arg(a[13], &weight_on_input) || !int_arg(a[14], &weight_layout) || !flag_arg(a[15], &inplace))
    MOE_NONE;
  const at::Tensor *x = gpu_tensor(a[0]), *w13 = gpu_tensor(a[2]), *w2 = gpu_tensor(a[3]);
  if (!x || !w13 || !w2 || x->dim() != 2 || w13->dim() != 3 || w2->dim() != 3) MOE_NONE;
  const at::Device dev = x->device();
  if (w13->device() != dev || w2->device() != dev || !x->is_contiguous()) MOE_NONE;
  const int64_t T = x->size(0), H = x->size(1), E = w13->size(0), N = w13->size(1), I = N / 2;
  if (T < 1 || T > 65536 || N % 2 || I < 1 || w13->size(2) != H || w2->size(0) != E || w2->size(1) != H || w2->size(2) != I)
    MOE_NONE;
  if (w13->stride(2) != 1 || w2->stride(2) != 1) MOE_NONE;
  const int act = dtype_code(x->scalar_type());
  if (act < 0 || w2->scalar_type() != w13->scalar_type()) MOE_NONE;
  const bool fp8 = w13->scalar_type() == at::kFloat8_e4m3fn;
  const at::Tensor *b13, *b2, *s13, *s2;
  const int64_t n13[2] = {E, N}, n2[2] = {E, H};
  if (!optional_tensor(a[4], dev, x->scalar_type(), n13, &b13) || !optional_tensor(a[5], dev, x->scalar_type(), n2, &b2) ||
      !optional_tensor(a[6], dev, at::kFloat, n13, &s13) || !optional_tensor(a[7], dev, at::kFloat, n2, &s2))
    MOE_NONE;
  if (fp8) {
    if (act == MOE_F32 || !s13 || !s2 || b13 || b2 || H % 16 || I % 16) MOE_NONE;
    for (const at::Tensor* w : {w13, w2}) {
      if ((E > 1 && w->stride(0) % 16) || w->stride(1) % 16) MOE_NONE;
      if (reinterpret_cast<uintptr_t>(w->data_ptr()) & 15u) MOE_NONE;
    }
    if (reinterpret_cast<uintptr_t>(x->data_ptr()) & 15u) MOE_NONE;
  } else if (w13->scalar_type() != x->scalar_type() || s13 || s2) {
    MOE_NONE;
  }
  MoeLayerArgs m{};
  if (K < 1 || K > E || T * K > INT32_MAX) MOE_NONE;
  if (a[1] != Py_None) {
    const at::Tensor* g = gpu_tensor(a[1]);
    if (!g || g->device() != dev || g->dim() != 2 || g->size(0) != T || g->size(1) != E || !g->is_contiguous()) MOE_NONE;
    m.logits_dtype = dtype_code(g->scalar_type());
    if (m.logits_dtype < 0) MOE_NONE;
    m.router_logits = g->data_ptr();
    m.renormalize = renormalize;
  } else {
    const at::Tensor *w, *ids;
    const int64_t tk[2] = {T, K};
    if (!optional_tensor(a[8], dev, at::kFloat, tk, &w) || !optional_tensor(a[9], dev, at::kInt, tk, &ids) || !w || !ids) MOE_NONE;
    m.topk_weights = static_cast<float*>(w->data_ptr());
    m.topk_ids = static_cast<int32_t*>(ids->data_ptr());
  }
  m.activation = static_cast<int32_t>(activation);
  m.apply_router_weight_on_input = weight_on_input;
  m.weight_layout = static_cast<int32_t>(weight_layout);
  c10::OptionalDeviceGuard guard(dev);
  m.x = x->data_ptr();
  m.w13 = w13->data_ptr();
  m.w2 = w2->data_ptr();
  m.w13_bias = b13 ? b13->data_ptr() : nullptr;
  m.w2_bias = b2 ? b2->data_ptr() : nullptr;
  m.w13_scale = s13 ? static_cast<const float*>(s13->data_ptr()) : nullptr;
  m.w2_scale = s2 ? static_cast<const float*>(s2->data_ptr()) : nullptr;
  m.w13_stride_e = w13->stride(0);
  m.w13_stride_n = w13->stride(1);
  m.w2_stride_e = w2->stride(0);
  m.w2_stride_n = w2->stride(1);
  m.T = static_cast<int32_t>(T);
  m.H = static_cast<int32_t>(H);
  m.I = static_cast<int32_t>(I);
  m.E = static_cast<int32_t>(E);
  m.K = static_cast<int32_t>(K);
  m.act_dtype = act;
  m.weight_dtype = fp8 ? static_cast<int>(MOE_E4M3) : act;
  m.swiglu_alpha = 1.702f;
  m.swiglu_limit = 7.0f;
  m.stream = current_stream(dev);
  m.workspace_bytes = moe_layer_workspace_bytes(&m);
  if (m.workspace_bytes <= 0) MOE_NONE;
  const at::ScalarType type = x->scalar_type();
  at::Tensor out = *x;
  check(enqueue([&] {
    if (!inplace) out = empty({T, H}, type, dev);
    m.out = out.data_ptr();
    const at::Tensor ws = empty({m.workspace_bytes}, at::kByte, dev);
    m.workspace = ws.data_ptr();
    return moe_layer(&m);
  }));
  if (inplace) {
    Py_INCREF(a[0]);
    return a[0];
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// topk(router_logits, top_k, renormalize) -> (weights, ids, token_expert_indices), or None.
PyObject* topk(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t K;
  bool renormalize;
  if (n != 3 || !int_arg(a[1], &K) || !flag_arg(a[2], &renormalize)) MOE_NONE;
  const at::Tensor* g = gpu_tensor(a[0]);
  if (!g || g->dim() != 2 || !g->is_contiguous() || g->size(0) < 1) MOE_NONE;
  const int dtype = dtype_code(g->scalar_type());
  const int64_t T = g->size(0), E = g->size(1);
  if (dtype < 0 || K < 1 || K > E || T * K > INT32_MAX) MOE_NONE;
  const at::Device dev = g->device();
  c10::OptionalDeviceGuard guard(dev);
  void* const stream = current_stream(dev);
  const void* const logits = g->data_ptr();
  at::Tensor w, ids, tei;
  check(enqueue([&] {
    w = empty({T, K}, at::kFloat, dev), ids = empty({T, K}, at::kInt, dev), tei = empty({T, K}, at::kInt, dev);
    return moe_topk_softmax_typed(logits, dtype, static_cast<float*>(w.data_ptr()),
                                  static_cast<int32_t*>(ids.data_ptr()), static_cast<int32_t*>(tei.data_ptr()),
                                  static_cast<int>(T), static_cast<int>(E), static_cast<int>(K), renormalize, stream);
  }));
  return tuple_of(w, ids, tei);
  END_HANDLE_TH_ERRORS
}

// rms_norm(x, residual | None, weight, eps) -> the normalised tensor (residual updated in place), or None.
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  float eps;
  if (n != 4 || !float_arg(a[3], &eps)) MOE_NONE;
  const at::Tensor *x = gpu_tensor(a[0]), *w = gpu_tensor(a[2]);
  const at::Tensor* res = a[1] == Py_None ? nullptr : gpu_tensor(a[1]);
  if (!x || !w || (!res && a[1] != Py_None) || x->dim() != 2) MOE_NONE;
  const at::Device dev = x->device();
  const int dtype = dtype_code(x->scalar_type());
  const int64_t T = x->size(0), H = x->size(1);
  if (dtype < 0 || T < 1 || H < 1 || H > INT32_MAX || !x->is_contiguous()) MOE_NONE;
  if (w->device() != dev || w->dim() != 1 || w->size(0) != H || w->scalar_type() != x->scalar_type() || !w->is_contiguous())
    MOE_NONE;
  if (res && (res->device() != dev || res->scalar_type() != x->scalar_type() || res->sizes() != x->sizes() || !res->is_contiguous()))
    MOE_NONE;
  c10::OptionalDeviceGuard guard(dev);
  void* const stream = current_stream(dev);
  void* const r = res ? res->data_ptr() : nullptr;
  const void *const in = x->data_ptr(), *const weight = w->data_ptr();
  const at::ScalarType type = x->scalar_type();
  at::Tensor out;
  check(enqueue([&] {
    out = empty({T, H}, type, dev);
    return moe_add_rms_norm(out.data_ptr(), H, r, H, in, H, weight, dtype, T, static_cast<int>(H), eps, stream);
  }));
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// False when a linear of these two is anything but the library's product of their bytes, so that it has to be asked for:
// tensor subclasses and wrappers, negated or zero tensors, function and dispatch modes (a flop counter, a tracer),
// transforms, and autocast to another type.
bool linear_is_plain(PyObject* px, const at::Tensor& x, PyObject* pg, const at::Tensor& g) {
  if (!THPVariable_CheckExact(px) || !THPVariable_CheckExact(pg) || at::impl::torch_function_mode_enabled()) return false;
  constexpr c10::DispatchKeySet dense({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView,
                                       c10::DispatchKey::AutocastCUDA});
  const uint64_t included = c10::impl::tls_local_dispatch_key_set().included_.raw_repr();
  if (((x.key_set() | g.key_set()).raw_repr() & ~dense.raw_repr()) | (included & ~c10::default_included_set.raw_repr())) return false;
  return !at::autocast::is_autocast_enabled(at::kCUDA) || at::autocast::get_autocast_dtype(at::kCUDA) == x.scalar_type();
}

// gate_topk(x, gate_weight, top_k, renormalize) -> (weights, ids, token_expert_indices), or None;
// gate_topk_few: the same for batches that moe_gate_topk_few serves, where a linear would be no other.
template <bool FEW>
PyObject* gate_topk(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t K;
  bool renormalize;
  if (n != 4 || !int_arg(a[2], &K) || !flag_arg(a[3], &renormalize)) MOE_NONE;
  const at::Tensor *x = gpu_tensor(a[0]), *g = gpu_tensor(a[1]);
  if (!x || !g || x->dim() != 2 || g->dim() != 2 || !x->is_contiguous() || !g->is_contiguous()) MOE_NONE;
  if (FEW && !linear_is_plain(a[0], *x, a[1], *g)) MOE_NONE;
  const at::Device dev = x->device();
  const int dtype = dtype_code(x->scalar_type());
  const int64_t T = x->size(0), H = x->size(1), E = g->size(0);
  if (T < 1 || g->device() != dev || g->scalar_type() != x->scalar_type() || g->size(1) != H || K < 1 || K > E ||
      T * K > INT32_MAX || T * H * 2 >= (int64_t{1} << 32))
    MOE_NONE;
  int64_t few_bytes = 0;
  if (FEW) {
    if (T > INT32_MAX || H > INT32_MAX || E > INT32_MAX) MOE_NONE;
    few_bytes = moe_gate_topk_few_bytes(static_cast<int>(T), static_cast<int>(H), static_cast<int>(E), dtype);
    if (!few_bytes) MOE_NONE;
  } else if ((dtype != MOE_BF16 && dtype != MOE_F16) || (E != 32 && E != 64 && E != 128) || H % 64) {
    MOE_NONE;
  }
  if ((reinterpret_cast<uintptr_t>(x->data_ptr()) | reinterpret_cast<uintptr_t>(g->data_ptr())) & 15u) MOE_NONE;
  c10::OptionalDeviceGuard guard(dev);
  void* const stream = current_stream(dev);
  const void *const in = x->data_ptr(), *const gate = g->data_ptr();
  at::Tensor w, ids, tei;
  check(enqueue([&] {
    w = empty({T, K}, at::kFloat, dev), ids = empty({T, K}, at::kInt, dev), tei = empty({T, K}, at::kInt, dev);
    if (FEW) {
      const at::Tensor scratch = empty({few_bytes / 4}, at::kFloat, dev);
      return moe_gate_topk_few(in, gate, dtype, static_cast<float*>(w.data_ptr()), static_cast<int32_t*>(ids.data_ptr()),
                               static_cast<int32_t*>(tei.data_ptr()), static_cast<int>(T), static_cast<int>(H),
                               static_cast<int>(E), static_cast<int>(K), renormalize, scratch.data_ptr(), few_bytes, stream);
    }
    return moe_gate_topk_softmax(in, gate, dtype, nullptr, static_cast<float*>(w.data_ptr()),
                                 static_cast<int32_t*>(ids.data_ptr()), static_cast<int32_t*>(tei.data_ptr()),
                                 static_cast<int>(T), static_cast<int>(H), static_cast<int>(E), static_cast<int>(K),
                                 renormalize, stream);
  }));
  return tuple_of(w, ids, tei);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(layer)), METH_FASTCALL, nullptr},
    {"topk", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(topk)), METH_FASTCALL, nullptr},
    {"rms_norm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(rms_norm)), METH_FASTCALL, nullptr},
    {"gate_topk", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(gate_topk<false>)), METH_FASTCALL, nullptr},
    {"gate_topk_few", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(gate_topk<true>)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_moe_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__moe_host(void) {
  PyObject* c = PyImport_ImportModule("torch._C");
  if (!c) return nullptr;
  g_raw_stream = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
  Py_DECREF(c);
  if (!g_raw_stream) return nullptr;
  return PyModule_Create(&module);
}
