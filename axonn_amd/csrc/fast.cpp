// The usual calls of a Linear layer without their way through Python: checks, output and workspace tensors and
// the library's entry point in one function each.  Whatever is not usual - another layout, type, device or
// alignment, an empty batch, a size that needs padding, a mode that watches tensors - answers None before anything is
// launched, and the caller (axonn_amd/ops.py, fully_connected.py) goes the general way from the start.  An error of the
// library is raised, as it is there: it can follow a launch (one that an earlier call left behind is reported by the
// next), and a second one would add the weight gradient again.
//
// Host time of a forward of 8 x 1024 x 1024 bf16 through a Linear without gradients 15.6 us in Python, 5.4 here (3.7 of
// it the library's call and its launch); forward and backward of 64 x 1024 x 1024, autograd's part included, 153 -> 99.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <vector>

#include "axn.h"

namespace {

// ---- entry points of libaxn_gfx950.so, bound by address ------------------------------------
#define ENTRY_POINTS(X)                                                                                          \
  X(axn_gemm_any_n) X(axn_gemm_dgrad_ws) X(axn_gemm_dgrad) X(axn_gemm_dgrad_f16) X(axn_gemm_wgrad_ws)            \
  X(axn_gemm_wgrad) X(axn_gemm_wgrad_f16) X(axn_gemm_bwd) X(axn_gemm_bwd_ws) X(axn_dgelu_dbias)                  \
  X(axn_gemm_workspace_bytes) X(axn_gemm_bwd_workspace_bytes) X(axn_dgelu_dbias_workspace_bytes)                 \
  X(axn_gemm_f32_workspace_bytes) X(axn_gemm_fwd_f32_ws) X(axn_gemm_dgrad_f32_ws) X(axn_gemm_wgrad_f32_ws)
struct Library {
#define DECLARE(name) decltype(&::name) name = nullptr;
  ENTRY_POINTS(DECLARE)
#undef DECLARE
} lib;
PyObject* check_status = nullptr;   // axonn_amd._native.check: raises the library's error

// Rows further apart are packed first by the general way.
constexpr int64_t kFarRows = 1 << 22;

// What the library would use, a function of the sizes alone: the last answers of a thread.
enum Need { FWD, DGRAD, WGRAD, F32_FWD, F32_DGRAD, F32_WGRAD, BOTH, BOTH_ADD, DBIAS };
size_t bytes_needed(Need kind, int64_t M, int64_t N, int64_t K) {
  struct Answer {
    int64_t kind, M, N, K;
    size_t bytes;
  };
  thread_local std::vector<Answer> answers(256, Answer{-1, 0, 0, 0, 0});
  const uint64_t h = (uint64_t)M * 0x9e3779b97f4a7c15u ^ (uint64_t)N * 0xc2b2ae3d27d4eb4fu ^ (uint64_t)K * 0x165667b19e3779f9u;
  Answer& a = answers[(h >> 40 ^ (uint64_t)kind * 29) & 255];
  if (a.kind == kind && a.M == M && a.N == N && a.K == K) return a.bytes;
  size_t bytes;
  switch (kind) {
    case BOTH: case BOTH_ADD: bytes = lib.axn_gemm_bwd_workspace_bytes(M, N, K, kind == BOTH_ADD); break;
    case DBIAS: bytes = lib.axn_dgelu_dbias_workspace_bytes(M, N); break;
    case F32_FWD: case F32_DGRAD: case F32_WGRAD: bytes = lib.axn_gemm_f32_workspace_bytes(kind - F32_FWD, M, N, K); break;
    default: bytes = lib.axn_gemm_workspace_bytes(kind, M, N, K);
  }
  a = Answer{kind, M, N, K, bytes};
  return bytes;
}

// ---- tensors -------------------------------------------------------------------------------
bool is16(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
int code_of(at::ScalarType t) { return t == at::kBFloat16 ? AXN_BF16 : t == at::kHalf ? AXN_F16 : AXN_F32; }

// A tensor as the kernels take it: plain, dense, on the current device, 16-byte aligned.
bool plain(const at::Tensor& t, c10::DeviceIndex device) {
  constexpr c10::DispatchKeySet usual = c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                                             c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
  return t.defined() && t.is_cuda() && t.get_device() == device && t.is_contiguous() && !t.is_neg() && !t.is_conj() &&
         (t.key_set().raw_repr() & ~usual.raw_repr()) == 0 && ((uintptr_t)t.const_data_ptr() & 15u) == 0;
}
// Modes and transforms that see tensors go by the general way, which they see (or which refuses them).
bool nothing_watches() {
  if (lib.axn_gemm_any_n == nullptr || at::impl::torch_function_mode_enabled()) return false;
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing() &&
         !tls.included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !tls.included_.has(c10::DispatchKey::Python);
}
at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like) {
  return at::empty(sizes, like.options().dtype(type).requires_grad(false));
}
struct Workspace {
  at::Tensor tensor;
  void* at = nullptr;
  size_t bytes = 0;
  Workspace(size_t n, const at::Tensor& like) : bytes(n) {
    if (n == 0) return;
    tensor = empty({(int64_t)n}, at::kByte, like);
    at = tensor.mutable_data_ptr();
  }
};
void* pointer(const at::Tensor& t) { return t.defined() ? const_cast<void*>(t.const_data_ptr()) : nullptr; }

struct Unlocked {   // the interpreter's lock is not held while kernels are launched
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

c10::DeviceIndex current_device_for(const at::Tensor& t) { return t.is_cuda() ? c10::hip::current_device() : c10::DeviceIndex(-1); }
at::Tensor tensor_or_none(PyObject* o) { return o == Py_None ? at::Tensor() : THPVariable_Unpack(o); }
bool is_tensor_or_none(PyObject* o) { return o == Py_None || THPVariable_CheckExact(o); }   // (no other subclass than Parameter)
PyObject* wrap(const at::Tensor& t) {
  if (t.defined()) return THPVariable_Wrap(t);
  Py_RETURN_NONE;
}
bool truth(PyObject* o) {
  const int yes = PyObject_IsTrue(o);
  if (yes < 0) throw python_error();
  return yes != 0;
}
at::ScalarType type_of(PyObject* o) {   // of AXN_*; anything else is no type
  const long c = PyLong_AsLong(o);
  return c == AXN_BF16 ? at::kBFloat16 : c == AXN_F16 ? at::kHalf : c == AXN_F32 ? at::kFloat : at::ScalarType::Undefined;
}

constexpr int kNotTaken = 1;   // beside the library's status: nothing was launched, the general way takes the call
PyObject* no_result(int status) {
  if (status == kNotTaken) Py_RETURN_NONE;
  Py_XDECREF(PyObject_CallFunction(check_status, "i", status));
  return nullptr;
}

// ---- forward -------------------------------------------------------------------------------
// act(X W^T + b) into y [.., N] (and z).
int forward(const at::Tensor& x, const at::Tensor& w, const at::Tensor& bias, int64_t M, int64_t N, int64_t K, bool gelu,
            bool save_z, bool out_f32, at::IntArrayRef shape, c10::DeviceIndex device, at::Tensor& y, at::Tensor& z) {
  const at::ScalarType type = x.scalar_type();
  const bool half = is16(type);
  if (!(half || type == at::kFloat) || w.scalar_type() != type || M < 1 || N < 1 || K < 1 || K >= kFarRows ||
      M > 0x7fffffff || N > 0x7ffffff8)
    return kNotTaken;
  if (half ? K % 8 != 0 : out_f32) return kNotTaken;
  int epilogue = bias.defined() ? (gelu ? AXN_EPI_BIAS_GELU : AXN_EPI_BIAS) : (gelu ? AXN_EPI_GELU : AXN_EPI_NONE);
  if (bias.defined()) {
    if (bias.numel() != N || !plain(bias, device)) return kNotTaken;
    if (half && bias.scalar_type() == type) epilogue |= AXN_BIAS_16BIT;
    else if (bias.scalar_type() != at::kFloat) return kNotTaken;
  } else if (out_f32) {
    return kNotTaken;
  }
  y = empty(shape, out_f32 ? at::kFloat : type, x);
  if (gelu && save_z) z = empty(shape, type, x);
  const auto stream = c10::hip::getCurrentHIPStream(device).stream();
  if (half) {
    const Workspace ws(out_f32 ? 0 : bytes_needed(FWD, M, N, K), x);
    return lib.axn_gemm_any_n(AXN_GEMM_FWD, pointer(x), pointer(w), pointer(bias), pointer(y), pointer(z), code_of(type),
                              M, N, K, K, K, N, epilogue, 0, out_f32 ? AXN_F32 : code_of(type), ws.at, ws.bytes, stream);
  }
  const Workspace ws(bytes_needed(F32_FWD, M, N, K), x);
  return lib.axn_gemm_fwd_f32_ws((const float*)pointer(x), (const float*)pointer(w), (const float*)pointer(bias),
                                 (float*)pointer(y), (float*)pointer(z), M, N, K, epilogue, ws.at, ws.bytes, stream);
}

// gemm_fwd(x, w, bias, gelu, save_z, out_f32) -> (y, z) or None
PyObject* gemm_fwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6 || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !is_tensor_or_none(args[2])) Py_RETURN_NONE;
  const at::Tensor x = THPVariable_Unpack(args[0]), w = THPVariable_Unpack(args[1]), bias = tensor_or_none(args[2]);
  const c10::DeviceIndex device = current_device_for(x);
  if (!plain(x, device) || !plain(w, device) || x.dim() != 2 || w.dim() != 2 || x.size(1) != w.size(1) || !nothing_watches())
    Py_RETURN_NONE;
  const int64_t M = x.size(0), N = w.size(0);
  const bool gelu = truth(args[3]), save_z = truth(args[4]), out_f32 = truth(args[5]);
  at::Tensor y, z;
  int status;
  {
    Unlocked unlocked;
    status = forward(x, w, bias, M, N, x.size(1), gelu, save_z, out_f32, {M, N}, device, y, z);
  }
  if (status != AXN_OK) return no_result(status);
  PyObject* out = PyTuple_New(2);
  PyTuple_SET_ITEM(out, 0, wrap(y));
  PyTuple_SET_ITEM(out, 1, wrap(z));
  return out;
  END_HANDLE_TH_ERRORS
}

// linear(x, weight, bias, out_features, in_features, gelu) -> act(x W^T + b) or None; for callers without gradients:
// it makes no node of a graph, and answers None where one, a cast or a tangent might be wanted.
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6 || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !is_tensor_or_none(args[2]) ||
      at::GradMode::is_enabled())
    Py_RETURN_NONE;
  const at::Tensor x = THPVariable_Unpack(args[0]), w = THPVariable_Unpack(args[1]);
  const at::Tensor bias = tensor_or_none(args[2]);
  const c10::DeviceIndex device = current_device_for(x);
  if (at::autocast::is_autocast_enabled(at::kCUDA) || !plain(x, device) || !plain(w, device) ||
      x.dim() < 1 || !nothing_watches() || x._fw_grad(0).defined() || w._fw_grad(0).defined() ||
      (bias.defined() && bias._fw_grad(0).defined()))
    Py_RETURN_NONE;
  const int64_t N = PyLong_AsLongLong(args[3]), K = PyLong_AsLongLong(args[4]);
  const bool gelu = truth(args[5]);   // (here: objects are asked with the interpreter's lock held)
  if (PyErr_Occurred()) return nullptr;
  if (N < 1 || K < 1 || x.size(-1) != K || w.numel() != N * K) Py_RETURN_NONE;
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = N;
  at::Tensor y, z;
  int status;
  {
    Unlocked unlocked;
    const bool out_f32 = bias.defined() && bias.scalar_type() == at::kFloat && x.scalar_type() != at::kFloat;
    status = forward(x, w, bias, x.numel() / K, N, K, gelu, false, out_f32, shape, device, y, z);
  }
  if (status != AXN_OK) return no_result(status);
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

// ---- backward ------------------------------------------------------------------------------
struct Backward {
  at::Tensor dy, z, w, x, out;   // out: dW is added to it
  bool need_dx, need_dw, want_db, widen;
  at::ScalarType bias_type, dw_type;   // of the bias gradient, if the kernels write it; of dW
  at::Tensor dx, dw, db;

  int run(c10::DeviceIndex device) {
    const at::ScalarType type = x.scalar_type();
    const bool half = is16(type);
    const int64_t M = dy.size(0), N = dy.size(1), K = w.size(1);
    if (!(half || type == at::kFloat) || M < 1 || N % 8 != 0 || N < 8 || K < 1 || (half && K % 8 != 0) ||
        std::max(N, K) >= kFarRows || M > 0x7fffffff)
      return kNotTaken;
    const at::ScalarType from = dy.scalar_type();
    const bool pass = z.defined() || want_db, wide = half && from == at::kFloat;
    if (from != type && !(wide && pass)) return kNotTaken;
    if (z.defined() && (z.scalar_type() != type || z.sizes() != dy.sizes())) return kNotTaken;
    if (need_dw && dw_type != at::kFloat && dw_type != type) return kNotTaken;
    const auto stream = c10::hip::getCurrentHIPStream(device).stream();
    const int code = code_of(type);
    if (pass) {
      at::Tensor dz;
      if (z.defined() || wide) dz = empty({M, N}, type, x);
      int flags = code | (wide ? AXN_DY_F32 : 0);
      const bool db16 = want_db && half && bias_type == type;
      if (db16) flags |= AXN_DBIAS_16BIT;
      if (want_db) db = empty({N}, db16 ? type : at::kFloat, x);
      const Workspace ws(want_db ? std::max<size_t>(bytes_needed(DBIAS, M, N, 0), 16) : 0, x);
      const int rc = lib.axn_dgelu_dbias(pointer(dy), pointer(z), pointer(dz), flags, (float*)pointer(db), M, N, N, 0, ws.at,
                                         ws.bytes, stream);
      if (rc != AXN_OK) return rc;
      if (dz.defined()) dy = dz;
    }
    const int beta = out.defined() ? 1 : 0;
    void *pdy = pointer(dy), *pw = pointer(w), *px = pointer(x);
    // (dW comes after the input gradient's workspace has gone back: less is held at once)
    const auto make_dx = [&] { dx = empty({M, K}, type, x); return dx.mutable_data_ptr(); };
    const auto make_dw = [&] { dw = beta ? out : empty({N * K}, dw_type, x); return dw.mutable_data_ptr(); };
    if (!half) {
      if (need_dx) {
        void* pdx = make_dx();
        const Workspace ws(bytes_needed(F32_DGRAD, M, N, K), x);
        const int rc = lib.axn_gemm_dgrad_f32_ws((float*)pdy, (float*)pw, (float*)pdx, M, N, K, ws.at, ws.bytes, stream);
        if (rc != AXN_OK) return rc;
      }
      if (need_dw) {
        void* pdw = make_dw();
        const Workspace ws(bytes_needed(F32_WGRAD, M, N, K), x);
        const int rc = lib.axn_gemm_wgrad_f32_ws((float*)pdy, (float*)px, (float*)pdw, M, N, K, beta, ws.at, ws.bytes, stream);
        if (rc != AXN_OK) return rc;
      }
      return AXN_OK;
    }
    const int dw_code = code_of(dw_type);
    const size_t both = need_dx && need_dw ? bytes_needed(beta ? BOTH_ADD : BOTH, M, N, K) : 0;
    if (both) {
      void *pdx = make_dx(), *pdw = make_dw();
      const Workspace ws(both, x);
      return lib.axn_gemm_bwd_ws(pdy, pw, px, pdx, pdw, code, M, N, K, N, K, K, K, K, beta, dw_code, ws.at, ws.bytes, stream);
    }
    const size_t ws_d = need_dx ? bytes_needed(DGRAD, M, N, K) : 0, ws_w = need_dw ? bytes_needed(WGRAD, M, N, K) : 0;
    if (need_dx && need_dw && ws_d == 0 && ws_w == 0) {
      void *pdx = make_dx(), *pdw = make_dw();
      return lib.axn_gemm_bwd(pdy, pw, px, pdx, pdw, code, M, N, K, N, K, K, K, K, beta, dw_code, stream);
    }
    if (need_dx) {
      const bool wider = ws_d && widen;
      dx = empty({M, K}, wider ? at::kFloat : type, x);
      void* pdx = pointer(dx);
      const Workspace ws(ws_d, x);
      int rc;
      if (wider) {
        rc = lib.axn_gemm_any_n(AXN_GEMM_DGRAD, pdy, pw, nullptr, pdx, nullptr, code, M, N, K, N, K, K, AXN_EPI_NONE, 0,
                                AXN_F32 | AXN_ROUNDED, ws.at, ws.bytes, stream);
      } else if (ws_d) {
        rc = lib.axn_gemm_dgrad_ws(pdy, pw, pdx, code, M, N, K, N, K, K, ws.at, ws.bytes, stream);
      } else {
        rc = (type == at::kHalf ? lib.axn_gemm_dgrad_f16 : lib.axn_gemm_dgrad)(pdy, pw, pdx, M, N, K, N, K, K, stream);
      }
      if (rc != AXN_OK) return rc;
    }
    if (!need_dw) return AXN_OK;
    void* pdw = make_dw();
    const Workspace ws(ws_w, x);
    if (ws_w)
      return lib.axn_gemm_wgrad_ws(pdy, px, pdw, code, M, N, K, N, K, K, beta, dw_code, ws.at, ws.bytes, stream);
    return (type == at::kHalf ? lib.axn_gemm_wgrad_f16 : lib.axn_gemm_wgrad)(pdy, px, pdw, M, N, K, N, K, K, beta, dw_code, stream);
  }
};

// backward(dy, z, w, x, out, need_dx, need_dw, want_db, bias type, dW type, widen) -> (dx, dw flat, db) or None
PyObject* backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11 || !THPVariable_CheckExact(args[0]) || !is_tensor_or_none(args[1]) || !THPVariable_CheckExact(args[2]) ||
      !THPVariable_CheckExact(args[3]) || !is_tensor_or_none(args[4]))
    Py_RETURN_NONE;
  Backward b;
  b.dy = THPVariable_Unpack(args[0]);
  b.z = tensor_or_none(args[1]);
  b.w = THPVariable_Unpack(args[2]);
  b.x = THPVariable_Unpack(args[3]);
  b.out = tensor_or_none(args[4]);
  b.need_dx = truth(args[5]);
  b.need_dw = truth(args[6]);
  b.want_db = truth(args[7]);
  b.bias_type = type_of(args[8]);
  b.dw_type = type_of(args[9]);
  b.widen = truth(args[10]);
  if (PyErr_Occurred()) return nullptr;
  const c10::DeviceIndex device = current_device_for(b.dy);
  if (!plain(b.dy, device) || !plain(b.w, device) || !plain(b.x, device) || b.dy.dim() != 2 || b.w.dim() != 2 || b.x.dim() != 2 ||
      b.w.scalar_type() != b.x.scalar_type() || b.w.size(0) != b.dy.size(1) || b.x.size(0) != b.dy.size(0) ||
      b.x.size(1) != b.w.size(1) || (b.z.defined() && !plain(b.z, device)) || !nothing_watches())
    Py_RETURN_NONE;
  if (b.out.defined() && (!b.need_dw || !plain(b.out, device) || b.out.scalar_type() != b.dw_type || b.out.numel() != b.w.numel()))
    Py_RETURN_NONE;
  int status;
  {
    Unlocked unlocked;
    status = b.run(device);
  }
  if (status != AXN_OK) return no_result(status);
  PyObject* out = PyTuple_New(3);
  PyTuple_SET_ITEM(out, 0, wrap(b.dx));
  PyTuple_SET_ITEM(out, 1, wrap(b.dw));
  PyTuple_SET_ITEM(out, 2, wrap(b.db));
  return out;
  END_HANDLE_TH_ERRORS
}

// bind({name: address, "check": axonn_amd._native.check}): the library's entry points, and what raises their errors
PyObject* bind(PyObject*, PyObject* table) {
  Library bound;
#define BIND(name)                                                                        \
  {                                                                                       \
    PyObject* address = PyMapping_GetItemString(table, #name);                            \
    if (address == nullptr) return nullptr;                                               \
    bound.name = (decltype(bound.name))(uintptr_t)PyLong_AsUnsignedLongLong(address);     \
    Py_DECREF(address);                                                                   \
    if (PyErr_Occurred()) return nullptr;                                                 \
  }
  ENTRY_POINTS(BIND)
#undef BIND
  PyObject* check = PyMapping_GetItemString(table, "check");
  if (check == nullptr) return nullptr;
  Py_XDECREF(check_status);
  check_status = check;
  lib = bound;
  Py_RETURN_NONE;
}
PyObject* entry_points(PyObject*, PyObject*) {
  PyObject* names = PyList_New(0);
#define NAME(name)                                        \
  {                                                       \
    PyObject* s = PyUnicode_FromString(#name);            \
    PyList_Append(names, s);                              \
    Py_DECREF(s);                                         \
  }
  ENTRY_POINTS(NAME)
#undef NAME
  return names;
}

PyMethodDef methods[] = {
    {"gemm_fwd", (PyCFunction)(void (*)(void))gemm_fwd, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void (*)(void))backward, METH_FASTCALL, nullptr},
    {"bind", bind, METH_O, nullptr},
    {"entry_points", entry_points, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "axn_fast", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_axn_fast() {
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && (PyModule_AddIntConstant(m, "ABI_VERSION", AXN_ABI_VERSION) != 0 ||
                       PyModule_AddStringConstant(m, "BUILT_FOR", AXN_BUILT_FOR) != 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
