// The host path of an ordinary call in native code: argument checks, plan and
// workspace lookup, output allocation and the C entry point's call, for calls
// that need nothing else.  Everything here answers "not mine" (None) for any
// other call -- an argument the Python layer would reject or convert in a way
// of its own, tensors of another device than the current one, a capture in
// progress, tracing or tensor modes, tuning environment variables, a shape or
// stream seen for the first time -- and the Python layer then does what it
// always did.  A one-token call spent 27 us in Python for 15 us of kernels.
//
// Plans (dispatch choices and workspace bytes by shape) and workspaces (by
// device and stream) come from the Python layer: it registers a plan after its
// own path has run the shape once (kept until tuning.reload_tables()), shows
// every eager buffer its pool makes, and clears them here when the pool drops
// its own.  All state is read and written with the GIL held.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cstdlib>
#include <tuple>
#include <unordered_map>

#include "../../include/w4a16_moe.h"

namespace {

struct PlanKey {
  int64_t dev, M, topk, E, N, K, group;
  bool operator==(const PlanKey& o) const {
    return dev == o.dev && M == o.M && topk == o.topk && E == o.E && N == o.N && K == o.K &&
           group == o.group;
  }
};
struct PlanHash {
  size_t operator()(const PlanKey& k) const {
    uint64_t h = 1469598103934665603ull;
    for (int64_t v : {k.dev, k.M, k.topk, k.E, k.N, k.K, k.group})
      h = (h ^ (uint64_t)v) * 1099511628211ull;
    return (size_t)h;
  }
};
struct Plan {
  size_t ws_bytes;
  bool has_tuning;
  w4a16_moe_tuning tuning;
};
// Batch sizes a serving program meets; past the bound the plans start over.
constexpr size_t kMaxPlans = 4096;
std::unordered_map<PlanKey, Plan, PlanHash>& plans() {
  static auto* p = new std::unordered_map<PlanKey, Plan, PlanHash>();
  return *p;
}
struct WsKey {
  int64_t dev, stream;
  bool operator==(const WsKey& o) const { return dev == o.dev && stream == o.stream; }
};
struct WsHash {
  size_t operator()(const WsKey& k) const {
    return std::hash<int64_t>()(k.stream) * 31 + (size_t)k.dev;
  }
};
std::unordered_map<WsKey, at::Tensor, WsHash>& workspaces() {  // never destroyed: no GPU frees at exit
  static auto* p = new std::unordered_map<WsKey, at::Tensor, WsHash>();
  return *p;
}

// Modes under which an operator call means something else than running it.
bool plain_mode() {
  return !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled() &&
         !at::tracer::impl::is_dispatch_enabled();
}

// An ordinary tensor of the current device with storage of its own (no
// subclass, no batched, functionalized, conjugated or other wrapper).
bool plain(PyObject* o, int64_t dev, at::Tensor* out) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return false;
  using c10::DispatchKey;
  constexpr c10::DispatchKeySet wrappers({DispatchKey::FuncTorchBatched, DispatchKey::Batched,
                                          DispatchKey::FuncTorchGradWrapper,
                                          DispatchKey::Functionalize, DispatchKey::Python,
                                          DispatchKey::Conjugate, DispatchKey::Negative,
                                          DispatchKey::ZeroTensor});
  if (t.key_set().has_any(wrappers) || t.get_device() != dev) return false;
  *out = t;
  return true;
}

// (asked first: nothing here touches the HIP runtime for host tensors)
bool on_gpu(PyObject* o) { return THPVariable_CheckExact(o) && THPVariable_Unpack(o).is_cuda(); }

bool as_int(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool aligned(const at::Tensor& t, uintptr_t a) {
  return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % a == 0;
}

bool env_set(const char* name) {
  const char* v = std::getenv(name);
  return v && *v;
}

// The call's stream, or false while it is being captured.
bool eager_stream(int64_t dev, hipStream_t* s) {
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None)
    return false;
  *s = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
  return true;
}

at::Tensor to_i32(const at::Tensor& ids) {
  return (ids.scalar_type() == at::kInt ? ids : ids.to(at::kInt)).contiguous();
}

// fused(hidden, w1_q, w2_q, w1_scale, w2_scale, topk_weights, topk_ids, group)
// -> tensor, a status (int) of the C entry point, or None (not mine).
PyObject* py_fused(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 8 || !on_gpu(args[0]) || !plain_mode()) Py_RETURN_NONE;
  const int64_t dev = c10::hip::current_device();
  at::Tensor x, w1, w2, s1, s2, tw, ti;
  int64_t group;
  if (!plain(args[0], dev, &x) || !plain(args[1], dev, &w1) || !plain(args[2], dev, &w2) ||
      !plain(args[3], dev, &s1) || !plain(args[4], dev, &s2) || !plain(args[5], dev, &tw) ||
      !plain(args[6], dev, &ti) || !as_int(args[7], &group))
    Py_RETURN_NONE;
  if (x.dim() != 2 || w1.dim() != 3 || w2.dim() != 3 || s1.dim() != 3 || s2.dim() != 3 ||
      ti.dim() != 2 || tw.dim() != 2)
    Py_RETURN_NONE;
  auto per_elt = [](const at::Tensor& w) -> int64_t {
    const auto d = w.scalar_type();
    return d == at::kInt ? 8 : d == at::kByte || d == at::kChar ? 2 : 0;
  };
  const int64_t M = x.size(0), K = x.size(1), E = w1.size(0), N = w1.size(1) / 2;
  const int64_t topk = ti.size(1);
  if (M < 1 || group < 1 || x.scalar_type() != at::kBFloat16 || w1.size(1) % 2 ||
      w1.size(2) * per_elt(w1) != K || w2.size(0) != E || w2.size(1) != K ||
      w2.size(2) * per_elt(w2) != N || K % group || N % group || K == 0 || N == 0)
    Py_RETURN_NONE;
  if (s1.scalar_type() != at::kBFloat16 || s2.scalar_type() != at::kBFloat16 || s1.size(0) != E ||
      s1.size(1) != 2 * N || s1.size(2) != K / group || s2.size(0) != E || s2.size(1) != K ||
      s2.size(2) != N / group)
    Py_RETURN_NONE;
  if (!w1.is_contiguous() || !w2.is_contiguous() || !s1.is_contiguous() || !s2.is_contiguous())
    Py_RETURN_NONE;
  if (ti.sizes() != tw.sizes() || ti.size(0) != M || topk < 1 ||
      (ti.scalar_type() != at::kInt && ti.scalar_type() != at::kLong) ||
      !at::isFloatingType(tw.scalar_type()))
    Py_RETURN_NONE;
  if (x.stride(1) != 1 || x.stride(0) % 8 != 0 || !aligned(x, 16)) Py_RETURN_NONE;
  if (env_set("W4A16_MOE_TUNING") || env_set("W4A16_MOE_CONFIG_DIR")) Py_RETURN_NONE;
  hipStream_t stream;
  if (!eager_stream(dev, &stream)) Py_RETURN_NONE;
  const auto plan_it = plans().find(PlanKey{dev, M, topk, E, N, K, group});
  if (plan_it == plans().end()) Py_RETURN_NONE;
  const Plan plan = plan_it->second;
  const auto ws_it = workspaces().find(WsKey{dev, (int64_t)(intptr_t)stream});
  if (ws_it == workspaces().end()) Py_RETURN_NONE;
  const at::Tensor ws = ws_it->second;  // held for the call
  if ((size_t)ws.numel() < plan.ws_bytes) Py_RETURN_NONE;
  const at::Tensor ids = to_i32(ti);
  const at::Tensor wts = (tw.scalar_type() == at::kFloat ? tw : tw.to(at::kFloat)).contiguous();
  const at::Tensor out =
      at::empty({M, K}, at::TensorOptions().dtype(at::kBFloat16).device(x.device()));
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = w4a16_moe_fused_experts_ex(
      x.const_data_ptr(), x.stride(0), w1.const_data_ptr(), w2.const_data_ptr(),
      s1.const_data_ptr(), s2.const_data_ptr(), static_cast<const float*>(wts.const_data_ptr()),
      static_cast<const int32_t*>(ids.const_data_ptr()), M, topk, E, N, K, group,
      out.mutable_data_ptr(), out.stride(0), ws.mutable_data_ptr(), (size_t)ws.numel(), stream,
      plan.has_tuning ? &plan.tuning : nullptr);
  Py_END_ALLOW_THREADS
  if (st != W4A16_OK) return PyLong_FromLong(st);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// router(logits, topk, renormalize) -> (weights, ids), a status, or None.
PyObject* py_router(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 3 || !on_gpu(args[0]) || !plain_mode()) Py_RETURN_NONE;
  const int64_t dev = c10::hip::current_device();
  at::Tensor x;
  int64_t k;
  if (!plain(args[0], dev, &x) || !as_int(args[1], &k) || !PyBool_Check(args[2])) Py_RETURN_NONE;
  const auto dt = x.scalar_type();
  if (x.dim() != 2 || k < 1 || (dt != at::kFloat && dt != at::kBFloat16) || x.stride(1) != 1)
    Py_RETURN_NONE;
  const int64_t M = x.size(0), E = x.size(1);
  if (M < 1) Py_RETURN_NONE;
  const auto opt = at::TensorOptions().device(x.device());
  const at::Tensor w = at::empty({M, k}, opt.dtype(at::kFloat));
  const at::Tensor ids = at::empty({M, k}, opt.dtype(at::kInt));
  const hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = w4a16_moe_router_topk_softmax(
      x.const_data_ptr(), dt == at::kFloat ? W4A16_LOGITS_F32 : W4A16_LOGITS_BF16,
      M > 1 ? x.stride(0) : E, M, E, k, args[2] == Py_True ? 1 : 0,
      static_cast<float*>(w.mutable_data_ptr()), static_cast<int32_t*>(ids.mutable_data_ptr()),
      stream);
  Py_END_ALLOW_THREADS
  if (st != W4A16_OK) return PyLong_FromLong(st);
  PyObject* r = PyTuple_New(2);
  if (!r) throw python_error();
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(w));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(ids));
  return r;
  END_HANDLE_TH_ERRORS
}

// align(topk_ids, block, E) -> (sorted, experts, num_post), a status, or None.
PyObject* py_align(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 3 || !on_gpu(args[0]) || !plain_mode()) Py_RETURN_NONE;
  const int64_t dev = c10::hip::current_device();
  at::Tensor ti;
  int64_t block, E;
  if (!plain(args[0], dev, &ti) || !as_int(args[1], &block) || !as_int(args[2], &E) ||
      ti.dim() != 2 || (ti.scalar_type() != at::kInt && ti.scalar_type() != at::kLong))
    Py_RETURN_NONE;
  const int64_t M = ti.size(0), topk = ti.size(1);
  int64_t em = 0, nb = 0;
  size_t scratch_bytes = 0;
  int st = w4a16_moe_align_sizes(M, topk, E, block, &em, &nb);
  if (st == W4A16_OK) st = w4a16_moe_align_scratch_size(M, topk, E, &scratch_bytes);
  if (st != W4A16_OK) return PyLong_FromLong(st);
  const at::Tensor ids = to_i32(ti);
  const auto opt = at::TensorOptions().dtype(at::kInt).device(ti.device());
  const at::Tensor sorted = at::empty({em}, opt), experts = at::empty({nb}, opt);
  const at::Tensor num_post = at::empty({1}, opt);
  at::Tensor scratch;
  if (scratch_bytes) scratch = at::empty({(int64_t)((scratch_bytes + 3) / 4)}, opt);
  const hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
  Py_BEGIN_ALLOW_THREADS
  st = w4a16_moe_align_block_size_ws(static_cast<const int32_t*>(ids.const_data_ptr()), M, topk, E, block,
                 static_cast<int32_t*>(sorted.mutable_data_ptr()),
                 static_cast<int32_t*>(experts.mutable_data_ptr()),
                 static_cast<int32_t*>(num_post.mutable_data_ptr()), nullptr, nullptr,
                 scratch.defined() ? scratch.mutable_data_ptr() : nullptr, scratch_bytes, stream);
  Py_END_ALLOW_THREADS
  if (st != W4A16_OK) return PyLong_FromLong(st);
  PyObject* r = PyTuple_New(3);
  if (!r) throw python_error();
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(sorted));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(experts));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(num_post));
  return r;
  END_HANDLE_TH_ERRORS
}

// has_plan(dev, M, topk, E, N, K, group)
PyObject* py_has_plan(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  int64_t v[7];
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "has_plan takes 7 integers");
    return nullptr;
  }
  for (int i = 0; i < 7; ++i)
    if (!as_int(args[i], &v[i])) Py_RETURN_FALSE;
  return PyBool_FromLong(plans().count(PlanKey{v[0], v[1], v[2], v[3], v[4], v[5], v[6]}) != 0);
}

// set_plan(dev, M, topk, E, N, K, group, ws_bytes, tuning fields or None)
PyObject* py_set_plan(PyObject*, PyObject* args) {
  long long dev, M, topk, E, N, K, group, bytes;
  PyObject* t;
  if (!PyArg_ParseTuple(args, "LLLLLLLLO", &dev, &M, &topk, &E, &N, &K, &group, &bytes, &t))
    return nullptr;
  Plan p{(size_t)bytes, t != Py_None, {}};
  if (p.has_tuning &&
      !PyArg_ParseTuple(t, "iiiiiiii", &p.tuning.gemv_only_max_m, &p.tuning.gemv_max_tokens,
                        &p.tuning.gemv_tokens_per_pass, &p.tuning.mfma_tile_m,
                        &p.tuning.gemv_units_per_wg, &p.tuning.gemv_lanes_per_row,
                        &p.tuning.w2_fused_max_m, &p.tuning.mfma_row_tiles))
    return nullptr;
  if (plans().size() >= kMaxPlans) plans().clear();
  plans()[PlanKey{dev, M, topk, E, N, K, group}] = p;
  Py_RETURN_NONE;
}

// set_workspace(dev, stream, tensor)
PyObject* py_set_workspace(PyObject*, PyObject* args) {
  long long dev, stream;
  PyObject* t;
  if (!PyArg_ParseTuple(args, "LLO", &dev, &stream, &t)) return nullptr;
  if (!THPVariable_Check(t)) {
    PyErr_SetString(PyExc_TypeError, "workspace must be a tensor");
    return nullptr;
  }
  workspaces()[WsKey{dev, stream}] = THPVariable_Unpack(t);
  Py_RETURN_NONE;
}

PyObject* py_clear_workspaces(PyObject*, PyObject*) {
  workspaces().clear();
  Py_RETURN_NONE;
}

PyObject* py_clear_plans(PyObject*, PyObject*) {
  plans().clear();
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"fused", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_fused)),
     METH_FASTCALL, nullptr},
    {"router", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_router)),
     METH_FASTCALL, nullptr},
    {"align", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_align)),
     METH_FASTCALL, nullptr},
    {"has_plan", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_has_plan)),
     METH_FASTCALL, nullptr},
    {"set_plan", py_set_plan, METH_VARARGS, nullptr},
    {"set_workspace", py_set_workspace, METH_VARARGS, nullptr},
    {"clear_workspaces", py_clear_workspaces, METH_NOARGS, nullptr},
    {"clear_plans", py_clear_plans, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "w4a16_fastcall", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_w4a16_fastcall(void) {
  PyObject* m = PyModule_Create(&module);
  // checked against the running torch by the loader
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
