// The layer's forward and its autograd node in native code, over the C ABI of librzlinear.so.
//
// A training step of a small layer is five kernels of a few microseconds; carried by a Python
// autograd.Function — argument handling, ctypes conversions, tensor bookkeeping, and a backward that needs the
// interpreter lock in the autograd engine's own thread — its host side took 125 to 140 us (M = 128, K = N =
// 1024, forward + backward), against 36 us of kernels.  Here the forward is one call of the module
// function `apply`, and the backward is a torch::autograd::Node that runs in the engine's thread without the
// interpreter lock (except to fetch a layer plan that it has not met before, and a parameter's main_grad).
//
// `apply` serves the plain case — dense GPU tensors of one device and dtype, a [H] contiguous hashed_weight, the
// eight constants as an int32 CPU tensor, an ordinary eager call.  For everything else (tensor subclasses,
// any active functorch transform, tracing, forward-mode tangents, an empty batch, arguments that the launchers refuse)
// it returns None before it has done anything, and the caller goes through the Python Function, whose checks and errors are the
// reference's.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/DeviceGuard.h>
#include <ATen/SequenceNumber.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/HIPContextLight.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <array>
#include <map>
#include <memory>
#include <mutex>

#include "../../include/rzlinear.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---- the library's entry points, as the Python side has loaded them -----------------------------
struct Library {
  decltype(&rz_forward_hashed) forward = nullptr;
  decltype(&rz_forward_hashed_workspace_bytes) forward_workspace = nullptr;
  decltype(&rz_input_grad_hashed) input_grad = nullptr;
  decltype(&rz_input_grad_hashed_workspace_bytes) input_grad_workspace = nullptr;
  decltype(&rz_weight_grad_hashed) weight_grad = nullptr;
  decltype(&rz_weight_grad_planned) weight_grad_planned = nullptr;
  decltype(&rz_weight_grad_hashed_workspace_bytes) weight_grad_workspace = nullptr;
  decltype(&rz_linear_backward_hashed) backward = nullptr;
  decltype(&rz_linear_backward_hashed_dx_workspace_bytes) backward_dx_workspace = nullptr;
  decltype(&rz_plan_query) plan_query = nullptr;
};
Library lib;
PyObject* plan_provider = nullptr;    // Python: (K, N, H, BK, BN, constants, levels, device index) -> plan tensor, or None
PyObject* status_check = nullptr;     // Python: raises for a non-zero status
PyObject* function_node = nullptr;    // Python: the Function's own node for given saved tensors and arguments
// What the Python side's `tuning` context has set (tests, benchmarks): a copy, which a call that is under way
// in another thread keeps alive.
std::shared_ptr<const rz_tuning> tuning_in_force;
std::shared_ptr<const rz_tuning> current_tuning() { return std::atomic_load(&tuning_in_force); }

struct Geometry {
  int K, N, H, BK, BN;
  float scale;
  int32_t R[8];
};

// ---- small pieces -------------------------------------------------------------------------------
int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return RZ_F32;
    case at::kBFloat16: return RZ_BF16;
    case at::kHalf: return RZ_F16;
    default: return -1;
  }
}

// a dense tensor that nothing wraps (no subclass, functorch level, lazy conjugate ...)
bool plain(const Tensor& t) {
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Functionalize,
                                         c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  return t.defined() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped);
}
bool plain_gpu(const Tensor& t) { return plain(t) && t.is_cuda(); }

// a forward-mode tangent rides on it (the Function has no jvp and says so)
bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }

// unit column stride (copied only if it has to be) and the row pitch
Tensor rows(const Tensor& t, int64_t* ld) {
  const bool as_is = t.stride(1) == 1 && (t.size(0) == 1 || t.stride(0) >= t.size(1));
  Tensor r = as_is ? t : t.contiguous();
  *ld = r.size(0) > 1 ? r.stride(0) : std::max<int64_t>(r.size(1), 1);
  return r;
}

Tensor empty(at::IntArrayRef sizes, const Tensor& like) {
  return at::detail::empty_cuda(sizes, like.scalar_type(), like.device(), std::nullopt);
}

// scratch memory of one call, from the allocator that tensors come from (the caching one, unless the program has put
// another in its place): handed back, in stream order, when the call returns
at::DataPtr scratch(size_t bytes) { return bytes ? at::cuda::getCUDADeviceAllocator()->allocate(bytes) : at::DataPtr(); }

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// a non-zero status becomes the Python side's RzLinearError
void check(int status) {
  if (status == RZ_OK) return;
  PyGILState_STATE gil = PyGILState_Ensure();
  PyObject* r = PyObject_CallFunction(status_check, "i", status);
  python_error err;
  if (r == nullptr) err.persist();
  Py_XDECREF(r);
  PyGILState_Release(gil);
  if (r == nullptr) throw err;
  TORCH_CHECK(false, "librzlinear: status ", status);
}

// Lets go of the interpreter lock for its lifetime, if this thread holds it.
struct WithoutGil {
  PyThreadState* held = PyGILState_Check() ? PyEval_SaveThread() : nullptr;
  ~WithoutGil() {
    if (held != nullptr) PyEval_RestoreThread(held);
  }
};

// ---- layer plans --------------------------------------------------------------------------------
// Built and owned by the Python side (_lib.layer_plan); kept here too, so that a step need not ask for them
// with the interpreter lock.  Emptied by _lib.clear_layer_plans().  (Never destroyed: the tensors must not
// outlive the GPU runtime by a static destructor.)
typedef std::array<int32_t, 15> PlanKey;
std::mutex plans_mutex;
std::map<PlanKey, Tensor>& plans = *new std::map<PlanKey, Tensor>();

Tensor layer_plan(const Geometry& g, int device) {
  PlanKey key = {g.K, g.N, g.H, g.BK, g.BN, device};
  std::copy(g.R, g.R + 8, key.begin() + 6);
  {
    std::lock_guard<std::mutex> lock(plans_mutex);
    auto it = plans.find(key);
    if (it != plans.end()) return it->second;
  }
  PyGILState_STATE gil = PyGILState_Ensure();
  Tensor plan;
  PyObject* r = PyObject_CallFunction(plan_provider, "iiiii(iiiiiiii)ii", g.K, g.N, g.H, g.BK, g.BN, g.R[0], g.R[1], g.R[2], g.R[3],
                                      g.R[4], g.R[5], g.R[6], g.R[7], RZ_HASH_TWO_LEVEL, device);
  python_error err;
  if (r == nullptr) err.persist();
  else if (THPVariable_Check(r)) plan = THPVariable_Unpack(r);
  const bool none = r == Py_None;
  Py_XDECREF(r);
  PyGILState_Release(gil);
  if (r == nullptr) throw err;
  if (none) return plan;   // (this call has to do without one, see _lib.layer_plan_for_call)
  TORCH_CHECK(plan.defined(), "a layer plan must be a tensor");
  std::lock_guard<std::mutex> lock(plans_mutex);
  plans.emplace(key, plan);
  return plan;
}

// ---- the three calls ----------------------------------------------------------------------------
int forward(const Geometry& g, const Tensor& input, const Tensor& hw, const Tensor& bias, Tensor* output) {
  at::DeviceGuard guard(input.device());
  int64_t ldx;
  const Tensor x = rows(input, &ldx);
  const int M = (int)x.size(0), code = dtype_code(x.scalar_type());
  *output = empty({M, g.N}, x);
  const std::shared_ptr<const rz_tuning> keep = current_tuning();
  const rz_tuning* t = keep.get();
  // (skinny problems cut the contraction and need a scratch buffer for the slices)
  const size_t need = lib.forward_workspace(M, g.K, g.N, g.H, g.BK, g.BN, code, t);
  const at::DataPtr ws = scratch(need);
  return lib.forward(x.data_ptr(), hw.data_ptr(), bias.defined() ? bias.data_ptr() : nullptr, output->data_ptr(), ws.get(), need, M,
                     g.K, g.N, g.H, g.BK, g.BN, g.R, RZ_HASH_TWO_LEVEL, g.scale, ldx, g.N, code, t, stream_of(x));
}

Tensor input_grad(const Geometry& g, const Tensor& dy, int64_t lddy, const Tensor& hw) {
  const int M = (int)dy.size(0), code = dtype_code(dy.scalar_type());
  Tensor dx = empty({M, g.K}, dy);
  const std::shared_ptr<const rz_tuning> keep = current_tuning();
  const rz_tuning* t = keep.get();
  const size_t need = lib.input_grad_workspace(M, g.K, g.N, g.H, g.BK, g.BN, code, t);
  const at::DataPtr ws = scratch(need);
  check(lib.input_grad(dy.data_ptr(), hw.data_ptr(), dx.data_ptr(), ws.get(), need, M, g.K, g.N, g.H, g.BK, g.BN, g.R,
                       RZ_HASH_TWO_LEVEL, g.scale, lddy, g.K, code, t, stream_of(dy)));
  return dx;
}

// (hw defined: the input gradient too, into *dx)
void weight_grad(const Geometry& g, const Tensor& input, const Tensor& dy, int64_t lddy, const Tensor& out, bool accumulate,
                 const Tensor& dbias, bool with_plans, const Tensor& hw, Tensor* dx) {
  int64_t ldx;
  const Tensor x = rows(input, &ldx);
  const int M = (int)x.size(0), code = dtype_code(dy.scalar_type());
  unsigned flags = accumulate ? RZ_WG_ACCUMULATE : 0u;
  if (out.scalar_type() == at::kFloat) flags |= RZ_WG_DHW_F32;
  const int with_dbias = dbias.defined() ? 1 : 0;
  const std::shared_ptr<const rz_tuning> keep = current_tuning();
  const rz_tuning* t = keep.get();
  // (a layer plan: where the library would work by windows of dHW, or fold stored tiles into it)
  Tensor plan;
  if (with_plans) {
    int32_t q[8] = {0};
    check(lib.plan_query(2, M, g.K, g.N, g.H, g.BK, g.BN, code, flags | RZ_PLAN_WITH_LAYER_PLAN, with_dbias, t, q));
    if (q[4] == 4 || q[4] == 5) plan = layer_plan(g, dy.device().index());
  }
  const size_t need = lib.weight_grad_workspace(M, g.K, g.N, g.H, g.BK, g.BN, code, flags, with_dbias, t);
  const at::DataPtr ws = scratch(need);
  void* db = dbias.defined() ? dbias.data_ptr() : nullptr;
  if (hw.defined()) {
    *dx = empty({M, g.K}, dy);
    const size_t need_dx = lib.backward_dx_workspace(M, g.K, g.N, g.H, g.BK, g.BN, code, flags | (plan.defined() ? RZ_PLAN_WITH_LAYER_PLAN : 0u),
                                                     with_dbias, t);
    const at::DataPtr ws_dx = scratch(need_dx);
    check(lib.backward(x.data_ptr(), dy.data_ptr(), hw.data_ptr(), dx->data_ptr(), out.data_ptr(), db, ws_dx.get(), need_dx, ws.get(), need,
                       plan.defined() ? plan.data_ptr<int32_t>() : nullptr, plan.defined() ? (size_t)plan.numel() * 4 : 0, M, g.K, g.N, g.H,
                       g.BK, g.BN, g.R, RZ_HASH_TWO_LEVEL, g.scale, ldx, lddy, g.K, code, flags, t, stream_of(dy)));
  } else if (plan.defined())
    check(lib.weight_grad_planned(x.data_ptr(), dy.data_ptr(), out.data_ptr(), db, ws.get(), need, plan.data_ptr<int32_t>(),
                                  (size_t)plan.numel() * 4, M, g.K, g.N, g.H, g.BK, g.BN, g.R, RZ_HASH_TWO_LEVEL, g.scale, ldx, lddy,
                                  code, flags, t, stream_of(dy)));
  else
    check(lib.weight_grad(x.data_ptr(), dy.data_ptr(), out.data_ptr(), db, ws.get(), need, M, g.K, g.N, g.H, g.BK, g.BN, g.R,
                          RZ_HASH_TWO_LEVEL, g.scale, ldx, lddy, code, flags, t, stream_of(dy)));
}

// ---- the autograd node --------------------------------------------------------------------------
// An edge and a gradient for every tensor that the Function is given, the hash constants among them, which never need
// one: these are the positions that a hook on the node sees.
enum { kInput = 0, kWeight = 1, kBias = 3 };   // (2: the hash constants)

struct RzLinearNode : public Node {
  SavedVariable input, hashed_weight, random_numbers;   // (what the Function saves, whichever gradients are wanted)
  Geometry g;
  c10::SmallVector<int64_t, 2> output_sizes;
  at::TensorOptions output_options;
  bool fuse_grad_accumulation = false, with_plans = true;
  // (compiled autograd only) the node that the Function would have left here
  std::shared_ptr<Node> of_function;

  std::string name() const override { return "RzLinearFunctionBackward"; }

  void release_variables() override {
    std::shared_ptr<Node> other;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      input.reset_data();
      hashed_weight.reset_data();
      random_numbers.reset_data();
      other.swap(of_function);
    }
    if (other) other->release_variables();
  }

  // Compiled autograd does not run a node: it collects what the node has saved and records a call of its backward.
  // The Function's node can be taken apart like that, so one is made, with the same edges, and stands in for this one.
  void compiled_args(torch::dynamo::autograd::CompiledNodeArgs& args) const override { const_cast<RzLinearNode*>(this)->function_twin().compiled_args(args); }
  variable_list apply_with_saved(const variable_list& inputs, torch::dynamo::autograd::SwapSavedVariables& saved) override {
    return function_twin().apply_with_saved(inputs, saved);
  }
  Node& function_twin() {
    if (of_function) return *of_function;
    const variable_list kept = saved();
    const bool has_bias = num_outputs() > kBias;
    PyGILState_STATE gil = PyGILState_Ensure();
    PyObject* r = PyObject_CallFunction(function_node, "NNNifiiOOO", THPVariable_Wrap(kept[0]), THPVariable_Wrap(kept[1]), THPVariable_Wrap(kept[2]),
                                        g.N, g.scale, g.BK, g.BN, has_bias ? Py_True : Py_False,
                                        has_bias && should_compute_output(kBias) ? Py_True : Py_False, fuse_grad_accumulation ? Py_True : Py_False);
    python_error err;
    if (r == nullptr) err.persist();
    else if (THPVariable_Check(r)) of_function = THPVariable_Unpack(r).grad_fn();
    Py_XDECREF(r);
    PyGILState_Release(gil);
    if (r == nullptr) throw err;
    TORCH_CHECK(of_function, "the Function left no node");
    of_function->set_next_edges(torch::autograd::edge_list(next_edges()));
    return *of_function;
  }

  // input, hashed_weight and the hash constants (an error if they have been freed, or changed in place since the forward)
  variable_list saved() {
    const WithoutGil released;   // (a saved-tensor hook of the thread that holds the mutex may be waiting for it)
    std::lock_guard<std::mutex> lock(mutex_);   // (another thread's backward through this graph may release them)
    return {input.unpack(), hashed_weight.unpack(), random_numbers.unpack()};
  }

  // What a saved-tensor hook hands back, and a gradient, may be anything: the pointers below go straight to kernels.
  void require(const Tensor& t, const char* name, int64_t rows, int64_t cols, const Tensor& grad) const {
    TORCH_CHECK(plain_gpu(t), "rzlinear_amd: ", name, " of the backward must be a plain dense tensor on a ROCm GPU");
    TORCH_CHECK(t.device() == grad.device(), "rzlinear_amd: tensors on different devices (", t.device(), ", ", grad.device(), ")");
    TORCH_CHECK_TYPE(t.scalar_type() == grad.scalar_type(), name, " is ", t.scalar_type(), " but output_grad is ", grad.scalar_type());
    TORCH_CHECK_VALUE(cols < 0 ? (t.dim() == 1 && t.size(0) == rows) : (t.dim() == 2 && t.size(0) == rows && t.size(1) == cols),
                      "rzlinear_amd: ", name, " of the backward has shape ", t.sizes());
  }

  // The gradient buffer of a parameter whose weight gradient is added in the kernels: its main_grad if it
  // carries one, else its .grad (the first layer to reach a parameter without one overwrites a fresh buffer).
  Tensor fused_target(Tensor& hw, bool* accumulate) {
    *accumulate = true;
    PyGILState_STATE gil = PyGILState_Ensure();
    PyObject* self = THPVariable_Wrap(hw);
    PyObject* main = self != nullptr ? PyObject_GetAttrString(self, "main_grad") : nullptr;
    if (main == nullptr) PyErr_Clear();
    const bool other = main != nullptr && main != Py_None && !THPVariable_Check(main);
    Tensor target;
    if (main != nullptr && main != Py_None && !other) target = THPVariable_Unpack(main);
    Py_XDECREF(main);
    Py_XDECREF(self);
    PyGILState_Release(gil);
    TORCH_CHECK_TYPE(!other, "main_grad must be a tensor");
    if (!target.defined()) {
      if (!hw.grad().defined()) {
        hw.mutable_grad() = at::empty_like(hw.detach());
        *accumulate = false;
      }
      target = hw.grad();
    }
    TORCH_CHECK(target.is_cuda() && target.device() == hw.device(), "rzlinear_amd: the gradient buffer must be on ", hw.device());
    TORCH_CHECK_VALUE(target.dim() == 1 && target.size(0) == g.H && target.is_contiguous(), "out must be a contiguous tensor of ", g.H, " elements");
    TORCH_CHECK_TYPE(target.scalar_type() == at::kFloat || target.scalar_type() == hw.scalar_type(), "out must be float32 or ", hw.scalar_type());
    return target;
  }

  variable_list apply(variable_list&& grads) override {
    // (a fused weight gradient reaches its buffer in every backward through the layer, whichever gradients that backward
    //  returns: autograd is not handed it and cannot ask for it)
    const bool need_input = task_should_compute_output(kInput), need_bias = num_outputs() > kBias && task_should_compute_output(kBias),
               need_weight = fuse_grad_accumulation ? should_compute_output(kWeight) : task_should_compute_output(kWeight);
    variable_list result(num_outputs());
    Tensor bias_grad;
    const variable_list kept = saved();
    const Tensor& x = kept[0];
    Tensor hw = kept[1];
    Tensor grad = grads[0].defined() ? grads[0] : at::zeros(output_sizes, output_options);
    require(grad, "output_grad", output_sizes[0], g.N, grad);
    if (need_input) require(hw, "hashed_weight", g.H, -1, grad);
    if (need_weight) require(x, "input", output_sizes[0], g.K, grad);
    at::DeviceGuard guard(grad.device());
    int64_t lddy;
    const Tensor dy = rows(grad, &lddy);
    if (need_input && !need_weight) result[kInput] = input_grad(g, dy, lddy, hw.contiguous());
    if (need_weight) {   // (with a bias: one pass over dy yields both gradients)
      if (need_bias) bias_grad = empty({g.N}, dy);
      bool accumulate = false;
      Tensor out;
      if (fuse_grad_accumulation) {
        out = fused_target(hw, &accumulate);
      } else {
        out = result[kWeight] = empty({g.H}, dy);
      }
      try {
        weight_grad(g, x, dy, lddy, out, accumulate, bias_grad, with_plans, need_input ? hw.contiguous() : Tensor(), &result[kInput]);
      } catch (...) {   // (nothing has been written to a fresh buffer: the next backward must not add to it)
        if (fuse_grad_accumulation && !accumulate) hw.mutable_grad() = Tensor();
        throw;
      }
    } else if (need_bias) {
      bias_grad = grad.sum(0);
    }
    if (need_bias) result[kBias] = std::move(bias_grad);
    return result;
  }
};

// ---- the node as Python sees it: grad_fn of the layer's output ----------------------------------
PyObject* saved_tensors(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  auto* node = static_cast<RzLinearNode*>(reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata.get());
  const variable_list kept = node->saved();
  return Py_BuildValue("NNN", THPVariable_Wrap(kept[0]), THPVariable_Wrap(kept[1]), THPVariable_Wrap(kept[2]));
  END_HANDLE_TH_ERRORS
}

PyTypeObject node_type;

bool register_node_type(PyObject* module) {
  using namespace torch::autograd;
  static PyGetSetDef properties[] = {THP_FUNCTION_DEFAULT_PROPERTIES,
                                     {"saved_tensors", saved_tensors, nullptr, "what the forward kept for the backward", nullptr},
                                     {nullptr, nullptr, nullptr, nullptr, nullptr}};
  if (_initFunctionPyTypeObject(node_type, "RzLinearFunctionBackward", properties, nullptr) == nullptr) return false;
  registerCppFunction(typeid(RzLinearNode), &node_type);
  return PyModule_AddObjectRef(module, "RzLinearFunctionBackward", reinterpret_cast<PyObject*>(&node_type)) == 0;
}

// ---- apply(input, hashed_weight, random_numbers, output_dim, init_factor, BK, BN, bias, fuse, with_plans) ----
PyObject* apply(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) {
    PyErr_SetString(PyExc_TypeError, "apply takes 10 arguments");
    return nullptr;
  }
  if (!THPVariable_Check(args[0]) || !THPVariable_Check(args[1]) || !THPVariable_Check(args[2])) Py_RETURN_NONE;
  const bool has_bias = args[7] != Py_None;
  if (has_bias && !THPVariable_Check(args[7])) Py_RETURN_NONE;
  const Tensor& x = THPVariable_Unpack(args[0]);
  const Tensor& hw = THPVariable_Unpack(args[1]);
  const Tensor& r = THPVariable_Unpack(args[2]);
  const Tensor bias = has_bias ? THPVariable_Unpack(args[7]) : Tensor();
  if (!plain_gpu(x) || !plain_gpu(hw) || (has_bias && !plain_gpu(bias)) || !plain(r) || lib.forward == nullptr) Py_RETURN_NONE;
  if (has_tangent(x) || has_tangent(hw) || has_tangent(bias)) Py_RETURN_NONE;
  if (c10::impl::dispatch_mode_enabled() || torch::jit::tracer::isTracing()) Py_RETURN_NONE;
  // (inside a functorch transform — the key is included as long as there is one — the Function, which has no rule for
  //  any, refuses every call, also one whose tensors the transform does not wrap)
  if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode)) Py_RETURN_NONE;
  const auto type = x.scalar_type();
  if (dtype_code(type) < 0 || hw.scalar_type() != type || hw.device() != x.device() || x.dim() != 2 || hw.dim() != 1 || !hw.is_contiguous()) Py_RETURN_NONE;
  if (!r.device().is_cpu() || r.scalar_type() != at::kInt || r.dim() != 1 || r.numel() != 8 || !r.is_contiguous()) Py_RETURN_NONE;
  long v[3];   // output_dim, BK, BN
  for (int i = 0; i < 3; i++) {
    PyObject* o = args[i == 0 ? 3 : i + 4];
    if (!PyLong_Check(o)) Py_RETURN_NONE;
    v[i] = PyLong_AsLong(o);
    if (v[i] == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
  }
  const double scale = PyFloat_AsDouble(args[4]);
  if (scale == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int64_t M = x.size(0), K = x.size(1), N = v[0], H = hw.size(0), BK = v[1], BN = v[2];
  if (M < 1 || M > INT32_MAX || K < 1 || K > INT32_MAX || N < 1 || N > INT32_MAX || H > INT32_MAX || BK < 1 || BK > 256 || BN < 1 || BN > 256 || H <= BK * BN) Py_RETURN_NONE;
  if (has_bias && (bias.scalar_type() != type || bias.device() != x.device() || bias.dim() != 1 || bias.numel() != N || !bias.is_contiguous())) Py_RETURN_NONE;
  const int fuse = PyObject_IsTrue(args[8]), with_plans = PyObject_IsTrue(args[9]);
  if (fuse < 0 || with_plans < 0) return nullptr;

  Geometry g = {(int)K, (int)N, (int)H, (int)BK, (int)BN, (float)scale, {}};
  std::copy(r.data_ptr<int32_t>(), r.data_ptr<int32_t>() + 8, g.R);
  Tensor output;
  int status;
  // what a profiler sees: the Function's name and arguments (the backward is named by the node)
  at::RecordFunction event(at::RecordScope::FUNCTION);
  if (event.isActive()) {
    const c10::IValue none;
    const std::array<c10::IValue, 10> inputs = {x, hw, r, none, none, none, none, none, has_bias ? c10::IValue(bias) : none, none};
    at::detail::record_function_with_scope(event, "RzLinearFunction", inputs, (int64_t)at::sequence_number::peek());
  }
  {
    PyThreadState* saved = PyEval_SaveThread();   // (a full launch queue makes the runtime wait)
    try {
      status = forward(g, x, hw, bias, &output);
      if (status == RZ_OK && torch::autograd::compute_requires_grad(x, hw, bias)) {
        auto node = std::shared_ptr<RzLinearNode>(new RzLinearNode(), torch::autograd::deleteNode);
        node->set_next_edges(has_bias ? torch::autograd::collect_next_edges(x, hw, r, bias) : torch::autograd::collect_next_edges(x, hw, r));
        node->input = SavedVariable(x, false);
        node->hashed_weight = SavedVariable(hw, false);
        node->random_numbers = SavedVariable(r, false);
        node->g = g;
        node->output_sizes = {M, N};
        node->output_options = x.options();
        node->fuse_grad_accumulation = fuse != 0;
        node->with_plans = with_plans != 0;
        torch::autograd::set_history(output, node);
      }
    } catch (...) {
      PyEval_RestoreThread(saved);
      throw;
    }
    PyEval_RestoreThread(saved);
  }
  if (status != RZ_OK) Py_RETURN_NONE;   // (nothing was launched: the Python path meets the same refusal and reports it)
  return THPVariable_Wrap(std::move(output));
  END_HANDLE_TH_ERRORS
}

// bind({entry point: address}, plan_provider, status_check, function_node)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *table, *provider, *checker, *maker;
  if (!PyArg_ParseTuple(args, "O!OOO", &PyDict_Type, &table, &provider, &checker, &maker)) return nullptr;
  auto address = [&](const char* name) -> void* {
    PyObject* o = PyDict_GetItemString(table, name);
    if (o == nullptr) PyErr_Format(PyExc_KeyError, "no address for %s", name);
    return o == nullptr ? nullptr : PyLong_AsVoidPtr(o);
  };
  Library l;
#define RZ_BIND(field, name) \
  if ((l.field = reinterpret_cast<decltype(l.field)>(address(#name))) == nullptr) return nullptr
  RZ_BIND(forward, rz_forward_hashed);
  RZ_BIND(forward_workspace, rz_forward_hashed_workspace_bytes);
  RZ_BIND(input_grad, rz_input_grad_hashed);
  RZ_BIND(input_grad_workspace, rz_input_grad_hashed_workspace_bytes);
  RZ_BIND(weight_grad, rz_weight_grad_hashed);
  RZ_BIND(weight_grad_planned, rz_weight_grad_planned);
  RZ_BIND(weight_grad_workspace, rz_weight_grad_hashed_workspace_bytes);
  RZ_BIND(backward, rz_linear_backward_hashed);
  RZ_BIND(backward_dx_workspace, rz_linear_backward_hashed_dx_workspace_bytes);
  RZ_BIND(plan_query, rz_plan_query);
#undef RZ_BIND
  Py_INCREF(provider);
  Py_INCREF(checker);
  Py_INCREF(maker);
  Py_XDECREF(plan_provider);
  Py_XDECREF(status_check);
  Py_XDECREF(function_node);
  plan_provider = provider;
  status_check = checker;
  function_node = maker;
  lib = l;
  Py_RETURN_NONE;
}

// set_tuning(address of a live rz_tuning, or 0)
PyObject* set_tuning(PyObject*, PyObject* arg) {
  void* p = PyLong_AsVoidPtr(arg);
  if (p == nullptr && PyErr_Occurred()) return nullptr;
  std::atomic_store(&tuning_in_force, p == nullptr ? std::shared_ptr<const rz_tuning>()
                                                   : std::make_shared<const rz_tuning>(*static_cast<const rz_tuning*>(p)));
  Py_RETURN_NONE;
}

PyObject* clear_plans(PyObject*, PyObject*) {
  std::map<PlanKey, Tensor> gone;
  {
    std::lock_guard<std::mutex> lock(plans_mutex);
    gone.swap(plans);
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"apply", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(apply)), METH_FASTCALL,
     "forward of the layer with its autograd node, or None where the Python Function has to take the call"},
    {"bind", bind, METH_VARARGS, "take the entry points of librzlinear.so"},
    {"set_tuning", set_tuning, METH_O, "address of the rz_tuning overrides in force, or 0"},
    {"clear_plans", clear_plans, METH_NOARGS, "forget the layer plans"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef definition = {PyModuleDef_HEAD_INIT, "_native", "native host path of the layer", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  PyObject* module = PyModule_Create(&definition);
  if (module != nullptr && !register_node_type(module)) Py_CLEAR(module);
  return module;
}
