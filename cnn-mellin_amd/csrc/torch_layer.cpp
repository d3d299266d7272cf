// The layers' host path: argument checks, output and workspace allocation, the autograd node and
// the calls into libmellin_hip, as one CPython function.  A call of a small layer is bound by
// what the host does: through Python (torch.autograd.Function, ctypes, one call and one
// allocation per pass) a 1-D layer's forward took 30 us of host time and a training step of it
// 140-240 us for 7 launches; here a call takes 5 us with one launch and 8 with two, and a
// step 52 where the host bounds it.
//
// corr(kind, dims, input, weight, bias, s, d, p, u, r, activation) returns the output tensor, or
// None for whatever it does not handle (other element types, CPU tensors, arguments that are
// errors): mconv.py then takes its own path, which has the checks and their messages.
// stack(...) is the same for a stack of layers with ReLUs (conv_stack.py), whose tensors then stay
// in the kernels' own layout from layer to layer.
#include <ATen/ATen.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/mellin_hip.h"

namespace {

using at::Tensor;

struct Geometry {
  int kind;                              // AX_MCORR / AX_LCORR
  int64_t batch, c_in, c_out, nf[2], ng[2], nh[2], s[2], d[2], p[2], u[2];
};

#define GEOMETRY_ARGS(g)                                                                                             \
  (g).batch, (g).c_in, (g).c_out, (g).nf[0], (g).nf[1], (g).ng[0], (g).ng[1], (g).nh[0], (g).nh[1], (g).s[0], (g).s[1], \
      (g).d[0], (g).d[1], (g).p[0], (g).p[1], (g).u[0], (g).u[1]

void check(int code) {
  TORCH_CHECK(code == MELLIN_OK, "libmellin_hip: ", mellin_last_error(), " (code ", code, ")");
}

void *launch_stream(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

const void *pointer(const Tensor &t) { return t.defined() ? t.const_data_ptr() : nullptr; }

Tensor scratch(const Tensor &like, size_t bytes) {
  return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : Tensor();
}

// A layer's copy of its input in the kernels' layout, from its forward call to its backward call.  All that are alive on a device
// take no more than kMostKept bytes together, however many layers and graphs there are (four of the widest layers); behind
// that, and where memory runs out, a backward call lays its input out again, as where nothing is kept: the same bits, and the
// time of a pass over it (128 -> 256 channels, 3 x 3 taps, 32 x 256 x 41, half: 567 us a step instead of 498).
constexpr int64_t kMostKept = (int64_t)1 << 30;
constexpr int kDevices = 64;
std::atomic<int64_t> kept_bytes[kDevices];

struct KeptInput {
  Tensor bytes;
  KeptInput() = default;
  KeptInput(const KeptInput &) = delete;
  KeptInput &operator=(const KeptInput &) = delete;
  ~KeptInput() { reset(); }
  // (leaves `bytes` undefined where there is no room)
  void allocate(const Tensor &like, size_t size) {
    const int device = like.device().index();
    if (!size || device < 0 || device >= kDevices) return;
    if (kept_bytes[device].fetch_add((int64_t)size) + (int64_t)size > kMostKept) {
      kept_bytes[device].fetch_sub((int64_t)size);
      return;
    }
    device_ = device;
    size_ = (int64_t)size;
    try {
      bytes = scratch(like, size);
    } catch (const c10::OutOfMemoryError &) {
      reset();
    }
  }
  void reset() {
    bytes.reset();
    if (size_) kept_bytes[device_].fetch_sub(size_);
    size_ = 0;
  }

 private:
  int device_ = 0;
  int64_t size_ = 0;
};

// The gradients of out = activation(bias + correlation(input, weight)).
struct Corr2dBackward : public torch::autograd::Node {
  Geometry g;
  bool relu = false, has_bias = false;
  int elem = 4;                          // as the library's entry points take it
  at::ScalarType param_kind = at::kFloat;
  torch::autograd::SavedVariable input_, weight_, out_;
  std::shared_ptr<KeptInput> kept_;      // if the forward call left one
  std::vector<int64_t> out_sizes;
  at::TensorOptions options;

  std::string name() const override { return "Corr2dBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    kept_.reset();
    input_.reset_data();
    weight_.reset_data();
    out_.reset_data();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
    at::AutoGradMode no_grad(false);
    Tensor input, weight, out, kept;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (kept_) kept = kept_->bytes;
      input = input_.unpack();
      weight = weight_.unpack();
      if (relu) out = out_.unpack(shared_from_this());
    }
    Tensor grad_out = grads[0].defined() ? grads[0] : at::zeros(out_sizes, options);
    if (grad_out.scalar_type() != input.scalar_type()) grad_out = grad_out.to(input.scalar_type());
    grad_out = grad_out.contiguous();
    const c10::OptionalDeviceGuard guard(input.device());
    Tensor grad_input, grad_weight, grad_bias;
    int want = relu ? MELLIN_WANT_RELU : 0;
    if (task_should_compute_output(0)) { want |= MELLIN_WANT_INPUT; grad_input = at::empty_like(input, at::MemoryFormat::Contiguous); }
    if (task_should_compute_output(1)) { want |= MELLIN_WANT_WEIGHT; grad_weight = at::empty(weight.sizes(), weight.options().dtype(param_kind)); }
    if (has_bias && task_should_compute_output(2)) { want |= MELLIN_WANT_BIAS; grad_bias = at::empty({g.c_out}, weight.options().dtype(param_kind)); }
    if (want & ~MELLIN_WANT_RELU) {
      const size_t need = (kept.defined() ? mellin_layer_backward_kept_workspace : mellin_layer_backward_workspace)(g.kind, elem, want, GEOMETRY_ARGS(g));
      Tensor ws = scratch(input, need);
      check(mellin_layer_backward_kept(g.kind, elem, want, pointer(input), pointer(weight), pointer(grad_out), pointer(out),
                                       GEOMETRY_ARGS(g), grad_input.defined() ? grad_input.data_ptr() : nullptr,
                                       grad_weight.defined() ? grad_weight.data_ptr() : nullptr,
                                       grad_bias.defined() ? grad_bias.data_ptr() : nullptr, pointer(kept),
                                       ws.defined() ? ws.data_ptr() : nullptr, need, launch_stream(input)));
    }
    return {grad_input, grad_weight, grad_bias};
  }
};

// an int, or a tuple of `n` ints (1-D layers: n = 1, the second axis being a unit one with `unit`)
bool parse(PyObject *o, int n, int64_t unit, int64_t (&v)[2]) {
  v[1] = unit;
  if (PyLong_CheckExact(o)) {
    v[0] = PyLong_AsLongLong(o);
    if (n == 2) v[1] = v[0];
  } else if (PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) == n) {
    for (int i = 0; i < n; ++i) {
      PyObject *e = PyTuple_GET_ITEM(o, i);
      if (!PyLong_CheckExact(e)) return false;
      v[i] = PyLong_AsLongLong(e);
    }
  } else {
    return false;
  }
  if (PyErr_Occurred()) { PyErr_Clear(); return false; }
  for (int i = 0; i < n; ++i)
    if (v[i] > (1 << 30) || v[i] < -(1 << 30)) return false;
  return true;
}

int64_t floor_div(int64_t a, int64_t b) {
  const int64_t q = a / b;
  return (a % b != 0 && ((a < 0) != (b < 0))) ? q - 1 : q;
}

int64_t valid_size(int kind, int64_t nf, int64_t ng, int64_t s, int64_t d, int64_t p, int64_t u) {
  const int64_t v = kind == MELLIN_AXIS_MCORR ? floor_div((ng + u - 1) * (p + 1), nf + d - 1) - s + 1
                                              : floor_div(u * (ng - 1) - d * (nf - 1) + p, s) + 1;
  return v > 0 ? v : 0;
}

// Whether the library's float and half kernels take `t`: memory of its own as it lies (no wrapper of a function
// transform, no view that negates) and no tangent.
bool plain(const Tensor &t) {
  using K = c10::DispatchKey;
  constexpr c10::DispatchKeySet wrapped({K::Python, K::FuncTorchBatched, K::BatchedNestedTensor, K::Batched, K::FuncTorchGradWrapper,
                                         K::Functionalize, K::ZeroTensor, K::Negative, K::Conjugate});
  return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped) && !t._fw_grad(0).defined();
}
// Whether someone follows the calls one by one (a tracer, a dispatch mode, a function transform); they are shown
// torch.autograd.Function, which they know.
bool followed() {
  return torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

PyObject *corr(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 11 || followed()) Py_RETURN_NONE;
  Geometry g;
  g.kind = (int)PyLong_AsLong(args[0]);
  const int dims = (int)PyLong_AsLong(args[1]);
  if (!THPVariable_CheckExact(args[2]) || !THPVariable_CheckExact(args[3]) ||
      !(args[4] == Py_None || THPVariable_CheckExact(args[4])))
    Py_RETURN_NONE;
  if (!parse(args[5], dims, 1, g.s) || !parse(args[6], dims, 1, g.d) || !parse(args[7], dims, 0, g.p) ||
      !parse(args[8], dims, 1, g.u))
    Py_RETURN_NONE;
  int64_t r[2];
  if (!parse(args[9], dims, 0, r)) Py_RETURN_NONE;
  bool relu = false;
  if (args[10] != Py_None) {
    if (!PyUnicode_Check(args[10]) || PyUnicode_CompareWithASCIIString(args[10], "relu") != 0) Py_RETURN_NONE;
    relu = true;
  }
  const Tensor &input0 = THPVariable_Unpack(args[2]), &weight0 = THPVariable_Unpack(args[3]);
  const Tensor bias0 = args[4] == Py_None ? Tensor() : THPVariable_Unpack(args[4]);
  if (!plain(input0) || !plain(weight0) || (bias0.defined() && !plain(bias0))) Py_RETURN_NONE;
  if (input0.dim() != dims + 2 || weight0.dim() != dims + 2 || (bias0.defined() && bias0.dim() != 1)) Py_RETURN_NONE;
  g.batch = input0.size(0);
  g.c_in = input0.size(1);
  g.c_out = weight0.size(0);
  if (weight0.size(1) != g.c_in || (bias0.defined() && bias0.size(0) != g.c_out)) Py_RETURN_NONE;
  const auto device = input0.device();
  if (weight0.device() != device || (bias0.defined() && bias0.device() != device)) Py_RETURN_NONE;
  for (int i = 0; i < 2; ++i) {
    g.nf[i] = i < dims ? weight0.size(2 + i) : 1;
    g.ng[i] = i < dims ? input0.size(2 + i) : 1;
    if (g.s[i] < 1 || g.d[i] < 1 || g.u[i] < 1 || g.nf[i] < 1 || g.ng[i] < 1 || g.nf[i] > (1 << 30) || g.ng[i] > (1 << 30))
      Py_RETURN_NONE;
    const int kind = i == 0 ? g.kind : MELLIN_AXIS_LCORR;
    if (kind == MELLIN_AXIS_MCORR && g.p[i] < 0) Py_RETURN_NONE;
    g.nh[i] = valid_size(kind, g.nf[i], g.ng[i], g.s[i], g.d[i], g.p[i], g.u[i]) + r[i];
    if (g.nh[i] < 1 || g.nh[i] > (1 << 30)) Py_RETURN_NONE;
  }
  if (g.batch < 1 || g.c_in < 1 || g.c_out < 1 || g.batch > 65535 || g.c_out > 65535 || g.c_in > (1 << 20)) Py_RETURN_NONE;
  // under autocast the floating-point arguments are cast to half (ext/torch.cpp:405-430)
  auto kind_of = input0.scalar_type();
  if (at::autocast::is_autocast_enabled(at::kCUDA)) {
    for (const Tensor *t : {&input0, &weight0, &bias0})
      if (t->defined() && (!t->is_floating_point() || t->scalar_type() == at::kDouble)) Py_RETURN_NONE;
    kind_of = at::kHalf;
  } else if (weight0.scalar_type() != kind_of || (bias0.defined() && bias0.scalar_type() != kind_of)) {
    Py_RETURN_NONE;
  }
  if (kind_of != at::kFloat && kind_of != at::kHalf) Py_RETURN_NONE;

  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(device);
    const bool differentiable =
        at::GradMode::is_enabled() && (input0.requires_grad() || weight0.requires_grad() || (bias0.defined() && bias0.requires_grad()));
    // half tensors of a layer with float parameters: the library rounds them, and keeps the rounded weight for the backward
    const bool wide = kind_of == at::kHalf && weight0.scalar_type() == at::kFloat && (!bias0.defined() || bias0.scalar_type() == at::kFloat);
    const int elem = wide ? MELLIN_ELEM_HALF_FLOAT : kind_of == at::kHalf ? 2 : 4;
    Tensor input, weight, bias, weight_half, kept;
    std::shared_ptr<KeptInput> keeps;
    {
      at::AutoGradMode no_grad(false);
      input = input0.scalar_type() == kind_of ? input0.contiguous() : input0.to(kind_of).contiguous();
      if (wide) {
        weight = weight0.contiguous();
        if (bias0.defined()) bias = bias0.contiguous();
        if (differentiable) weight_half = at::empty(weight.sizes(), input.options());
      } else {
        weight = weight0.scalar_type() == kind_of ? weight0.contiguous() : weight0.to(kind_of).contiguous();
        if (bias0.defined()) bias = bias0.scalar_type() == kind_of ? bias0.contiguous() : bias0.to(kind_of).contiguous();
      }
      out = dims == 2 ? at::empty({g.batch, g.c_out, g.nh[0], g.nh[1]}, input.options())
                      : at::empty({g.batch, g.c_out, g.nh[0]}, input.options());
      // (hooks on saved tensors decide where those live, and what the backward call reads)
      if (differentiable && weight0.requires_grad() && !at::SavedTensorDefaultHooks::get_hooks()) {
        if (const size_t size = mellin_layer_kept_bytes(g.kind, elem, GEOMETRY_ARGS(g))) {
          keeps = std::make_shared<KeptInput>();
          keeps->allocate(input, size);
          kept = keeps->bytes;
        }
      }
      const size_t need = (kept.defined() ? mellin_layer_forward_kept_workspace : mellin_layer_forward_workspace)(g.kind, elem, GEOMETRY_ARGS(g));
      Tensor ws = scratch(input, need);
      check(mellin_layer_forward_kept(g.kind, elem, relu ? MELLIN_ACT_RELU : MELLIN_ACT_NONE, pointer(input), pointer(weight),
                                      pointer(bias), GEOMETRY_ARGS(g), out.data_ptr(),
                                      weight_half.defined() ? weight_half.data_ptr() : nullptr, kept.defined() ? kept.data_ptr() : nullptr,
                                      ws.defined() ? ws.data_ptr() : nullptr, need, launch_stream(input)));
    }
    if (differentiable) {
      auto node = std::shared_ptr<Corr2dBackward>(new Corr2dBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(input0, weight0, bias0));
      node->g = g;
      node->relu = relu;
      node->has_bias = bias0.defined();
      node->kept_ = std::move(keeps);
      node->input_ = torch::autograd::SavedVariable(input, false);
      node->weight_ = torch::autograd::SavedVariable(wide ? weight_half : weight, false);
      node->elem = elem;
      node->param_kind = wide ? at::kFloat : kind_of;
      node->out_sizes = out.sizes().vec();
      node->options = out.options();
      torch::autograd::set_history(out, node);
      if (relu) node->out_ = torch::autograd::SavedVariable(out, true);
    }
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// A tensor in the kernels' layout, [image][group of eight channels][plane + behind][8 channels], from byte `at` on, as it lies.
Tensor unblocked(const Tensor &bytes, int64_t at, at::ScalarType kind, int64_t n, int64_t c, int64_t rows, int64_t cols, int64_t behind) {
  const int64_t groups = (c + 7) / 8, plane = rows * cols, count = n * groups * (plane + behind) * 8;
  return bytes.narrow(0, at, count * (int64_t)c10::elementSize(kind)).view(kind).view({n, groups, plane + behind, 8})
      .narrow(2, 0, plane).permute({0, 1, 3, 2}).reshape({n, groups * 8, rows, cols}).narrow(1, 0, c);
}

// The gradients of a stack of layers with ReLUs.  Edges: the input, then weight and bias of every layer.  The last layer may be
// a projection of a row's columns (MELLIN_STACK_NO_RELU; half tensors): only what it is made of can be differentiated twice.
struct StackBackward : public torch::autograd::Node {
  int kind = 0, elem = 4;
  std::vector<mellin_stack_layer> layers;              // geometry; the pointers are filled in for each call
  torch::autograd::SavedVariable input_, out_;
  std::vector<torch::autograd::SavedVariable> weights_;
  std::vector<bool> has_bias;
  Tensor saved_;
  int first = 0;                                       // the lowest layer that gradients can be asked of
  size_t workspace = 0;
  at::ScalarType param_kind = at::kFloat;

  bool projects() const { return layers.back().pool == MELLIN_STACK_NO_RELU; }
  // A projection alone learns: its weight, the input and the layers below are not read again, and may change.
  bool frozen() const { return projects() && first == (int)layers.size() - 1; }

  std::string name() const override { return "StackBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    input_.reset_data();
    out_.reset_data();
    for (auto &w : weights_) w.reset_data();
    saved_.reset();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
    const bool create_graph = at::GradMode::is_enabled();
    at::AutoGradMode no_grad(false);
    const size_t n = layers.size();
    Tensor input, out, saved;
    std::vector<Tensor> weights(n);
    {
      std::lock_guard<std::mutex> lock(mutex_);
      out = out_.unpack(shared_from_this());           // (raises if the variables have been released)
      saved = saved_;
      input = frozen() ? saved : input_.unpack();      // (frozen: some memory)
      for (size_t i = 0; i < n; ++i) weights[i] = weights_[i].unpack();
    }
    torch::autograd::variable_list result(1 + 2 * n);
    Tensor grad_out = grads[0].defined() ? grads[0] : at::zeros_like(out);
    if (grad_out.scalar_type() != out.scalar_type()) grad_out = grad_out.to(out.scalar_type());
    grad_out = grad_out.contiguous();
    const c10::OptionalDeviceGuard guard(input.device());
    std::vector<mellin_stack_layer> call = layers;
    if (task_should_compute_output(0)) result[0] = at::empty_like(input, at::MemoryFormat::Contiguous);
    for (size_t i = 0; i < n; ++i) {
      const Tensor &w = weights[i];
      const int64_t *d = layers[i].dims;
      if (elem != MELLIN_ELEM_HALF_FLOAT) call[i].weight = pointer(w);
      else if ((int)i >= first) call[i].weight_half = const_cast<void *>(pointer(w));
      if (task_should_compute_output(1 + 2 * i)) {
        result[1 + 2 * i] = at::empty({d[2], d[1], d[3], d[4]}, out.options().dtype(param_kind));
        call[i].grad_weight = result[1 + 2 * i].data_ptr();
      }
      if (has_bias[i] && task_should_compute_output(2 + 2 * i)) {
        result[2 + 2 * i] = at::empty({d[2]}, out.options().dtype(param_kind));
        call[i].grad_bias = result[2 + 2 * i].data_ptr();
      }
    }
    auto launch = [&](size_t bytes) {
      Tensor ws = scratch(input, bytes);
      return mellin_stack_backward(kind, elem, (int)n, call.data(), pointer(input), pointer(out), pointer(grad_out), saved.const_data_ptr(),
                                   (size_t)saved.numel(), result[0].defined() ? result[0].data_ptr() : nullptr, ws.data_ptr(), bytes,
                                   launch_stream(input));
    };
    int rc = launch(workspace);
    if (rc == MELLIN_ERR_WORKSPACE) {                  // (refused before any launch: a setting for the first layer has changed since)
      size_t ignored[2], bytes = 0;
      if (mellin_stack_bytes(kind, elem, 2, (int)n, call.data(), &ignored[0], &ignored[1], &bytes)) rc = launch(bytes);
    }
    check(rc);
    if (create_graph && projects() && grads[0].defined() && (result[2 * n - 1].defined() || result[2 * n].defined()))
      differentiable_projection(grads[0], input, weights, saved, result[2 * n - 1], result[2 * n]);
    return result;
  }

  // With create_graph: the projection's gradients as operations on the features that the forward call saved.
  void differentiable_projection(const Tensor &grad, const Tensor &input, const std::vector<Tensor> &weights, const Tensor &saved,
                                 Tensor &grad_weight, Tensor &grad_bias) {
    const c10::impl::ExcludeDispatchKeyGuard no_cast(c10::autocast_dispatch_keyset);
    at::AutoGradMode with_grad(true);
    const Tensor g = grad.to(at::kHalf);               // (N, classes, T', 1)
    if (grad_bias.defined()) grad_bias = g.sum(at::IntArrayRef({0, 2, 3})).to(param_kind);
    if (!grad_weight.defined()) return;
    const Tensor h = features(input, weights, saved);  // (N, C, T', F')
    grad_weight = g.squeeze(3).transpose(0, 1).flatten(1).mm(h.permute({0, 2, 1, 3}).flatten(2).flatten(0, 1)).to(param_kind)
                      .view(grad_weight.sizes());
  }

  // The projection's input as the forward call saved it, with the layers below as its graph: the same node over them alone,
  // whose part of `saved` comes last.
  Tensor features(const Tensor &input, const std::vector<Tensor> &weights, const Tensor &saved) {
    const size_t below = layers.size() - 1;
    const int64_t *d = layers[below].dims, n = d[0], c = d[1], rows = d[5], cols = d[6];
    Tensor h, second, out;
    std::shared_ptr<StackBackward> node;
    {
      at::AutoGradMode no_grad(false);
      h = unblocked(saved, 0, at::kHalf, n, c, rows, cols, 1).contiguous();
      if (frozen()) return h;
      node = std::shared_ptr<StackBackward>(new StackBackward(), torch::autograd::deleteNode);
      node->layers.assign(layers.begin(), layers.end() - 1);
      mellin_stack_layer &top = node->layers.back();
      const bool pooled = top.pool;
      top.pool = 0;                                    // (its output below is that in front of the pooling)
      size_t saved_bytes = 0, forward_bytes = 0;
      TORCH_CHECK(mellin_stack_bytes(kind, elem, first << 8 | 2, (int)below, node->layers.data(), &saved_bytes, &forward_bytes, &node->workspace),
                  "libmellin_hip: no backward call for the layers below a projection");
      const int64_t rest = saved.numel() - (int64_t)saved_bytes;
      node->saved_ = saved.narrow(0, rest, (int64_t)saved_bytes);
      out = h;
      if (pooled) {                                    // the larger of a pair where it was, zeros elsewhere
        const int64_t which_bytes = n * ((c + 7) / 8) * rows * cols * 8;
        second = unblocked(saved, rest - (which_bytes + 255) / 256 * 256, at::kByte, n, c, rows, cols, 0).to(at::kBool);
        out = at::zeros({n, c, rows, top.dims[8]}, h.options());
        out.slice(3, 0, 2 * cols, 2).copy_(h.masked_fill(second, 0));
        out.slice(3, 1, 2 * cols, 2).copy_(h.masked_fill(second.logical_not(), 0));
      }
    }
    torch::autograd::edge_list edges(next_edges().begin(), next_edges().begin() + 1 + 2 * below);
    node->set_next_edges(std::move(edges));
    node->kind = kind;
    node->elem = elem;
    node->first = first;
    node->param_kind = param_kind;
    node->input_ = torch::autograd::SavedVariable(input, false);
    for (size_t i = 0; i < below; ++i) {
      node->weights_.emplace_back(weights[i], false);
      node->has_bias.push_back(has_bias[i]);
    }
    torch::autograd::set_history(out, node);
    node->out_ = torch::autograd::SavedVariable(out, true);
    return second.defined() ? at::where(second, out.slice(3, 1, 2 * cols, 2), out.slice(3, 0, 2 * cols, 2)) : out;
  }
};

PyObject *stack(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 3 || !THPVariable_CheckExact(args[1]) || !PyList_CheckExact(args[2]) || followed()) Py_RETURN_NONE;
  // (hooks on saved tensors expect the layers' inputs, as the layers themselves save them)
  if (at::GradMode::is_enabled() && at::SavedTensorDefaultHooks::get_hooks()) Py_RETURN_NONE;
  const int kind = (int)PyLong_AsLong(args[0]);
  const Tensor &input0 = THPVariable_Unpack(args[1]);
  const Py_ssize_t n = PyList_GET_SIZE(args[2]);
  if (n < 2 || !plain(input0) || input0.dim() != 4) Py_RETURN_NONE;
  std::vector<mellin_stack_layer> layers(n);
  std::vector<Tensor> weights(n), biases(n);
  auto kind_of = input0.scalar_type();
  const bool cast = at::autocast::is_autocast_enabled(at::kCUDA);
  if (cast) {
    if (!input0.is_floating_point() || kind_of == at::kDouble) Py_RETURN_NONE;
    kind_of = at::kHalf;
  }
  if (kind_of != at::kFloat && kind_of != at::kHalf) Py_RETURN_NONE;
  at::ScalarType param_kind = at::kFloat;
  int first = input0.requires_grad() ? 0 : (int)n;     // the lowest layer that learns (input gradients: all)
  int64_t c = input0.size(1), x = input0.size(2), y = input0.size(3);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *t = PyList_GET_ITEM(args[2], i);
    if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 7) Py_RETURN_NONE;
    PyObject *w = PyTuple_GET_ITEM(t, 0), *b = PyTuple_GET_ITEM(t, 1);
    if (!THPVariable_CheckExact(w) || !(b == Py_None || THPVariable_CheckExact(b))) Py_RETURN_NONE;
    weights[i] = THPVariable_Unpack(w);
    if (b != Py_None) biases[i] = THPVariable_Unpack(b);
    const Tensor &wt = weights[i], &bt = biases[i];
    if (!plain(wt) || wt.dim() != 4 || wt.device() != input0.device() || wt.size(1) != c) Py_RETURN_NONE;
    if (bt.defined() && (!plain(bt) || bt.dim() != 1 || bt.size(0) != wt.size(0) || bt.device() != input0.device())) Py_RETURN_NONE;
    if (i == 0) param_kind = wt.scalar_type();
    if (wt.scalar_type() != param_kind || (bt.defined() && bt.scalar_type() != param_kind)) Py_RETURN_NONE;
    Geometry g;
    int64_t r[2];
    if (!parse(PyTuple_GET_ITEM(t, 2), 2, 1, g.s) || !parse(PyTuple_GET_ITEM(t, 3), 2, 1, g.d) || !parse(PyTuple_GET_ITEM(t, 4), 2, 0, g.p) ||
        !parse(PyTuple_GET_ITEM(t, 5), 2, 0, r))
      Py_RETURN_NONE;
    g.kind = kind;
    g.batch = input0.size(0);
    g.c_in = c;
    g.c_out = wt.size(0);
    g.ng[0] = x;
    g.ng[1] = y;
    for (int k = 0; k < 2; ++k) {
      g.u[k] = 1;
      g.nf[k] = wt.size(2 + k);
      const int axis = k == 0 ? kind : MELLIN_AXIS_LCORR;
      if (g.s[k] < 1 || g.d[k] < 1 || g.nf[k] < 1 || g.ng[k] < 1 || g.nf[k] > (1 << 30) || g.ng[k] > (1 << 30)) Py_RETURN_NONE;
      if (axis == MELLIN_AXIS_MCORR && g.p[k] < 0) Py_RETURN_NONE;
      g.nh[k] = valid_size(axis, g.nf[k], g.ng[k], g.s[k], g.d[k], g.p[k], 1) + r[k];
      if (g.nh[k] < 1 || g.nh[k] > (1 << 30)) Py_RETURN_NONE;
    }
    if (g.batch < 1 || g.c_in < 1 || g.c_out < 1 || g.batch > 65535 || g.c_out > 65535 || g.c_in > (1 << 20)) Py_RETURN_NONE;
    const int64_t dims[17] = {GEOMETRY_ARGS(g)};
    layers[i] = mellin_stack_layer{};
    std::copy(dims, dims + 17, layers[i].dims);
    layers[i].pool = PyTuple_GET_ITEM(t, 6) == Py_True ? 1 : 0;
    if (PyTuple_GET_ITEM(t, 6) == Py_None) {           // a projection of a row's columns
      if (i != n - 1 || n < 3 || kind_of != at::kHalf || g.nf[0] != 1 || g.nf[1] != y || g.nh[0] != x || g.nh[1] != 1 || g.s[0] != 1 || g.d[0] != 1 ||
          g.p[0] != 0 || g.d[1] != 1 || g.p[1] != 0)
        Py_RETURN_NONE;
      layers[i].pool = MELLIN_STACK_NO_RELU;
    }
    if (wt.requires_grad() || (bt.defined() && bt.requires_grad())) first = std::min(first, (int)i);
    c = g.c_out;
    x = g.nh[0];
    y = layers[i].pool == 1 ? g.nh[1] / 2 : g.nh[1];
  }
  // float parameters of half tensors (autocast) are rounded by the library; any other mixture is not for this path
  const bool wide = kind_of == at::kHalf && param_kind == at::kFloat;
  if (!wide && param_kind != kind_of) Py_RETURN_NONE;
  if (wide && !cast) Py_RETURN_NONE;
  const int elem = wide ? MELLIN_ELEM_HALF_FLOAT : kind_of == at::kHalf ? 2 : 4;
  const bool differentiable = first < (int)n && at::GradMode::is_enabled();
  const int train = differentiable ? MELLIN_STACK_TRAIN_FROM(first) : 0;
  size_t saved_bytes = 0, forward_bytes = 0, backward_bytes = 0;
  if (!mellin_stack_bytes(kind, elem, train, (int)n, layers.data(), &saved_bytes, &forward_bytes, &backward_bytes)) Py_RETURN_NONE;

  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(input0.device());
    Tensor input, saved;
    std::vector<Tensor> kept(n);
    {
      at::AutoGradMode no_grad(false);
      input = input0.scalar_type() == kind_of ? input0.contiguous() : input0.to(kind_of).contiguous();
      std::vector<mellin_stack_layer> call = layers;
      std::vector<Tensor> dense(2 * n);
      for (Py_ssize_t i = 0; i < n; ++i) {
        dense[2 * i] = weights[i].contiguous();
        call[i].weight = dense[2 * i].const_data_ptr();
        if (biases[i].defined()) {
          dense[2 * i + 1] = biases[i].contiguous();
          call[i].bias = dense[2 * i + 1].const_data_ptr();
        }
        kept[i] = dense[2 * i];
        if (wide && differentiable && i >= first) {
          kept[i] = at::empty(weights[i].sizes(), input.options());
          call[i].weight_half = kept[i].data_ptr();
        }
      }
      const int64_t *d = layers[n - 1].dims;
      out = at::empty({d[0], d[2], d[7], d[8]}, input.options());
      saved = scratch(input, saved_bytes);
      Tensor ws = scratch(input, forward_bytes);
      check(mellin_stack_forward(kind, elem, train, (int)n, call.data(), pointer(input), out.data_ptr(), saved.data_ptr(),
                                 saved_bytes, ws.data_ptr(), forward_bytes, launch_stream(input)));
    }
    if (differentiable) {
      auto node = std::shared_ptr<StackBackward>(new StackBackward(), torch::autograd::deleteNode);
      torch::autograd::edge_list edges;
      auto edge = [&](const Tensor &t) {
        edges.push_back(t.defined() && t.requires_grad() ? torch::autograd::impl::gradient_edge(t) : torch::autograd::Edge());
      };
      edge(input0);
      for (Py_ssize_t i = 0; i < n; ++i) {
        edge(weights[i]);
        edge(biases[i]);
        node->has_bias.push_back(biases[i].defined());
      }
      node->set_next_edges(std::move(edges));
      node->kind = kind;
      node->elem = elem;
      node->first = first;
      node->layers = std::move(layers);
      const bool frozen = node->frozen();
      for (Py_ssize_t i = 0; i < n; ++i) node->weights_.emplace_back(frozen ? Tensor() : kept[i], false);
      if (!frozen) node->input_ = torch::autograd::SavedVariable(input, false);
      node->saved_ = std::move(saved);
      node->workspace = backward_bytes;
      node->param_kind = wide ? at::kFloat : kind_of;
      torch::autograd::set_history(out, node);
      node->out_ = torch::autograd::SavedVariable(out, true);
    }
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The gradients of LogCompressionLift, at the eps and tau of the forward call, which it left in `params_`: the parameters
// themselves may be another step's by now (a second loss whose graph is older than the step).
struct LogLiftBackward : public torch::autograd::Node {
  torch::autograd::SavedVariable input_, params_;
  at::DimVector eps_sizes, tau_sizes;
  int64_t outer = 0, t = 0, inner = 0;

  std::string name() const override { return "LogLiftBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    input_.reset_data();
    params_.reset_data();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
    at::AutoGradMode no_grad(false);
    Tensor input, params;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      input = input_.unpack();
      params = params_.unpack();
    }
    const Tensor grad = grads[0].defined() ? grads[0].contiguous() : at::zeros(input.sizes(), input.options());
    const c10::OptionalDeviceGuard guard(input.device());
    // (gradients become .grad as they are: each has memory of its own)
    Tensor grad_input, grad_eps, grad_tau;
    if (task_should_compute_output(1)) grad_eps = at::empty(eps_sizes, input.options());
    if (task_should_compute_output(2)) grad_tau = at::empty(tau_sizes, input.options());
    if (task_should_compute_output(0)) grad_input = at::empty_like(input, at::MemoryFormat::Contiguous);
    const size_t need = mellin_log_lift_backward_workspace(4, outer, t, inner);
    Tensor ws = scratch(input, need);
    check(mellin_log_lift_backward_kept_f32((const float *)pointer(input), (const float *)pointer(grad), (const float *)pointer(params),
                                            MELLIN_PW_LOG | MELLIN_PW_LIFT, outer, t, inner,
                                            grad_input.defined() ? (float *)grad_input.data_ptr() : nullptr,
                                            grad_eps.defined() ? (float *)grad_eps.data_ptr() : nullptr,
                                            grad_tau.defined() ? (float *)grad_tau.data_ptr() : nullptr,
                                            ws.defined() ? ws.data_ptr() : nullptr, need, launch_stream(input)));
    return {grad_input, grad_eps, grad_tau};
  }
};

PyObject *log_lift(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 4 || followed()) Py_RETURN_NONE;
  for (int i = 0; i < 3; ++i)
    if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
  const Tensor &input0 = THPVariable_Unpack(args[0]), &log_eps = THPVariable_Unpack(args[1]), &log_tau = THPVariable_Unpack(args[2]);
  const int64_t dim = PyLong_AsLongLong(args[3]);
  if (!plain(input0) || input0.scalar_type() != at::kFloat || dim < 0 || dim >= input0.dim() || input0.numel() == 0) Py_RETURN_NONE;
  for (const Tensor *p : {&log_eps, &log_tau})
    if (!plain(*p) || p->scalar_type() != at::kFloat || p->numel() != 1 || p->device() != input0.device()) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(input0.device());
    const bool differentiable = at::GradMode::is_enabled() && (input0.requires_grad() || log_eps.requires_grad() || log_tau.requires_grad());
    int64_t outer = 1, inner = 1;
    for (int64_t i = 0; i < input0.dim(); ++i) (i < dim ? outer : inner) *= i == dim ? 1 : input0.size(i);
    const int64_t t = input0.size(dim);
    Tensor input, params;
    {
      at::AutoGradMode no_grad(false);
      input = input0.contiguous();
      out = at::empty_like(input, at::MemoryFormat::Contiguous);
      params = at::empty({2}, input.options());
      check(mellin_log_lift_forward_keep_f32((const float *)pointer(input), (const float *)pointer(log_eps), (const float *)pointer(log_tau),
                                             MELLIN_PW_LOG | MELLIN_PW_LIFT, outer, t, inner, (float *)out.data_ptr(),
                                             (float *)params.data_ptr(), launch_stream(input)));
    }
    if (differentiable) {
      auto node = std::shared_ptr<LogLiftBackward>(new LogLiftBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(input0, log_eps, log_tau));
      node->input_ = torch::autograd::SavedVariable(input, false);
      node->params_ = torch::autograd::SavedVariable(params, false);
      node->eps_sizes = at::DimVector(log_eps.sizes());
      node->tau_sizes = at::DimVector(log_tau.sizes());
      node->outer = outer;
      node->t = t;
      node->inner = inner;
      torch::autograd::set_history(out, node);
    }
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// Windows of utterances in the order of torch.nn.utils.rnn.pack_padded_sequence (longest first, then time step by time step):
// (data, batch_sizes, sorted_indices, unsorted_indices).  The order is worked out here, as the reference does on the CPU, and
// goes to the GPU from pinned memory, so that nothing waits for what the GPU has been given before (padding, unfolding and
// packing by PyTorch took 58 to 92 us of host time and a synchronous copy).
PyObject *pack_windows(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 4 || followed() || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !PyLong_CheckExact(args[2]) ||
      !PyLong_CheckExact(args[3]))
    Py_RETURN_NONE;
  const Tensor &x0 = THPVariable_Unpack(args[0]), &lens0 = THPVariable_Unpack(args[1]);
  const int64_t size = PyLong_AsLongLong(args[2]), stride = PyLong_AsLongLong(args[3]);
  if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
  if (!plain(x0) || x0.scalar_type() != at::kFloat || x0.dim() != 3 || (x0.requires_grad() && at::GradMode::is_enabled())) Py_RETURN_NONE;
  const int64_t n = x0.size(0), frames = x0.size(1), row = x0.size(2), lim = (int64_t)1 << 31;
  if (n < 1 || frames < 1 || row < 1 || size < 1 || stride < 1 || size >= lim || n * frames >= lim || size * row >= lim) Py_RETURN_NONE;
  if (!lens0.device().is_cpu() || lens0.layout() != at::kStrided || lens0.scalar_type() != at::kLong || lens0.dim() != 1 ||
      lens0.size(0) != n || lens0.requires_grad())
    Py_RETURN_NONE;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)launch_stream(x0), &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) Py_RETURN_NONE;
  Tensor counts, order;
  int64_t windows = 0;
  {
    at::AutoGradMode no_grad(false);
    counts = at::empty({n}, lens0.options());
    const Tensor lens = lens0.contiguous();
    const int64_t *l = lens.const_data_ptr<int64_t>();
    int64_t *c = counts.mutable_data_ptr<int64_t>();
    for (int64_t i = 0; i < n; ++i) {
      if (l[i] < 1 || l[i] > frames) Py_RETURN_NONE;         // (errors, with PyTorch's messages)
      c[i] = (l[i] - 1) / stride + 1;
      windows += c[i];
    }
    std::tie(counts, order) = at::sort(counts, -1, true);
  }
  if (windows >= lim) Py_RETURN_NONE;
  const int64_t *c = counts.const_data_ptr<int64_t>(), *o = order.const_data_ptr<int64_t>();
  at::AutoGradMode no_grad(false);
  const c10::OptionalDeviceGuard guard(x0.device());
  Tensor batch_sizes = at::empty({c[0]}, lens0.options()), table = at::empty({2 * n + windows}, lens0.options().pinned_memory(true));
  int64_t *b = batch_sizes.mutable_data_ptr<int64_t>(), *p = table.mutable_data_ptr<int64_t>(), *entry = p + 2 * n;
  for (int64_t i = 0; i < n; ++i) {
    p[i] = o[i];
    p[n + o[i]] = i;
  }
  int64_t live = n;
  for (int64_t step = 0; step < c[0]; ++step) {
    while (c[live - 1] <= step) --live;
    b[step] = live;
    const int64_t first = step * stride, whole = std::min(size, frames - first);
    for (int64_t i = 0; i < live; ++i) *entry++ = (o[i] * frames + first) | whole << 32;
  }
  const Tensor x = x0.contiguous(), there = table.to(x0.device(), /*non_blocking=*/true);
  Tensor data = at::empty({windows, size, row}, x.options());
  check(mellin_pack_windows_f32((const float *)pointer(x), there.const_data_ptr<int64_t>() + 2 * n, windows, size, row, (float *)data.data_ptr(),
                                launch_stream(x)));
  PyObject *result = PyTuple_New(4);
  if (!result) return nullptr;
  PyTuple_SET_ITEM(result, 0, THPVariable_Wrap(std::move(data)));
  PyTuple_SET_ITEM(result, 1, THPVariable_Wrap(std::move(batch_sizes)));
  PyTuple_SET_ITEM(result, 2, THPVariable_Wrap(there.narrow(0, 0, n)));
  PyTuple_SET_ITEM(result, 3, THPVariable_Wrap(there.narrow(0, n, n)));
  return result;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"log_lift", (PyCFunction)(void *)log_lift, METH_FASTCALL,
     "log_lift(input, log_eps, log_tau, dim): log compression and lift, or None if not handled"},
    {"pack_windows", (PyCFunction)(void *)pack_windows, METH_FASTCALL,
     "pack_windows(x, lens, size, stride): (data, batch_sizes, sorted_indices, unsorted_indices), or None if not handled"},
    {"stack", (PyCFunction)(void *)stack, METH_FASTCALL,
     "stack(kind, input, [(weight, bias, s, d, p, r, pool), ...]): the last layer's output behind its ReLU (without one if its "
     "pool is None: a projection of each row's columns, in half), or None if not handled"},
    {"corr", (PyCFunction)(void *)corr, METH_FASTCALL,
     "corr(kind, dims, input, weight, bias, s, d, p, u, r, activation): the layer's output, or None if not handled"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mellin_torch", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__mellin_torch() { return PyModule_Create(&module); }
