// The layers' host path: argument checks, output and workspace allocation, the autograd node and
// the calls into libmellin_hip, as one CPython function.  A call of a small layer is bound by
// what the host does: through Python (torch.autograd.Function, ctypes, one call and one
// allocation per pass) a 1-D layer's forward took 30 us of host time and a training step of it
// 140-240 us for 7 launches; here 4 and 30.
//
// corr(kind, dims, input, weight, bias, s, d, p, u, r, activation) returns the output tensor, or
// None for whatever it does not handle (other element types, CPU tensors, arguments that are
// errors): mconv.py then takes its own path, which has the checks and their messages.
#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>

#include <mutex>

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

// The gradients of out = activation(bias + correlation(input, weight)).
struct Corr2dBackward : public torch::autograd::Node {
  Geometry g;
  bool relu = false, has_bias = false;
  int elem = 4;                          // as the library's entry points take it
  at::ScalarType param_kind = at::kFloat;
  torch::autograd::SavedVariable input_, weight_, out_;
  std::vector<int64_t> out_sizes;
  at::TensorOptions options;

  std::string name() const override { return "Corr2dBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    input_.reset_data();
    weight_.reset_data();
    out_.reset_data();
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
    at::AutoGradMode no_grad(false);
    Tensor input, weight, out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
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
      const size_t need = mellin_layer_backward_workspace(g.kind, elem, want, GEOMETRY_ARGS(g));
      Tensor ws = scratch(input, need);
      check(mellin_layer_backward(g.kind, elem, want, pointer(input), pointer(weight), pointer(grad_out), pointer(out),
                                  GEOMETRY_ARGS(g), grad_input.defined() ? grad_input.data_ptr() : nullptr,
                                  grad_weight.defined() ? grad_weight.data_ptr() : nullptr,
                                  grad_bias.defined() ? grad_bias.data_ptr() : nullptr,
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

// Whether the library's float and half kernels take `t` (and nothing watches it that this path does not serve).
bool plain(const Tensor &t) { return t.is_cuda() && t.layout() == at::kStrided && !t._fw_grad(0).defined(); }

PyObject *corr(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 11) Py_RETURN_NONE;
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
    Tensor input, weight, bias, weight_half;
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
      const size_t need = mellin_layer_forward_workspace(g.kind, elem, GEOMETRY_ARGS(g));
      Tensor ws = scratch(input, need);
      check(mellin_layer_forward(g.kind, elem, relu ? MELLIN_ACT_RELU : MELLIN_ACT_NONE, pointer(input), pointer(weight),
                                 pointer(bias), GEOMETRY_ARGS(g), out.data_ptr(),
                                 weight_half.defined() ? weight_half.data_ptr() : nullptr, ws.defined() ? ws.data_ptr() : nullptr, need, launch_stream(input)));
    }
    if (differentiable) {
      auto node = std::shared_ptr<Corr2dBackward>(new Corr2dBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(input0, weight0, bias0));
      node->g = g;
      node->relu = relu;
      node->has_bias = bias0.defined();
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

PyMethodDef methods[] = {
    {"corr", (PyCFunction)(void *)corr, METH_FASTCALL,
     "corr(kind, dims, input, weight, bias, s, d, p, u, r, activation): the layer's output, or None if not handled"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mellin_torch", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__mellin_torch() { return PyModule_Create(&module); }
