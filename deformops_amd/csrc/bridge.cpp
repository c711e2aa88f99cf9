// The autograd bridge of plain eager MSDA calls, as a Python extension module.
//
// forward() is what the Python bridge would do for real tensors outside any trace:
// bring the operands into the kernels' dtypes and layouts, allocate the output and
// call msda_forward on torch's current stream; and, where a gradient is needed, record
// an autograd node whose backward allocates the three gradients and the workspace and
// calls msda_backward_workspace. In C++ because a small call is bound by host time: the
// node runs on the autograd engine's thread, where a Python node first has to take the
// interpreter's lock from the thread that waits for it. The reference's bridge is a
// Python autograd registration over boxed C++ ops (backends/cuda/_msda_bridge.py:186-261).
//
// The library's entry points come as addresses (init), so that this module works with
// whichever build of the library Python has loaded.

#include <ATen/Functions.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <cstdint>
#include <cstdlib>
#include <string>

#include "deformops_amd.h"

namespace {

using at::Tensor;
using torch::autograd::variable_list;

decltype(&msda_forward) g_forward = nullptr;
decltype(&msda_backward_workspace) g_backward = nullptr;
decltype(&msda_backward_workspace_size) g_workspace_size = nullptr;
decltype(&msda_last_error) g_last_error = nullptr;

void init(uintptr_t forward, uintptr_t backward, uintptr_t workspace_size, uintptr_t last_error) {
  g_forward = reinterpret_cast<decltype(g_forward)>(forward);
  g_backward = reinterpret_cast<decltype(g_backward)>(backward);
  g_workspace_size = reinterpret_cast<decltype(g_workspace_size)>(workspace_size);
  g_last_error = reinterpret_cast<decltype(g_last_error)>(last_error);
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MSDA_F32;
    case at::kHalf: return MSDA_F16;
    case at::kBFloat16: return MSDA_BF16;
    case at::kDouble: return MSDA_F64;
    default: break;
  }
  TORCH_CHECK(false, "msda: unsupported dtype ", t);
}

void check(int status) {
  if (status == MSDA_OK) return;
  const char* message = g_last_error();
  TORCH_CHECK(false, message && *message ? std::string(message) : "msda call failed with status " + std::to_string(status));
}

// The operands as the kernels take them: contiguous, weights in the value dtype,
// locations in float32 or the value dtype, both level tables int32 or both int64.
struct Operands {
  Tensor value, shapes, starts, loc, attn;
};

at::ScalarType location_dtype(at::ScalarType value, at::ScalarType loc) {
  if (value == at::kDouble) return at::kDouble;
  return loc == at::kFloat || loc == value ? loc : at::kFloat;
}

Operands normalized(const Tensor& value, const Tensor& shapes, const Tensor& starts, const Tensor& loc,
                    const Tensor& attn) {
  const bool tables_ok = shapes.scalar_type() == starts.scalar_type() &&
                         (shapes.scalar_type() == at::kLong || shapes.scalar_type() == at::kInt);
  return Operands{value.contiguous(), (tables_ok ? shapes : shapes.to(at::kLong)).contiguous(),
                  (tables_ok ? starts : starts.to(at::kLong)).contiguous(),
                  loc.to(location_dtype(value.scalar_type(), loc.scalar_type())).contiguous(),
                  attn.to(value.scalar_type()).contiguous()};
}

struct Sizes {
  int64_t B, S, H, D, Q, L, P;
};

Sizes sizes_of(const Operands& o) {
  return Sizes{o.value.size(0), o.value.size(1), o.value.size(2), o.value.size(3),
               o.loc.size(1),   o.shapes.size(0), o.loc.size(4)};
}

int index_code(const Tensor& shapes) { return shapes.scalar_type() == at::kInt ? MSDA_I32 : MSDA_I64; }

void* current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor launch_forward(const Operands& o, bool softmax) {
  const Sizes s = sizes_of(o);
  const c10::OptionalDeviceGuard guard(o.value.device());
  Tensor out = at::empty({s.B, s.Q, s.H * s.D}, o.value.options());
  check(g_forward(o.value.data_ptr(), dtype_code(o.value.scalar_type()), o.shapes.data_ptr(), o.starts.data_ptr(),
                  index_code(o.shapes), o.loc.data_ptr(), dtype_code(o.loc.scalar_type()), o.attn.data_ptr(),
                  out.data_ptr(), s.B, s.S, s.H, s.D, s.Q, s.L, s.P, softmax ? MSDA_SOFTMAX : 0,
                  current_stream(o.value)));
  return out;
}

// The three gradients, in the operands' dtypes and layouts. The workspace's memory may be
// handed out again when the call returns: the caching allocator orders its reuse after
// this call's kernels on the same stream.
variable_list launch_backward(const Operands& o, const Tensor& grad_output, bool softmax) {
  const Sizes s = sizes_of(o);
  const c10::OptionalDeviceGuard guard(o.value.device());
  const int flags = softmax ? MSDA_SOFTMAX : 0, dtype = dtype_code(o.value.scalar_type());
  const Tensor grad = grad_output.to(o.value.scalar_type()).contiguous();
  Tensor grad_value = at::empty_like(o.value), grad_loc = at::empty_like(o.loc), grad_attn = at::empty_like(o.attn);
  int64_t bytes = 0;
  check(g_workspace_size(dtype, s.B, s.S, s.H, s.D, s.Q, s.L, s.P, flags, &bytes));
  Tensor workspace = at::empty({bytes}, o.value.options().dtype(at::kByte));
  check(g_backward(o.value.data_ptr(), dtype, o.shapes.data_ptr(), o.starts.data_ptr(), index_code(o.shapes),
                   o.loc.data_ptr(), dtype_code(o.loc.scalar_type()), o.attn.data_ptr(), grad.data_ptr(),
                   grad_value.data_ptr(), grad_loc.data_ptr(), grad_attn.data_ptr(), s.B, s.S, s.H, s.D, s.Q, s.L, s.P,
                   flags, workspace.data_ptr(), bytes, current_stream(o.value)));
  return {grad_value, grad_loc, grad_attn};
}

// Whether the five operands are plain memory of one GPU and agree in rank and size: the
// launches take addresses and sizes at their word.
bool agree(const std::array<Tensor, 5>& t) {
  const Tensor &value = t[0], &shapes = t[1], &starts = t[2], &loc = t[3], &attn = t[4];
  for (const Tensor& x : t)
    if (!x.is_cuda() || x.device() != value.device() || x.layout() != at::kStrided) return false;
  if (value.dim() != 4 || shapes.dim() != 2 || starts.dim() != 1 || loc.dim() != 6) return false;
  const int64_t B = value.size(0), H = value.size(2), L = shapes.size(0), Q = loc.size(1), P = loc.size(4);
  if (shapes.size(1) != 2 || starts.size(0) != L || loc.size(0) != B || loc.size(2) != H || loc.size(3) != L ||
      loc.size(5) != 2)
    return false;
  const bool flat = attn.dim() == 4 && attn.size(3) == L * P;
  const bool split = attn.dim() == 5 && attn.size(3) == L && attn.size(4) == P;
  return (flat || split) && attn.size(0) == B && attn.size(1) == Q && attn.size(2) == H;
}

struct MSDA : torch::autograd::Function<MSDA> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& value, const Tensor& shapes,
                        const Tensor& starts, const Tensor& loc, const Tensor& attn, bool softmax) {
    ctx->save_for_backward({value, shapes, starts, loc, attn});
    ctx->saved_data["softmax"] = softmax;
    return launch_forward(Operands{value, shapes, starts, loc, attn}, softmax);
  }

  static variable_list backward(torch::autograd::AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    variable_list out;
    {
      const at::NoGradGuard no_grad;
      // Saved-tensor hooks may hand back other tensors than they were given: any layout
      // will do, but not host memory or other sizes.
      const std::array<Tensor, 5> t = {saved[0], saved[1], saved[2], saved[3], saved[4]};
      TORCH_CHECK(agree(t) && grads[0].device() == t[0].device() &&
                      grads[0].sizes() == at::IntArrayRef({t[0].size(0), t[3].size(1), t[0].size(2) * t[0].size(3)}),
                  "msda: the operands unpacked for the backward are not on the output's device or not of the sizes "
                  "that were saved");
      out = launch_backward(normalized(t[0], t[1], t[2], t[3], t[4]), grads[0], ctx->saved_data["softmax"].toBool());
    }
    // The kernels' gradients carry no graph: where one is asked for and would lead
    // through the output's gradient, they come back behind a node that raises.
    if (at::GradMode::is_enabled() && grads[0].requires_grad()) {
      for (Tensor& t : out) t = t.detach().set_requires_grad(true);
      auto error = std::make_shared<torch::autograd::DelayedError>(
          "trying to differentiate twice a function that was marked with @once_differentiable", int64_t(out.size()));
      out = (*error)(std::move(out));
    }
    return {out[0], Tensor(), Tensor(), out[1], out[2], Tensor()};
  }
};

Tensor forward(const Tensor& value, const Tensor& shapes, const Tensor& starts, const Tensor& loc, const Tensor& attn,
               bool softmax) {
  const pybind11::gil_scoped_release no_gil;
  // There is no forward-mode rule. A tangent is refused in every grad mode, as an
  // autograd.Function without a jvp refuses it: the launch alone would answer without one.
  for (const Tensor* t : {&value, &loc, &attn})
    TORCH_CHECK_NOT_IMPLEMENTED(!t->_fw_grad(/*level=*/0).defined(),
                                "msda: forward-mode differentiation is not supported (an operand has a tangent)");
  const Operands o = normalized(value, shapes, starts, loc, attn);
  if (at::GradMode::is_enabled() && (o.value.requires_grad() || o.loc.requires_grad() || o.attn.requires_grad()))
    return MSDA::apply(o.value, o.shapes, o.starts, o.loc, o.attn, softmax);
  return launch_forward(o, softmax);
}

// Whether DEFORMOPS_VALIDATE asks for the level-table checks (core/sanitize.py).
bool value_checks_enabled() {
  const char* v = std::getenv("DEFORMOPS_VALIDATE");
  return v && *v && std::string(v) != "0";  // other falsy spellings take the checked path too
}

// Whether a call with these operands needs nothing but the launch: what the registry's
// structural checks (core/sanitize.py::check_msda_call), its policy for GPU tensors and
// the kernels' own limits (backends/hip/_bridge.py::supports_context) would pass.
bool takes(const std::array<Tensor, 5>& t) {
  const Tensor &value = t[0], &shapes = t[1], &starts = t[2], &loc = t[3], &attn = t[4];
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::Functionalize,
                                         c10::DispatchKey::Python, c10::DispatchKey::Negative});
  for (const Tensor& x : t)
    if (x.key_set().has_any(wrapped)) return false;
  if (!agree(t)) return false;
  const int64_t S = value.size(1), H = value.size(2), D = value.size(3), L = shapes.size(0), samples = L * loc.size(4);
  const at::ScalarType dtype = value.scalar_type(), loc_dtype = loc.scalar_type();
  const bool f64 = dtype == at::kDouble;
  auto kernel_dtype = [](at::ScalarType d) {
    return d == at::kFloat || d == at::kHalf || d == at::kBFloat16 || d == at::kDouble;
  };
  if (!kernel_dtype(dtype) || !kernel_dtype(loc_dtype) || attn.scalar_type() != dtype) return false;
  for (const Tensor* x : {&shapes, &starts})
    if (x->scalar_type() != at::kLong && x->scalar_type() != at::kInt) return false;
  if (samples > 4096 || D == 0 || S * H * D >= (int64_t(1) << 31)) return false;
  const int64_t es = int64_t(value.element_size());
  int64_t cv = 16 / es;
  while (cv > 1 && D % cv) cv /= 2;
  if (D / cv > 64) return false;
  auto align16 = [](int64_t n) { return (n + 15) / 16 * 16; };
  const int64_t lds = align16(16 * L + samples * (f64 ? 48 : 32)) + align16(samples * 2 * (f64 ? 8 : 4)) + align16(samples * es);
  return lds <= 64 * 1024;
}

// A call of the five operands, or None when anything about it needs the registry's own
// path: a tensor subclass, a dispatch or function mode, a trace, a functorch transform,
// a malformed or unsupported call (whose error that path raises).
pybind11::object try_forward(pybind11::handle value, pybind11::handle shapes, pybind11::handle starts,
                             pybind11::handle loc, pybind11::handle attn, bool softmax) {
  std::array<Tensor, 5> t;
  const std::array<PyObject*, 5> raw = {value.ptr(), shapes.ptr(), starts.ptr(), loc.ptr(), attn.ptr()};
  for (int i = 0; i < 5; ++i) {
    if (!THPVariable_CheckExact(raw[i])) return pybind11::none();
    t[i] = THPVariable_Unpack(raw[i]);
  }
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
      torch::jit::tracer::isTracing() || value_checks_enabled() || !takes(t))
    return pybind11::none();
  return pybind11::cast(forward(t[0], t[1], t[2], t[3], t[4], softmax));
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("init", &init);
  m.def("forward", &forward);
  m.def("try_forward", &try_forward);
}
