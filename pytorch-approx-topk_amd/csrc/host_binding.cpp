// The host side of a call: from tensors to the C ABI, without Python in between.
//
// In small calls the host is what counts: through Python and ctypes, fp32 [4, 65536] k=1024
// took 11.8 us per call around one kernel of 3.1 us.  This module holds
//   run:     outputs, workspace and the native call for rows in place, for the wrappers that are
//            no operators (compact indices, the arg-max entry points);
//   topk:    the operator's kernel for the GPU (dispatch key CUDA, which is HIP's here);
//   topk_grad: the same for the gradient's operator;
//   differentiable_topk: the operator with the gradient, as an autograd node.
// Each takes the common case, contiguous rows of plain GPU tensors and arguments that hold;
// whatever else there is goes to the Python function of the same meaning, which also raises the errors.
//
// The native library is loaded by _native.py with the first call that needs it, which hands its entry points over as
// addresses (`bind`); until then the Python functions take every call.
#include <atomic>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/extension.h>

#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>

#include "../../include/approx_topk_hip.h"

namespace {

using at::Tensor;
using c10::optional;

// ---- the native library ----
decltype(&atk_strerror) g_strerror;
decltype(&atk_stage1_workspace_bytes) g_stage1_workspace;
decltype(&atk_stage1) g_stage1;
decltype(&atk_stage1_i32) g_stage1_i32;
decltype(&atk_topk_workspace_bytes_used) g_topk_workspace;
decltype(&atk_topk) g_topk;
decltype(&atk_topk_i32) g_topk_i32;
decltype(&atk_topk_grad) g_topk_grad;
std::atomic<bool> g_bound{false};  // set behind them, once (the kernels below run without the interpreter's lock)

bool bound() { return g_bound.load(std::memory_order_acquire); }

// the Python functions that take what the fast paths do not (held until the process ends)
PyObject* g_topk_any = nullptr;
PyObject* g_topk_grad_any = nullptr;
PyObject* g_gradient_any = nullptr;

void check(int status) {
  if (status != ATK_OK) throw std::runtime_error(g_strerror(status));
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return ATK_F32;
    case at::kHalf: return ATK_F16;
    case at::kBFloat16: return ATK_BF16;
    case at::kDouble: return ATK_F64;
    case at::kByte: return ATK_U8;
    case at::kChar: return ATK_I8;
    case at::kShort: return ATK_I16;
    case at::kInt: return ATK_I32;
    case at::kLong: return ATK_I64;
    default: return -1;
  }
}

// A dense GPU tensor and nothing else: no subclass, no transform's wrapper, no lazy conjugation.
bool plain(const Tensor& t) {
  static const c10::DispatchKeySet keys = c10::DispatchKeySet(c10::DispatchKey::CUDA) |
                                          c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
                                          c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) |
                                          c10::autocast_dispatch_keyset;  // (every tensor has its backend's)
  return t.is_cuda() && t.layout() == at::kStrided && (t.key_set().raw_repr() & ~keys.raw_repr()) == 0;
}

// The device of a call made current while it lasts, at no cost when it is.
struct OnDevice {
  explicit OnDevice(c10::Device device) : impl() {
    was = impl.getDevice();
    changed = was.index() != device.index();
    if (changed) impl.setDevice(device);
  }
  ~OnDevice() {
    if (changed) impl.uncheckedSetDevice(was);
  }
  c10::hip::HIPGuardImplMasqueradingAsCUDA impl;
  c10::Device was{c10::DeviceType::CUDA, 0};
  bool changed;
};

void* stream_of(const Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// Both stages (k < k0) or the first alone (k == k0) over contiguous rows; the arguments have been checked.
std::tuple<Tensor, Tensor> run_rows(const Tensor& xs, int64_t k0, int64_t j, int64_t k, int layout, bool narrow,
                                    bool want_values, bool two_stage) {
  const int code = dtype_code(xs.scalar_type());
  const int64_t n = xs.size(-1), rows = xs.numel() / n;
  c10::SmallVector<int64_t, 6> shape(xs.sizes().begin(), xs.sizes().end());
  shape.back() = k;
  Tensor values;
  if (want_values) values = at::empty(shape, xs.options());
  Tensor indices = at::empty(shape, xs.options().dtype(narrow ? at::kInt : at::kLong));
  OnDevice guard(xs.device());
  const void* x = xs.const_data_ptr();
  void* v = want_values ? values.mutable_data_ptr() : nullptr;
  const size_t need = two_stage ? g_topk_workspace(x, rows, n, n, k0, (int)j, k, layout, code)
                                : g_stage1_workspace(rows, n, k0, (int)j, layout, code);
  Tensor ws;
  if (need) ws = at::empty({(int64_t)need}, xs.options().dtype(at::kByte));
  void* w = need ? ws.mutable_data_ptr() : nullptr;
  void* stream = stream_of(xs);
  int status;
  if (narrow) {
    int32_t* i = indices.mutable_data_ptr<int32_t>();
    status = two_stage ? g_topk_i32(x, rows, n, n, k0, (int)j, k, layout, code, v, i, w, need, stream)
                       : g_stage1_i32(x, rows, n, n, k0, (int)j, layout, code, v, i, w, need, stream);
  } else {
    int64_t* i = indices.mutable_data_ptr<int64_t>();
    status = two_stage ? g_topk(x, rows, n, n, k0, (int)j, k, layout, code, v, i, w, need, stream)
                       : g_stage1(x, rows, n, n, k0, (int)j, layout, code, v, i, w, need, stream);
  }
  check(status);
  return {values, indices};
}

bool rows_in_place(const Tensor& xs) {
  return bound() && plain(xs) && xs.dim() > 0 && xs.numel() > 0 && xs.is_contiguous() && dtype_code(xs.scalar_type()) >= 0;
}

// ---- approx_topk::topk on the GPU ----
std::tuple<Tensor, Tensor> topk(const Tensor& xs, int64_t k, int64_t dim, int64_t j, int64_t k_mult, bool interleaved,
                                optional<bool> multithread_buckets) {
  const int64_t last = xs.dim() - 1;
  int64_t k0;
  if ((dim == last || dim == -1) && k > 0 && k_mult > 0 && !__builtin_mul_overflow(k, k_mult, &k0) && j >= 1 && j <= 4 &&
      k0 % j == 0 && rows_in_place(xs) && k0 <= xs.size(-1))
    return run_rows(xs, k0, j, k, interleaved ? ATK_INTERLEAVED : ATK_BALANCED, false, true, k_mult != 1);
  py::gil_scoped_acquire gil;
  return py::reinterpret_borrow<py::object>(g_topk_any)(xs, k, dim, j, k_mult, interleaved, multithread_buckets)
      .cast<std::tuple<Tensor, Tensor>>();
}

// ---- approx_topk::topk_grad on the GPU ----
constexpr int64_t kMaxGradRow = (int64_t(1) << 31) - 1;

Tensor topk_grad(const Tensor& grad_values, const Tensor& indices, int64_t n, int64_t k0, int64_t j, bool interleaved) {
  if (bound() && plain(grad_values) && plain(indices) && indices.scalar_type() == at::kLong && indices.dim() > 0 &&
      indices.numel() > 0 && grad_values.sizes() == indices.sizes() && grad_values.device() == indices.device() &&
      dtype_code(grad_values.scalar_type()) >= 0) {
    const Tensor grad = grad_values.contiguous(), index = indices.contiguous();
    const int64_t k = index.size(-1);
    c10::SmallVector<int64_t, 6> shape(index.sizes().begin(), index.sizes().end());
    shape.back() = n;
    Tensor grad_x = at::empty(shape, grad.options());
    OnDevice guard(grad.device());
    check(g_topk_grad(grad.const_data_ptr(), index.const_data_ptr<int64_t>(), index.numel() / k, n, k0, (int)j, k,
                      interleaved ? ATK_INTERLEAVED : ATK_BALANCED, dtype_code(grad.scalar_type()),
                      grad_x.mutable_data_ptr(), stream_of(grad)));
    return grad_x;
  }
  py::gil_scoped_acquire gil;
  return py::reinterpret_borrow<py::object>(g_topk_grad_any)(grad_values, indices, n, k0, j, interleaved).cast<Tensor>();
}

TORCH_LIBRARY_IMPL(approx_topk, CUDA, m) {
  m.impl("topk", TORCH_FN(topk));
  m.impl("topk_grad", TORCH_FN(topk_grad));
}

// ---- the operator with its gradient ----
Tensor call_topk_grad(const Tensor& grad_values, const Tensor& indices, int64_t n, int64_t k0, int64_t j, bool interleaved) {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("approx_topk::topk_grad", "")
                             .typed<Tensor(const Tensor&, const Tensor&, c10::SymInt, c10::SymInt, c10::SymInt, bool)>();
  return op.call(grad_values, indices, n, k0, j, interleaved);
}

struct TopkWithGradient : torch::autograd::Function<TopkWithGradient> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& xs, int64_t k,
                                                int64_t dim, int64_t j, int64_t k_mult, bool interleaved,
                                                optional<bool> multithread_buckets) {
    static const auto op =
        c10::Dispatcher::singleton()
            .findSchemaOrThrow("approx_topk::topk", "")
            .typed<std::tuple<Tensor, Tensor>(const Tensor&, c10::SymInt, c10::SymInt, c10::SymInt, c10::SymInt, bool,
                                              optional<bool>)>();
    at::AutoDispatchBelowADInplaceOrView guard;
    auto [values, indices] = op.call(xs, k, dim, j, k_mult, interleaved, multithread_buckets);
    std::vector<int64_t> call = {dim >= 0 ? dim : dim + xs.dim(), k * k_mult, j, interleaved, (int64_t)xs.scalar_type()};
    call.insert(call.end(), xs.sizes().begin(), xs.sizes().end());
    ctx->saved_data["call"] = std::move(call);
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({indices});
    // (not marked as non-differentiable: integers are not anyway, and compiled autograd takes no node with marks)
    return {values, indices};
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 const torch::autograd::variable_list& grads) {
    const Tensor indices = ctx->get_saved_variables()[0];
    const std::vector<int64_t> call = ctx->saved_data["call"].toIntVector();
    const int64_t dim = call[0], k0 = call[1], j = call[2];
    const bool interleaved = call[3] != 0;
    const at::IntArrayRef shape = at::IntArrayRef(call).slice(5);
    const Tensor& grad = grads[0];
    Tensor grad_xs;
    // a plain gradient whose own derivative nobody asks for: the operator's autograd kernel would find nothing to do
    if (grad.defined() && !shape.empty() && dim == (int64_t)shape.size() - 1 && indices.numel() && shape.back() <= kMaxGradRow &&
        plain(grad) && !(at::GradMode::is_enabled() && grad.requires_grad()) && !grad._fw_grad(0).defined() &&
        !at::impl::torch_function_mode_enabled()) {
      at::AutoDispatchBelowAutograd guard;
      grad_xs = call_topk_grad(grad, indices, shape.back(), k0, j, interleaved);
    } else {
      py::gil_scoped_acquire gil;
      py::tuple sizes(shape.size());
      for (size_t d = 0; d < shape.size(); ++d) sizes[d] = shape[d];
      const py::object dtype = py::reinterpret_borrow<py::object>((PyObject*)torch::getTHPDtype((at::ScalarType)call[4]));
      grad_xs = py::reinterpret_borrow<py::object>(g_gradient_any)(grad.defined() ? py::cast(grad) : py::object(py::none()),
                                                                   indices, sizes, dtype, dim, k0, j, interleaved)
                    .cast<Tensor>();
    }
    return {grad_xs, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

template <typename F> void take(F& fn, const py::dict& addresses, const char* name) {
  fn = reinterpret_cast<F>(addresses[name].cast<uintptr_t>());
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.attr("built_for") = ATK_BUILT_FOR;
  m.def("set_general", [](py::object topk_any, py::object topk_grad_any) {
    g_topk_any = topk_any.release().ptr();
    g_topk_grad_any = topk_grad_any.release().ptr();
  });
  m.def("set_gradient", [](py::object gradient_any) { g_gradient_any = gradient_any.release().ptr(); });
  m.def("bind", [](const py::dict& addresses) {
    if (bound()) return;  // (the library stays the one that was loaded first)
    take(g_strerror, addresses, "atk_strerror");
    take(g_stage1_workspace, addresses, "atk_stage1_workspace_bytes");
    take(g_stage1, addresses, "atk_stage1");
    take(g_stage1_i32, addresses, "atk_stage1_i32");
    take(g_topk_workspace, addresses, "atk_topk_workspace_bytes_used");
    take(g_topk_i32, addresses, "atk_topk_i32");
    take(g_topk_grad, addresses, "atk_topk_grad");
    take(g_topk, addresses, "atk_topk");
    g_bound.store(true, std::memory_order_release);
  });
  // None where the rows are not the common case
  m.def("run", [](const Tensor& xs, int64_t k0, int64_t j, int64_t k, int layout, bool narrow, bool want_values,
                  bool two_stage) -> py::object {
    if (!rows_in_place(xs) || k0 < 1 || k < 1 || j < 1 || j > 4) return py::none();
    std::tuple<Tensor, Tensor> out;
    {
      py::gil_scoped_release no_gil;
      out = run_rows(xs, k0, j, k, layout, narrow, want_values, two_stage);
    }
    return py::make_tuple(want_values ? py::cast(std::get<0>(out)) : py::none(), std::get<1>(out));
  });
  m.def("differentiable_topk", [](const Tensor& xs, int64_t k, int64_t dim, int64_t j, int64_t k_mult, bool interleaved,
                                  optional<bool> multithread_buckets) {
    py::gil_scoped_release no_gil;
    auto out = TopkWithGradient::apply(xs, k, dim, j, k_mult, interleaved, multithread_buckets);
    return std::make_tuple(out[0], out[1]);
  });
  // arguments of other types: None, for the Python function that accepts or refuses them
  m.def("run", [](const py::args&) { return py::none(); });
  m.def("differentiable_topk", [](const py::args&) { return py::none(); });
}
