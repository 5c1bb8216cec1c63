// The eager route of logbmm, maxbmm, prodmaxbmm and samplebmm in native code: checks, allocations, the library
// calls and the autograd nodes of genmul.py's Functions, for operands that need no conversion.
//
// What it is for: a small product's forward and gradients wait for the host.  A Python node costs its own
// construction, a hand-over of the interpreter lock to the autograd engine's thread and back, and a nested node
// for logbmm's first backward; (16, 64^3) forward and both gradients, 25 us of kernels:
// 107 us by the Python Functions, 54 here, 49 for one multiplication of torch's own with its gradients.
//
// Which calls it takes (`plain`): tensors of the exact types Tensor / Parameter, float32 / float16 / bfloat16, 3-D,
// contiguous, of one batch size, on one GPU, without a forward-mode tangent, under no trace, dispatch mode or functorch
// transform, whose reduction is not cut in Python.  For any other the functions return None and genmul.py goes on as
// it does without them - conversions, double precision, the messages of what is refused.
#include <ATen/core/TorchDispatchUtils.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include "genbmm_gfx950.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }

void check(int code, const char* what) {
  TORCH_CHECK(code == 0, "genbmm_amd: ", what, " failed (", code, "): ", genbmm_error_string(code));
}

template <class T>
T* at_(const Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}

// f(entry point of t's element type, pointer to an element of that type)
#define GENBMM_BY_TYPE(t, name, ...)                                                    \
  [&] {                                                                                 \
    switch ((t).scalar_type()) {                                                        \
      case at::kHalf: { using E = uint16_t; return name##_f16(__VA_ARGS__); }           \
      case at::kBFloat16: { using E = uint16_t; return name##_bf16(__VA_ARGS__); }      \
      default: { using E = float; return name(__VA_ARGS__); }                           \
    }                                                                                   \
  }()

struct Dims {
  int B, M, K, N;
};
Dims dims_of(const Tensor& a, const Tensor& b) { return {(int)a.size(0), (int)a.size(1), (int)a.size(2), (int)b.size(2)}; }

at::TensorOptions workspace(const Tensor& t) { return t.options().dtype(at::kFloat); }

// `g` as the kernels read it: contiguous() keeps the lazy negative bit of a tensor whose strides already fit
Tensor incoming(const Tensor& g, at::ScalarType type) { return g.to(type).contiguous().resolve_neg(); }

// A saved-tensor hook may hand back something else than it was given: a tensor on the host, of another type, size or
// order or with the lazy negative bit is refused here, before its address reaches a kernel.
void require(const Tensor& t, const char* name, const Tensor& like, at::ScalarType type, at::IntArrayRef sizes) {
  TORCH_CHECK(t.is_cuda() && t.device() == like.device(), name, " is on ", t.device(), ", expected ", like.device());
  TORCH_CHECK(t.scalar_type() == type, name, " must be ", type, ", got ", t.scalar_type());
  TORCH_CHECK(!t.is_neg(), name, " has the lazy negative bit: no memory holds its values");
  TORCH_CHECK(t.is_contiguous() && t.sizes() == sizes, name, " must be contiguous, of sizes ", sizes, ", got ", t.sizes());
}

// a forward-mode tangent: a C++ node refuses it as a RuntimeError, the Python nodes as its NotImplementedError
bool has_tangent(const Tensor& t) { return t._fw_grad(/*level=*/0).defined(); }

// -------------------------------------------------------------------- logbmm
struct LogBmm : torch::autograd::Function<LogBmm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b, int64_t path) {
    const c10::DeviceGuard guard(a.device());
    const Dims d = dims_of(a, b);
    Tensor out = at::empty({d.B, d.M, d.N}, a.options());
    Tensor stats = at::empty({(int64_t)genbmm_logbmm_stats_size_path(d.B, d.M, d.K, d.N, (int)path)}, workspace(a));
    check(GENBMM_BY_TYPE(a, genbmm_logbmm_fwd_path, at_<E>(a), at_<E>(b), at_<E>(out), at_<float>(stats), d.B, d.M, d.K,
                         d.N, (int)path, stream_of(a)),
          "genbmm_logbmm_fwd_path");
    ctx->save_for_backward({a, b, out, stats});
    ctx->saved_data["path"] = path;
    ctx->saved_data["type"] = a.scalar_type();
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &a = saved[0], &b = saved[1];
    // `out` as a value: what it owes to a and b is part of the gradients' own derivative
    const Tensor g = incoming(grads[0], ctx->saved_data["type"].toScalarType()), out = saved[2].detach();
    const int64_t path = ctx->saved_data["path"].toInt();
    TORCH_CHECK(a.dim() == 3 && b.dim() == 3, "a and b must have 3 dimensions");
    const Dims d = dims_of(a, b);
    const at::ScalarType type = g.scalar_type();
    require(g, "the incoming gradient", g, type, {d.B, d.M, d.N});
    require(a, "a", g, type, {d.B, d.M, d.K});
    require(b, "b", g, type, {d.B, d.K, d.N});
    require(out, "the result", g, type, {d.B, d.M, d.N});
    require(saved[3], "the forward's workspace", g, at::kFloat,
            {(int64_t)genbmm_logbmm_stats_size_path(d.B, d.M, d.K, d.N, (int)path)});
    // differentiated again, where the Python node has the formula, or along a tangent, which it refuses
    if (at::GradMode::is_enabled() || has_tangent(g) || has_tangent(a) || has_tangent(b)) {
      const py::gil_scoped_acquire gil;
      const py::tuple r = py::module_::import("genbmm_amd.genmul").attr("_LogBmmGrad").attr("apply")(a, b, g, out, saved[3], path);
      return {r[0].cast<Tensor>(), r[1].cast<Tensor>(), Variable()};
    }
    const c10::DeviceGuard guard(a.device());
    Tensor ga = at::empty_like(a), gb = at::empty_like(b);
    check(GENBMM_BY_TYPE(a, genbmm_logbmm_bwd_path, at_<E>(a), at_<E>(b), at_<E>(out), at_<E>(g), at_<float>(saved[3]),
                         at_<E>(ga), at_<E>(gb), d.B, d.M, d.K, d.N, (int)path, stream_of(a)),
          "genbmm_logbmm_bwd_path");
    return {ga, gb, Variable()};
  }
};

// ------------------------------------------------- max / sample / prod-max
// saved: the index of every cell and, for the product semiring, the two factors of its term
variable_list argmax_backward(AutogradContext* ctx, const Tensor& grad, bool prod) {
  const variable_list saved = ctx->get_saved_variables();
  const Tensor& idx = saved[0];
  const at::ScalarType type = ctx->saved_data["type"].toScalarType();
  const int B = grad.size(0), M = grad.size(1), K = ctx->saved_data["K"].toInt(), N = grad.size(2);
  const Tensor g = incoming(grad, type);
  require(g, "the incoming gradient", g, type, {B, M, N});
  require(idx, "the indices", g, at::kInt, {B, M, N});
  if (prod) require(saved[1], "the factors", g, at::kFloat, {2, B, M, N});
  const c10::DeviceGuard guard(g.device());
  Tensor ga = at::empty({B, M, K}, g.options()), gb = at::empty({B, K, N}, g.options());
  if (prod)
    check(GENBMM_BY_TYPE(g, genbmm_prodmax_bwd, nullptr, nullptr, at_<int32_t>(idx), at_<float>(saved[1]), at_<E>(g),
                         at_<E>(ga), at_<E>(gb), B, M, K, N, stream_of(g)),
          "genbmm_prodmax_bwd");
  else
    check(GENBMM_BY_TYPE(g, genbmm_argmax_bwd, at_<int32_t>(idx), at_<E>(g), at_<E>(ga), at_<E>(gb), B, M, K, N,
                         stream_of(g)),
          "genbmm_argmax_bwd");
  return {ga, gb};
}
void keep_dims(AutogradContext* ctx, const Tensor& a) {
  ctx->saved_data["type"] = a.scalar_type();
  ctx->saved_data["K"] = a.size(2);
}

struct MaxBmm : torch::autograd::Function<MaxBmm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b) {
    const c10::DeviceGuard guard(a.device());
    const Dims d = dims_of(a, b);
    Tensor out = at::empty({d.B, d.M, d.N}, a.options()), idx = at::empty({d.B, d.M, d.N}, a.options().dtype(at::kInt));
    check(GENBMM_BY_TYPE(a, genbmm_maxbmm_fwd, at_<E>(a), at_<E>(b), at_<E>(out), at_<int32_t>(idx), d.B, d.M, d.K, d.N,
                         stream_of(a)),
          "genbmm_maxbmm_fwd");
    ctx->save_for_backward({idx});
    keep_dims(ctx, a);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) { return argmax_backward(ctx, grads[0], false); }
};

struct ProdMaxBmm : torch::autograd::Function<ProdMaxBmm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b) {
    const c10::DeviceGuard guard(a.device());
    const Dims d = dims_of(a, b);
    Tensor out = at::empty({d.B, d.M, d.N}, a.options()), idx = at::empty({d.B, d.M, d.N}, a.options().dtype(at::kInt));
    Tensor factors = at::empty({2, d.B, d.M, d.N}, workspace(a));
    check(GENBMM_BY_TYPE(a, genbmm_prodmaxbmm_fwd, at_<E>(a), at_<E>(b), at_<E>(out), at_<int32_t>(idx),
                         at_<float>(factors), d.B, d.M, d.K, d.N, stream_of(a)),
          "genbmm_prodmaxbmm_fwd");
    ctx->save_for_backward({idx, factors});
    keep_dims(ctx, a);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) { return argmax_backward(ctx, grads[0], true); }
};

struct SampleBmm : torch::autograd::Function<SampleBmm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b, int64_t seed, int64_t offset) {
    const c10::DeviceGuard guard(a.device());
    const Dims d = dims_of(a, b);
    Tensor out = at::empty({d.B, d.M, d.N}, a.options()), idx = at::empty({d.B, d.M, d.N}, a.options().dtype(at::kInt));
    Tensor stats = at::empty({(int64_t)genbmm_samplebmm_stats_size(d.B, d.M, d.K, d.N)}, workspace(a));
    check(GENBMM_BY_TYPE(a, genbmm_samplebmm_fwd, at_<E>(a), at_<E>(b), at_<E>(out), at_<int32_t>(idx), at_<float>(stats),
                         (uint64_t)seed, (uint64_t)offset, d.B, d.M, d.K, d.N, stream_of(a)),
          "genbmm_samplebmm_fwd");
    ctx->save_for_backward({idx});
    keep_dims(ctx, a);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list r = argmax_backward(ctx, grads[0], false);
    r.resize(4);
    return r;
  }
};

// ------------------------------------------------------------------ entry
// A GPU tensor with storage of its own and nothing in front of it: what is not one of these keys is a wrapper
// (functorch, a fake or proxy tensor, a Python subclass), a lazy conjugate or negative, or another layout.
bool bare(const Tensor& t) {
  constexpr c10::DispatchKeySet known =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA,
                           c10::DispatchKey::AutocastCUDA});
  return t.is_cuda() && t.layout() == at::kStrided && (t.key_set() - known).highestFunctionalityKey() == c10::DispatchKey::Undefined && t.has_storage();
}

// nothing around the call that records or replaces torch operations
bool eager() {
  return !torch::jit::tracer::isTracing() && !c10::impl::dispatch_mode_enabled() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

bool plain(const py::handle& pa, const py::handle& pb) {
  if (!THPVariable_CheckExact(pa.ptr()) || !THPVariable_CheckExact(pb.ptr())) return false;
  const Tensor &a = THPVariable_Unpack(pa.ptr()), &b = THPVariable_Unpack(pb.ptr());
  if (!bare(a) || !bare(b) || a.dim() != 3 || b.dim() != 3 || a.scalar_type() != b.scalar_type() || a.device() != b.device())
    return false;
  const at::ScalarType type = a.scalar_type();
  if (type != at::kFloat && type != at::kHalf && type != at::kBFloat16) return false;
  const int64_t B = a.size(0), M = a.size(1), K = a.size(2), N = b.size(2);
  if (b.size(0) != B || b.size(1) != K || !a.is_contiguous() || !b.is_contiguous()) return false;
  if (has_tangent(a) || has_tangent(b)) return false;
  constexpr int64_t most = 0x7fffffff;
  if (B > most || M > most || N > most) return false;
  if (K >= 4096) return false;  // genmul._reduction_splits may cut it
  return eager();
}

template <class F>
py::object on(const py::handle& pa, const py::handle& pb, F&& f) {
  if (!plain(pa, pb)) return py::none();
  const Tensor a = THPVariable_Unpack(pa.ptr()), b = THPVariable_Unpack(pb.ptr());
  Tensor out;
  {
    const py::gil_scoped_release nogil;
    out = f(a, b);
  }
  return py::cast(out);
}

// What _lib.py asks of every tensor of the Python Functions' calls, some twenty times in a product and its gradients:
// plain C functions, since a method of the tensor or a pybind11 function takes 100 to 200 ns.  Forward and gradients of
// a small product on one machine: without any look at the negative bit multiply_log 126 us, logbmm on 4-D operands 163;
// here 116 and 154 (on one that was twice as fast: 61 and 88 without, 63 and 93 with the look taken in Python).
PyObject* is_dense(PyObject*, PyObject* o) {  // already as the kernels read it, and nobody watches torch make sure
  HANDLE_TH_ERRORS
  if (THPVariable_CheckExact(o)) {
    const Tensor& t = THPVariable_Unpack(o);
    if (bare(t) && t.is_contiguous() && eager()) Py_RETURN_TRUE;
  }
  Py_RETURN_FALSE;
  END_HANDLE_TH_ERRORS
}
PyObject* address(PyObject*, PyObject* o) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor");
  const Tensor& t = THPVariable_Unpack(o);
  TORCH_CHECK(!t.is_neg(), "genbmm_amd: a tensor with the lazy negative bit has no memory that holds its values");
  return PyLong_FromVoidPtr(t.data_ptr());
  END_HANDLE_TH_ERRORS
}
PyMethodDef kMethods[] = {{"is_dense", is_dense, METH_O, nullptr}, {"address", address, METH_O, nullptr}, {}};

}  // namespace

PYBIND11_MODULE(_host, m) {
  if (PyModule_AddFunctions(m.ptr(), kMethods) != 0) throw py::error_already_set();
  m.def("plain", &plain);
  m.def("logbmm", [](const py::handle& a, const py::handle& b, int64_t path, int64_t half_path) {
    return on(a, b, [&](const Tensor& x, const Tensor& y) {
      return LogBmm::apply(x, y, x.scalar_type() == at::kFloat ? path : half_path);
    });
  });
  m.def("maxbmm", [](const py::handle& a, const py::handle& b) {
    return on(a, b, [](const Tensor& x, const Tensor& y) { return MaxBmm::apply(x, y); });
  });
  m.def("prodmaxbmm", [](const py::handle& a, const py::handle& b) {
    return on(a, b, [](const Tensor& x, const Tensor& y) { return ProdMaxBmm::apply(x, y); });
  });
  m.def("samplebmm", [](const py::handle& a, const py::handle& b, uint64_t seed, uint64_t offset) {
    return on(a, b, [&](const Tensor& x, const Tensor& y) { return SampleBmm::apply(x, y, (int64_t)seed, (int64_t)offset); });
  });
}
