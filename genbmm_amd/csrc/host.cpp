// The eager route of logbmm, maxbmm, prodmaxbmm, samplebmm and of the banded products (+,x), log and max in native
// code: checks, allocations, the library calls and the autograd nodes of genmul.py's and sparse.py's Functions, for
// operands that need no conversion.
//
// What it is for: a small product's forward and gradients wait for the host.  A Python node costs its own
// construction, a hand-over of the interpreter lock to the autograd engine's thread and back, and a nested node
// for logbmm's first backward; (16, 64^3) forward and both gradients, 25 us of kernels:
// 107 us by the Python Functions, 54 here, 49 for one multiplication of torch's own with its gradients.  Narrow bands
// likewise: 129 x 247, 6 and 12 diagonals, multiply with both gradients 91 -> 53 us, 98 x 641, 30 and 17, multiply_max 91 -> 53.
//
// Which calls it takes (`plain`): tensors of the exact types Tensor / Parameter, float32 / float16 / bfloat16, 3-D,
// contiguous, of one batch size, on one GPU, without a forward-mode tangent, under no trace, dispatch mode or functorch
// transform, whose reduction is not cut in Python; band tensors (`plain_bands`) likewise, of one size, whose widths are
// those of their bands and which no dense product takes the place of.  For any other the functions return None and
// the Python side goes on as it does without them - conversions, double precision, the messages of what is refused.
#include <ATen/core/TorchDispatchUtils.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <algorithm>

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

// ------------------------------------------------------------ banded products
struct Bands {
  int a_lu, a_ld, b_lu, b_ld;
};
Bands bands_of(AutogradContext* ctx) {
  const auto v = ctx->saved_data["bands"].toIntVector();
  return {(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
}

// saved: the operands and what the forward left beside the result - the index of every cell (max), the result and the
// workspace (log), nothing ((+,x))
template <int MODE>
struct BandProduct : torch::autograd::Function<BandProduct<MODE>> {
  static constexpr bool kLog = MODE == GENBMM_BAND_LOG, kMax = MODE == GENBMM_BAND_MAX;
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b, int64_t a_lu, int64_t a_ld, int64_t b_lu,
                        int64_t b_ld) {
    const c10::DeviceGuard guard(a.device());
    const Bands w{(int)a_lu, (int)a_ld, (int)b_lu, (int)b_ld};
    const int B = a.size(0), n = a.size(1);
    Tensor out = at::empty({B, n, a.size(2) + b.size(2) - 1}, a.options()), idx, ws;
    if (kMax) idx = at::empty(out.sizes(), a.options().dtype(at::kInt));
    if (kLog) ws = at::empty({(int64_t)genbmm_banded_workspace_size(w.a_lu, w.a_ld, w.b_lu, w.b_ld, B, n)}, workspace(a));
    check(GENBMM_BY_TYPE(a, genbmm_banded_fwd, at_<E>(a), w.a_lu, w.a_ld, at_<E>(b), w.b_lu, w.b_ld, at_<E>(out),
                         kMax ? at_<int32_t>(idx) : nullptr, kLog ? at_<float>(ws) : nullptr, B, n, MODE, stream_of(a)),
          "genbmm_banded_fwd");
    if (kLog) ctx->save_for_backward({a, b, out, ws});
    else if (kMax) ctx->save_for_backward({a, b, idx});
    else ctx->save_for_backward({a, b});
    ctx->saved_data["bands"] = std::vector<int64_t>{a_lu, a_ld, b_lu, b_ld};
    ctx->saved_data["type"] = a.scalar_type();
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &a = saved[0], &b = saved[1];
    const Tensor g = incoming(grads[0], ctx->saved_data["type"].toScalarType());
    const Bands w = bands_of(ctx);
    const at::ScalarType type = g.scalar_type();
    const int64_t B = g.size(0), n = g.size(1), wa = w.a_lu + w.a_ld + 1, wb = w.b_lu + w.b_ld + 1;
    require(g, "the incoming gradient", g, type, {B, n, wa + wb - 1});
    require(a, "a", g, type, {B, n, wa});
    require(b, "b", g, type, {B, n, wb});
    Tensor out, ws, scratch;
    if (kMax) require(saved[2], "the indices", g, at::kInt, g.sizes());
    if (kLog) {
      out = saved[2].detach();  // as a value (LogBmm)
      ws = saved[3];
      require(out, "the result", g, type, g.sizes());
      require(ws, "the forward's workspace", g, at::kFloat,
              {(int64_t)genbmm_banded_workspace_size(w.a_lu, w.a_ld, w.b_lu, w.b_ld, (int)B, (int)n)});
      if (at::GradMode::is_enabled() || has_tangent(g) || has_tangent(a) || has_tangent(b)) {
        const py::gil_scoped_acquire gil;
        const py::tuple r = py::module_::import("genbmm_amd.sparse")
                                .attr("_BandedLogGrad")
                                .attr("apply")(a, b, g, out, ws, py::make_tuple(w.a_lu, w.a_ld, w.b_lu, w.b_ld));
        return {r[0].cast<Tensor>(), r[1].cast<Tensor>(), Variable(), Variable(), Variable(), Variable()};
      }
    }
    const c10::DeviceGuard guard(g.device());
    Tensor ga = at::empty_like(a), gb = at::empty_like(b);
    if (kLog) {  // (a buffer of this call's own: see sparse._backward)
      const int64_t need = genbmm_banded_scratch_size(w.a_lu, w.a_ld, w.b_lu, w.b_ld, (int)B, (int)n);
      if (need > 0) scratch = at::empty({need}, workspace(g));
    }
    check(GENBMM_BY_TYPE(g, genbmm_banded_bwd_scratch, at_<E>(a), w.a_lu, w.a_ld, at_<E>(b), w.b_lu, w.b_ld,
                         kLog ? at_<E>(out) : nullptr, kMax ? at_<int32_t>(saved[2]) : nullptr,
                         kLog ? at_<float>(ws) : nullptr, scratch.defined() ? at_<float>(scratch) : nullptr, at_<E>(g),
                         at_<E>(ga), at_<E>(gb), (int)B, (int)n, MODE, stream_of(g)),
          "genbmm_banded_bwd_scratch");
    return {ga, gb, Variable(), Variable(), Variable(), Variable()};
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

constexpr int64_t kMost = 0x7fffffff;

// two 3-D contiguous tensors of one type and one GPU, with nothing around them
bool plain_pair(const py::handle& pa, const py::handle& pb) {
  if (!THPVariable_CheckExact(pa.ptr()) || !THPVariable_CheckExact(pb.ptr())) return false;
  const Tensor &a = THPVariable_Unpack(pa.ptr()), &b = THPVariable_Unpack(pb.ptr());
  if (!bare(a) || !bare(b) || a.dim() != 3 || b.dim() != 3 || a.scalar_type() != b.scalar_type() || a.device() != b.device())
    return false;
  const at::ScalarType type = a.scalar_type();
  if (type != at::kFloat && type != at::kHalf && type != at::kBFloat16) return false;
  return a.is_contiguous() && b.is_contiguous() && !has_tangent(a) && !has_tangent(b);
}

bool plain(const py::handle& pa, const py::handle& pb) {
  if (!plain_pair(pa, pb)) return false;
  const Tensor &a = THPVariable_Unpack(pa.ptr()), &b = THPVariable_Unpack(pb.ptr());
  const int64_t B = a.size(0), M = a.size(1), K = a.size(2), N = b.size(2);
  if (b.size(0) != B || b.size(1) != K || B > kMost || M > kMost || N > kMost) return false;
  if (K >= 4096) return false;  // genmul._reduction_splits may cut it
  return eager();
}

// `dense`: a product that sparse._dense_pays may send through dense matrices where both bands are wide
bool plain_bands(const py::handle& pa, int64_t a_lu, int64_t a_ld, const py::handle& pb, int64_t b_lu, int64_t b_ld, bool dense) {
  if (!plain_pair(pa, pb)) return false;
  const Tensor &a = THPVariable_Unpack(pa.ptr()), &b = THPVariable_Unpack(pb.ptr());
  const int64_t B = a.size(0), n = a.size(1), wa = a.size(2), wb = b.size(2);
  if (b.size(0) != B || b.size(1) != n || std::min({a_lu, a_ld, b_lu, b_ld}) < 0) return false;
  if (B > kMost || n > kMost || wa > kMost || wb > kMost || wa != a_lu + a_ld + 1 || wb != b_lu + b_ld + 1) return false;
  if (dense && std::min(wa, wb) > 128) return false;
  return eager();
}

template <class F>
py::object on(const py::handle& pa, const py::handle& pb, bool takes, F&& f) {
  if (!takes) return py::none();
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
    return on(a, b, plain(a, b), [&](const Tensor& x, const Tensor& y) {
      return LogBmm::apply(x, y, x.scalar_type() == at::kFloat ? path : half_path);
    });
  });
  m.def("maxbmm", [](const py::handle& a, const py::handle& b) {
    return on(a, b, plain(a, b), [](const Tensor& x, const Tensor& y) { return MaxBmm::apply(x, y); });
  });
  m.def("prodmaxbmm", [](const py::handle& a, const py::handle& b) {
    return on(a, b, plain(a, b), [](const Tensor& x, const Tensor& y) { return ProdMaxBmm::apply(x, y); });
  });
#define GENBMM_BAND(name, mode, dense)                                                                             \
  m.def(name, [](const py::handle& a, int64_t a_lu, int64_t a_ld, const py::handle& b, int64_t b_lu, int64_t b_ld) { \
    return on(a, b, plain_bands(a, a_lu, a_ld, b, b_lu, b_ld, dense), [&](const Tensor& x, const Tensor& y) {        \
      return BandProduct<mode>::apply(x, y, a_lu, a_ld, b_lu, b_ld);                                                 \
    });                                                                                                              \
  })
  GENBMM_BAND("band_mul", GENBMM_BAND_MUL, true);
  GENBMM_BAND("band_log", GENBMM_BAND_LOG, true);
  GENBMM_BAND("band_max", GENBMM_BAND_MAX, false);
  m.def("samplebmm", [](const py::handle& a, const py::handle& b, uint64_t seed, uint64_t offset) {
    return on(a, b, plain(a, b), [&](const Tensor& x, const Tensor& y) { return SampleBmm::apply(x, y, (int64_t)seed, (int64_t)offset); });
  });
}
