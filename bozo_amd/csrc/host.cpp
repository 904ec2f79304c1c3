// The eager call path in native code: output and workspace allocation, the
// tension_buf descriptors, the library call and the autograd nodes of the
// window op, the global block, RoPE and the decode step.
//
// A forward + backward through Python autograd Functions and ctypes cost the
// host about 170 us, most of it in the engine's device thread (the GIL taken
// there, a dozen descriptors built by ctypes), while the kernels of a training
// layer take 27 to 130 us.  Forward + backward: B4 H4 T256 d32 W32 float32 190
// -> 69 us (kernels 27), B32 H12 T1024 d64 W64 bf16 172 -> 113 (the kernels'
// own time); a decode step of 64 sequences 19.7 -> 11.2 us (likewise).
//
// The GIL is released for the whole call, as ctypes does.  Nothing is kept
// from one call for the next.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>

#include "tension_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

PyObject* g_tension_error = nullptr;  // bozo_amd._lib.TensionError

struct TensionFail : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check(int status, const char* what) {
  if (status == TENSION_OK) return;
  const char* kind = status == TENSION_ERR_ARG           ? "bad argument"
                     : status == TENSION_ERR_UNSUPPORTED ? "unsupported"
                     : status == TENSION_ERR_LAUNCH      ? "launch failure"
                                                         : "error";
  throw TensionFail(std::string(what) + ": " + kind + ": " + tension_last_error());
}

// A failure inside the backward crosses the engine as a Python exception, so
// it reaches the caller as TensionError there too.
template <typename F>
auto in_backward(F f) -> decltype(f()) {
  try {
    return f();
  } catch (const TensionFail& e) {
    py::gil_scoped_acquire gil;
    PyErr_SetString(g_tension_error, e.what());
    python_error pe;
    pe.persist();
    throw pe;
  }
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return TENSION_F32;
    case at::kBFloat16: return TENSION_BF16;
    case at::kHalf: return TENSION_F16;
    case at::kDouble: return TENSION_F64;
    default: return -1;
  }
}

// One tensor's descriptor; get() is null for an absent tensor.  `written`: the
// kernels write it, so a lazily cloned tensor gets memory of its own first (its
// storage is shared until a mutable pointer is taken).
struct Buf {
  tension_buf b{};
  bool on = false;
  Buf() = default;
  explicit Buf(const Tensor& t, bool written = false) {
    if (!t.defined()) return;
    const int code = dtype_code(t);
    if (code < 0) throw py::type_error(std::string("unsupported dtype ") + c10::toString(t.scalar_type()));
    if (t.dim() > 4) throw py::value_error("a tension_buf describes at most 4 dimensions");
    on = true;
    b.ptr = written ? t.mutable_data_ptr() : const_cast<void*>(t.const_data_ptr());
    b.dtype = code;
    for (int64_t i = 0; i < t.dim(); ++i) b.s[i] = t.stride(i);
  }
  const tension_buf* get() const { return on ? &b : nullptr; }
};
Buf written(const Tensor& t) { return Buf(t, true); }

// Unit innermost stride is all the kernels need.
Tensor rows(const Tensor& t) {
  if (!t.defined()) return t;
  return t.dim() == 0 || t.stride(-1) != 1 || t.numel() == 0 ? t.contiguous() : t;
}

Tensor opt(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

// Side inputs (bias) in float32, or float64 for float64 calls.
Tensor side(const Tensor& t, const Tensor& like) {
  if (!t.defined()) return t;
  return rows(t.to(like.scalar_type() == at::kDouble ? at::kDouble : at::kFloat));
}

tension_stream_t stream_of(const Tensor& t) {
  const hipStream_t s = c10::hip::getCurrentHIPStream(t.device().index());
  return (tension_stream_t)s;
}

Tensor empty(at::IntArrayRef shape, at::ScalarType dt, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(dt).device(like.device()));
}
Tensor empty(at::IntArrayRef shape, const Tensor& like) { return empty(shape, like.scalar_type(), like); }

int acc_code(const Tensor& q, const Tensor& k, const Tensor& v) {
  return q.scalar_type() == at::kDouble || k.scalar_type() == at::kDouble || v.scalar_type() == at::kDouble ? TENSION_F64
                                                                                                           : TENSION_F32;
}

Tensor workspace(int64_t bytes, const Tensor& like) {
  return bytes > 0 ? empty({bytes}, at::kByte, like) : Tensor();
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// ------------------------------------------------------------- local window

// Tau-mass with float32 Q / K at head dim 32 / 64, where the backward takes its
// coefficients from the forward's rows: with a bf16 V (the reference's autocast
// flow) for windows wider than 64 (narrower bands form them in registers, which
// is faster), with a float32 V at every window (its dQ kernel keeps no band in
// registers).
bool saved_rows_flow(const Tensor& Q, const Tensor& K, const Tensor& V, int64_t W, int64_t flags) {
  const int64_t D = Q.size(-1);
  if (!(flags & TENSION_NORM_MASS) || Q.scalar_type() != at::kFloat || K.scalar_type() != at::kFloat ||
      (D != 32 && D != 64))
    return false;
  if (V.scalar_type() == at::kBFloat16) return W > 64;
  return V.scalar_type() == at::kFloat;
}

// (out, tau, mass); tau and mass undefined unless asked for.
std::tuple<Tensor, Tensor, Tensor> window_fwd(const Tensor& Q, const Tensor& K, const Tensor& V, const Tensor& bias,
                                              int64_t W, double scale, int64_t flags, bool want_tau, bool want_mass) {
  const c10::DeviceGuard guard(Q.device());
  const int64_t B = Q.size(0), T = Q.size(1), H = Q.size(2), D = Q.size(3);
  Tensor out = empty(Q.sizes(), Q), tau, mass;
  if (want_tau) tau = empty({B, T, H, W}, Q);
  if (want_mass) mass = empty({B, T, H}, at::kFloat, Q);
  const Buf q(Q), k(K), v(V), o = written(out), t = written(tau), b(bias), m = written(mass);
  check(tension_window_fwd(q.get(), k.get(), v.get(), o.get(), t.get(), b.get(), m.get(), B, T, H, D, W, scale,
                           (int32_t)flags, stream_of(Q)),
        "tension_window_fwd");
  return {out, tau, mass};
}

std::tuple<Tensor, Tensor, Tensor> window_bwd(const Tensor& Q, const Tensor& K, const Tensor& V, const Tensor& d_out,
                                              const Tensor& d_tau, const Tensor& bias, const Tensor& out,
                                              const Tensor& mass, int64_t W, double scale, int64_t flags) {
  const c10::DeviceGuard guard(Q.device());
  const int64_t B = Q.size(0), T = Q.size(1), H = Q.size(2), D = Q.size(3);
  const Tensor dOut = d_out.defined() ? rows(d_out) : at::zeros_like(Q), dTau = rows(d_tau);
  Tensor dQ = empty(Q.sizes(), Q), dK = empty(K.sizes(), K), dV = empty(V.sizes(), V);
  const Tensor ws = workspace(tension_window_bwd_workspace(B, T, H, acc_code(Q, K, V), (int32_t)flags), Q);
  const Buf q(Q), k(K), v(V), go(dOut), gt(dTau), b(bias), gq = written(dQ), gk = written(dK), gv = written(dV);
  if (out.defined()) {
    const Buf o(out), m(mass);
    check(tension_window_bwd_saved(q.get(), k.get(), v.get(), go.get(), gt.get(), b.get(), o.get(), m.get(), gq.get(),
                                   gk.get(), gv.get(), ptr(ws), B, T, H, D, W, scale, (int32_t)flags, stream_of(Q)),
          "tension_window_bwd_saved");
  } else {
    check(tension_window_bwd(q.get(), k.get(), v.get(), go.get(), gt.get(), b.get(), gq.get(), gk.get(), gv.get(),
                             ptr(ws), B, T, H, D, W, scale, (int32_t)flags, stream_of(Q)),
          "tension_window_bwd");
  }
  return {dQ, dK, dV};
}

struct WindowFn : torch::autograd::Function<WindowFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& Q, const Tensor& K, const Tensor& V,
                               const OptTensor& bias, int64_t W, double scale, int64_t flags, bool return_tau) {
    ctx->set_materialize_grads(false);  // an unused output's gradient stays absent
    const Tensor b = side(opt(bias), Q);
    const bool saved = saved_rows_flow(Q, K, V, W, flags);
    auto [out, tau, mass] = window_fwd(Q, K, V, b, W, scale, flags, return_tau, saved);
    ctx->save_for_backward({Q, K, V, b, saved ? out : Tensor(), mass});
    ctx->saved_data["W"] = W;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["flags"] = flags;
    if (return_tau) return {out, tau};
    return {out};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&]() -> variable_list {
      const variable_list s = ctx->get_saved_variables();
      auto [dQ, dK, dV] = window_bwd(s[0], s[1], s[2], g[0], g.size() > 1 ? g[1] : Tensor(), s[3], s[4], s[5],
                                     ctx->saved_data["W"].toInt(), ctx->saved_data["scale"].toDouble(),
                                     ctx->saved_data["flags"].toInt());
      return {dQ, dK, dV, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    });
  }
};

// ------------------------------------------------------------- global block

// (out, tau_local or undefined, mass): the tau mass per query is kept with the
// output, so the backward gets its per-query coefficients from these rows.
std::tuple<Tensor, Tensor, Tensor> global_fwd(const Tensor& Q, const Tensor& K, const Tensor& V, const Tensor& bias,
                                              double scale, int64_t Wl) {
  const c10::DeviceGuard guard(Q.device());
  const int64_t B = Q.size(0), T = Q.size(1), H = Q.size(2), D = Q.size(3);
  Tensor out = at::empty_like(Q), tl;
  if (Wl > 0) tl = empty({B, T, H, Wl}, Q);
  Tensor mass = empty({B, T, H}, at::kFloat, Q);
  const Buf q(Q), k(K), v(V), o = written(out), t = written(tl), b(bias), m = written(mass);
  check(tension_global_fwd(q.get(), k.get(), v.get(), o.get(), t.get(), b.get(), m.get(), B, T, H, D, Wl, scale, 0,
                           stream_of(Q)),
        "tension_global_fwd");
  return {out, tl, mass};
}

std::tuple<Tensor, Tensor, Tensor> global_bwd(const Tensor& Q, const Tensor& K, const Tensor& V, const Tensor& d_out,
                                              const Tensor& d_tl, const Tensor& bias, const Tensor& out,
                                              const Tensor& mass, int64_t Wl, double scale) {
  const c10::DeviceGuard guard(Q.device());
  const int64_t B = Q.size(0), T = Q.size(1), H = Q.size(2), D = Q.size(3);
  const Tensor dOut = d_out.defined() ? rows(d_out) : at::zeros_like(Q);
  const Tensor dTl = Wl > 0 ? rows(d_tl) : Tensor();
  Tensor dQ = empty(Q.sizes(), Q), dK = empty(K.sizes(), K), dV = empty(V.sizes(), V);
  const Tensor ws = workspace(tension_global_bwd_workspace(B, T, H, acc_code(Q, K, V), 0), Q);
  const Buf q(Q), k(K), v(V), go(dOut), gt(dTl), b(bias), o(out), m(mass), gq = written(dQ), gk = written(dK),
      gv = written(dV);
  check(tension_global_bwd(q.get(), k.get(), v.get(), go.get(), gt.get(), b.get(), o.get(), m.get(), gq.get(),
                           gk.get(), gv.get(), ptr(ws), B, T, H, D, Wl, scale, 0, stream_of(Q)),
        "tension_global_bwd");
  return {dQ, dK, dV};
}

struct GlobalFn : torch::autograd::Function<GlobalFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& Q, const Tensor& K, const Tensor& V,
                               const OptTensor& bias, double scale, int64_t Wl) {
    ctx->set_materialize_grads(false);
    const Tensor b = side(opt(bias), Q);
    auto [out, tl, mass] = global_fwd(Q, K, V, b, scale, Wl);
    ctx->save_for_backward({Q, K, V, b, out, mass});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["Wl"] = Wl;
    if (Wl > 0) return {out, tl};
    return {out};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&]() -> variable_list {
      const variable_list s = ctx->get_saved_variables();
      auto [dQ, dK, dV] = global_bwd(s[0], s[1], s[2], g[0], g.size() > 1 ? g[1] : Tensor(), s[3], s[4], s[5],
                                     ctx->saved_data["Wl"].toInt(), ctx->saved_data["scale"].toDouble());
      return {dQ, dK, dV, Tensor(), Tensor(), Tensor()};
    });
  }
};

// --------------------------------------------------------------------- RoPE

Tensor rope_call(const Tensor& x, const Tensor& cos, const Tensor& sin, int64_t pos_offset, at::ScalarType out_dtype,
                 int64_t inverse) {
  const c10::DeviceGuard guard(x.device());
  Tensor y = empty(x.sizes(), out_dtype, x);
  const Buf bx(x), by = written(y);
  check(tension_rope(bx.get(), by.get(), cos.data_ptr<float>(), sin.data_ptr<float>(), cos.size(0), x.size(0),
                     x.size(1), x.size(2), x.size(3), pos_offset, (int32_t)inverse, stream_of(x)),
        "tension_rope");
  return y;
}

struct RopeFn : torch::autograd::Function<RopeFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& cos, const Tensor& sin,
                        int64_t pos_offset, int64_t out_dtype) {
    ctx->save_for_backward({cos, sin});
    ctx->saved_data["pos"] = pos_offset;
    ctx->saved_data["dtype"] = (int64_t)x.scalar_type();
    return rope_call(x, cos, sin, pos_offset, (at::ScalarType)out_dtype, 0);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    return in_backward([&]() -> variable_list {
      const variable_list s = ctx->get_saved_variables();
      return {rope_call(rows(g[0]), s[0], s[1], ctx->saved_data["pos"].toInt(),
                        (at::ScalarType)ctx->saved_data["dtype"].toInt(), 1),
              Tensor(), Tensor(), Tensor(), Tensor()};
    });
  }
};

// ------------------------------------------------------------------- decode

// One step, or nothing when an operand does not fit the others (the caller
// then says which).
OptTensor decode_step(const Tensor& q, const Tensor& kn, const Tensor& vn, const Tensor& kc, const Tensor& vc,
                      const Tensor& pos_in, const OptTensor& pos_out_, double scale, int64_t flags,
                      const OptTensor& tau_) {
  const Tensor pos_out = opt(pos_out_), tau = opt(tau_);
  if (q.dim() != 3 || kc.dim() != 4 || !q.is_cuda()) return std::nullopt;
  const int64_t N = q.size(0), H = q.size(1), D = q.size(2), W = kc.size(2);
  auto same = [&](const Tensor& t) { return !t.defined() || t.device() == q.device(); };
  auto counter = [&](const Tensor& t) {
    return !t.defined() || (t.scalar_type() == at::kInt && t.dim() == 1 && t.size(0) == N && t.is_contiguous());
  };
  auto known = [&](const Tensor& t) { return !t.defined() || dtype_code(t) >= 0; };
  if (kn.sizes() != q.sizes() || vn.sizes() != q.sizes() || vc.sizes() != kc.sizes() || kc.size(0) != N ||
      kc.size(1) != H || kc.size(3) != D || !counter(pos_in) || !counter(pos_out) ||
      (tau.defined() && tau.sizes() != at::IntArrayRef({N, H, W})))
    return std::nullopt;
  for (const Tensor& t : {q, kn, vn, kc, vc, pos_in, pos_out, tau})
    if (!same(t)) return std::nullopt;
  for (const Tensor& t : {q, kn, vn, kc, vc, tau})
    if (!known(t)) return std::nullopt;
  const c10::DeviceGuard guard(q.device());
  Tensor out = at::empty_like(q);
  const Tensor qr = rows(q), knr = rows(kn), vnr = rows(vn);
  // the caller's own tensors, appended to and written in place; taken ahead of
  // the operands that are read, which may be views of the same storage
  const Buf bkc = written(kc), bvc = written(vc), bt = written(tau), bo = written(out);
  int32_t* const pout = pos_out.defined() ? pos_out.mutable_data_ptr<int32_t>() : nullptr;
  const Buf bq(qr), bkn(knr), bvn(vnr);
  check(tension_decode_step(bq.get(), bkn.get(), bvn.get(), bkc.get(), bvc.get(), bo.get(), bt.get(),
                            pos_in.const_data_ptr<int32_t>(), pout, N, H, D, W, scale, (int32_t)flags, stream_of(q)),
        "tension_decode_step");
  return out;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  using release = py::call_guard<py::gil_scoped_release>;
  g_tension_error = py::object(py::module_::import("bozo_amd._lib").attr("TensionError")).release().ptr();
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const TensionFail& e) {
      PyErr_SetString(g_tension_error, e.what());
    }
  });
  m.def("saved_rows_flow", &saved_rows_flow);
  m.def("window_fwd", [](const Tensor& Q, const Tensor& K, const Tensor& V, const OptTensor& bias, int64_t W, double scale,
                         int64_t flags, bool want_tau, bool want_mass) {
    auto [out, tau, mass] = window_fwd(Q, K, V, opt(bias), W, scale, flags, want_tau, want_mass);
    return std::make_tuple(out, want_tau ? OptTensor(tau) : std::nullopt, want_mass ? OptTensor(mass) : std::nullopt);
  }, release());
  m.def("window_bwd", [](const Tensor& Q, const Tensor& K, const Tensor& V, const OptTensor& dOut, const OptTensor& dTau,
                         const OptTensor& bias, const OptTensor& out, const OptTensor& mass, int64_t W, double scale,
                         int64_t flags) {
    return window_bwd(Q, K, V, opt(dOut), opt(dTau), opt(bias), opt(out), opt(mass), W, scale, flags);
  }, release());
  m.def("window", [](const Tensor& Q, const Tensor& K, const Tensor& V, const OptTensor& bias, int64_t W, double scale,
                     int64_t flags, bool return_tau) {
    return WindowFn::apply(rows(Q), rows(K), rows(V), bias, W, scale, flags, return_tau);
  }, release());
  m.def("global_fwd", [](const Tensor& Q, const Tensor& K, const Tensor& V, const OptTensor& bias, double scale, int64_t Wl) {
    auto [out, tl, mass] = global_fwd(Q, K, V, opt(bias), scale, Wl);
    return std::make_tuple(out, Wl > 0 ? OptTensor(tl) : std::nullopt, mass);
  }, release());
  m.def("global_bwd", [](const Tensor& Q, const Tensor& K, const Tensor& V, const OptTensor& dOut, const OptTensor& dTl,
                         const OptTensor& bias, const Tensor& out, const Tensor& mass, int64_t Wl, double scale) {
    return global_bwd(Q, K, V, opt(dOut), opt(dTl), opt(bias), out, mass, Wl, scale);
  }, release());
  m.def("global_", [](const Tensor& Q, const Tensor& K, const Tensor& V, const OptTensor& bias, double scale, int64_t Wl) {
    return GlobalFn::apply(rows(Q), rows(K), rows(V), bias, scale, Wl);
  }, release());
  m.def("rope_call", [](const Tensor& x, const Tensor& cos, const Tensor& sin, int64_t pos_offset, py::object dtype,
                        int64_t inverse) {
    const at::ScalarType dt = torch::python::detail::py_object_to_dtype(dtype);
    py::gil_scoped_release r;
    return rope_call(x, cos, sin, pos_offset, dt, inverse);
  });
  m.def("rope", [](const Tensor& x, const Tensor& cos, const Tensor& sin, int64_t pos_offset, py::object dtype) {
    const int64_t dt = dtype.is_none() ? (int64_t)x.scalar_type()
                                       : (int64_t)torch::python::detail::py_object_to_dtype(dtype);
    py::gil_scoped_release r;
    return RopeFn::apply(rows(x), cos.contiguous(), sin.contiguous(), pos_offset, dt);
  });
  m.def("decode_step", &decode_step, release());
}
