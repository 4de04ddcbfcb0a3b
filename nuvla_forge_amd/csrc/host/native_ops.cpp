// The host side of the fused ops in C++: argument checks, output and workspace
// allocation, kernel launches and the autograd node of one call, without the
// Python frames of the general path (kernels/*.py).  At the sizes of a small
// model the ops are bound by that host work: the adaLN seam at B 8 T 6 N 384,
// forward + backward, takes ~75 us of it in Python (seven allocations on
// autograd's thread, two ctypes calls, the Function's own machinery) and the
// kernels 17.
//
// Each entry takes the plain call only -- strided device tensors of one
// device, the shapes and types the kernels take, no tracing, no dispatch or
// function mode, no functorch transform, no forward-mode tangent -- and
// answers None to any other, which then runs the general path: it raises
// what it always raised, and stays visible to the tracer or mode.  Saved
// tensors go through save_for_backward, so saved-tensor hooks see them and
// autograd frees them after the backward.  Nothing is kept between calls.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/torch.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include "nuvla_forge_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr int64_t kMaxRow = 16384;  // widest adaLN row the kernels take

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return NF_DTYPE_F32;
    case at::kBFloat16: return NF_DTYPE_BF16;
    case at::kHalf: return NF_DTYPE_F16;
    default: return -1;
  }
}
int code_of(const Tensor &t) { return code_of(t.scalar_type()); }

void check(int rc, const char *what) {
  TORCH_CHECK(rc == 0, what, " failed (status ", rc, "): ", nf_last_error());
}

void *stream_of(const Tensor &t) {
  return static_cast<void *>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor bytes(size_t n, const Tensor &like) {
  return at::empty({(int64_t)(n > 0 ? n : 1)}, like.options().dtype(at::kByte));
}

// Nothing that could see or replace the ops of the general path is active.
bool quiet() {
  return !torch::jit::tracer::isTracing() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !at::impl::torch_function_mode_enabled() &&
         !c10::impl::tls_is_dispatch_key_included(
             c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// A strided device tensor with memory of its own kind.
bool plain(const Tensor &t, c10::Device dev) {
  if (!t.defined() || !dev.is_cuda() || t.device() != dev || t.layout() != at::kStrided) return false;
  const c10::DispatchKeySet ks = t.key_set();
  for (c10::DispatchKey k :
       {c10::DispatchKey::Python, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
        c10::DispatchKey::ZeroTensor, c10::DispatchKey::Functionalize,
        c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
        c10::DispatchKey::NestedTensor})
    if (ks.has(k)) return false;
  return !t._fw_grad(0).defined();
}

// ---------------------------------------------------------------------------
// adaLN seam
// ---------------------------------------------------------------------------
struct Seam : torch::autograd::Function<Seam> {
  static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &y,
                               const Tensor &gate, const Tensor &weight, const Tensor &scale,
                               const Tensor &shift, int64_t t, double eps) {
    const c10::DeviceGuard guard(x.device());
    const int64_t m = x.size(0), n = x.size(1);
    Tensor h = at::empty({m, n}, x.options()), out = at::empty({m, n}, x.options());
    Tensor rstd = at::empty({m}, x.options().dtype(at::kFloat));
    check(nf_adaln_fwd(x.data_ptr(), x.stride(0), y.data_ptr(), y.stride(0), gate.data_ptr(),
                       gate.stride(0), weight.data_ptr(), scale.data_ptr(), scale.stride(0),
                       shift.data_ptr(), shift.stride(0), h.data_ptr(), out.data_ptr(),
                       rstd.data_ptr<float>(), m, n, t, (float)eps, code_of(x), code_of(y),
                       code_of(gate), code_of(weight), code_of(scale), code_of(shift),
                       stream_of(x)),
          "nf_adaln_fwd");
    ctx->save_for_backward({x, y, gate, weight, scale, rstd});
    ctx->saved_data["t"] = t;
    ctx->saved_data["shift"] = (int64_t)shift.scalar_type();
    ctx->set_materialize_grads(false);
    return {h, out};
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list res(8);
    if (!grads[0].defined() && !grads[1].defined()) return res;
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &y = s[1], &gate = s[2], &weight = s[3], &scale = s[4], &rstd = s[5];
    const c10::DeviceGuard guard(x.device());
    const int64_t m = x.size(0), n = x.size(1), t = ctx->saved_data["t"].toInt(), b = m / t;
    const auto dt_shift = (at::ScalarType)ctx->saved_data["shift"].toInt();
    Tensor dh, dout;
    if (grads[0].defined()) dh = grads[0].to(x.scalar_type()).contiguous();
    if (grads[1].defined()) dout = grads[1].to(x.scalar_type()).contiguous();
    for (const Tensor *g : {&dh, &dout})
      TORCH_CHECK_VALUE(!g->defined() || g->device() == x.device(),
                        "fused_adaln_residual_rmsnorm backward: an upstream gradient is not on "
                        "the forward's device");
    Tensor dx = at::empty({m, n}, x.options()), dy = at::empty({m, n}, y.options());
    Tensor dgate, dweight, dscale, dshift;
    if (ctx->needs_input_grad(2)) dgate = at::empty({b, n}, gate.options());
    if (ctx->needs_input_grad(3)) dweight = at::empty({n}, weight.options());
    if (ctx->needs_input_grad(4)) dscale = at::empty({b, n}, scale.options());
    if (ctx->needs_input_grad(5)) dshift = at::empty({b, n}, scale.options().dtype(dt_shift));
    const size_t nbytes = nf_adaln_bwd_workspace(m, n, t);
    Tensor ws = bytes(nbytes, x);
    check(nf_adaln_bwd_full(ptr(dh), ptr(dout), x.data_ptr(), x.stride(0), y.data_ptr(),
                            y.stride(0), gate.data_ptr(), gate.stride(0), weight.data_ptr(),
                            scale.data_ptr(), scale.stride(0), rstd.data_ptr<float>(),
                            dx.data_ptr(), dy.data_ptr(), ptr(dgate), ptr(dweight), ptr(dscale),
                            ptr(dshift), ws.data_ptr(), nbytes, m, n, t, code_of(x), code_of(y),
                            code_of(gate), code_of(weight), code_of(scale), code_of(dt_shift),
                            stream_of(x)),
          "nf_adaln_bwd_full");
    if (ctx->needs_input_grad(0)) res[0] = dx;
    if (ctx->needs_input_grad(1)) res[1] = dy;
    res[2] = dgate;
    res[3] = dweight;
    res[4] = dscale;
    res[5] = dshift;
    return res;
  }
};

// (x, y) element types the row kernels take: equal, or fp32 x with 16-bit y
bool seam_types(const Tensor &x, const Tensor &y) {
  const int cx = code_of(x), cy = code_of(y);
  return cx >= 0 && cy >= 0 && (cx == cy || cx == NF_DTYPE_F32);
}

bool seam_plain(const Tensor &x, const Tensor &y, const Tensor &gate, const Tensor &weight,
                const Tensor &scale, const Tensor &shift, int64_t t) {
  const c10::Device dev = x.device();
  for (const Tensor *v : {&x, &y, &gate, &weight, &scale, &shift})
    if (!plain(*v, dev) || code_of(*v) < 0) return false;
  if (x.dim() != 2 || y.dim() != 2 || x.size(0) == 0 || x.size(1) == 0 ||
      x.size(1) > kMaxRow || y.sizes() != x.sizes() || !seam_types(x, y))
    return false;
  const int64_t m = x.size(0), n = x.size(1);
  if (t <= 0 || m % t != 0 || x.stride(1) != 1 || y.stride(1) != 1) return false;
  for (const Tensor *v : {&gate, &scale, &shift})
    if (v->dim() != 2 || v->size(0) != m / t || v->size(1) != n || v->stride(1) != 1)
      return false;
  return weight.dim() == 1 && weight.size(0) == n && weight.is_contiguous();
}

// ---------------------------------------------------------------------------
// SwiGLU
// ---------------------------------------------------------------------------
struct SwiGLU : torch::autograd::Function<SwiGLU> {
  static Tensor forward(AutogradContext *ctx, const Tensor &a_in, const Tensor &b_in) {
    const c10::DeviceGuard guard(a_in.device());
    const Tensor a = a_in.contiguous(), b = b_in.contiguous();
    Tensor out = at::empty(a.sizes(), a.options());
    check(nf_swiglu_fwd(a.data_ptr(), b.data_ptr(), out.data_ptr(), a.numel(), code_of(a),
                        stream_of(a)),
          "nf_swiglu_fwd");
    ctx->save_for_backward({a, b});
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &a = s[0], &b = s[1];
    const c10::DeviceGuard guard(a.device());
    const Tensor g = grads[0].contiguous().to(a.scalar_type());
    TORCH_CHECK_VALUE(g.device() == a.device(),
                      "fused_swiglu backward: dout is not on the forward's device");
    Tensor da = at::empty(a.sizes(), a.options()), db = at::empty(b.sizes(), b.options());
    check(nf_swiglu_bwd(g.data_ptr(), a.data_ptr(), b.data_ptr(), da.data_ptr(), db.data_ptr(),
                        a.numel(), code_of(a), stream_of(a)),
          "nf_swiglu_bwd");
    return {da, db};
  }
};

// ---------------------------------------------------------------------------
// gate/up projection with the SwiGLU in its epilogue
// ---------------------------------------------------------------------------
// bf16 with unit-stride rows
Tensor rows_bf16(const Tensor &t) {
  const Tensor r = t.to(at::kBFloat16);
  return r.stride(-1) == 1 ? r : r.contiguous();
}

// `t` with rows of whole 16-byte vectors (its width is a multiple of 8): a copy of a
// view whose base or row stride is not.  Every tile of the backward would read it
// element by element: x[:, 1:385] of M 9408 D 384 H 1536, forward + backward,
// 485 us, 231 with the copy.
Tensor vector_rows(const Tensor &t) {
  const bool whole = reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && t.stride(0) % 8 == 0;
  return whole ? t : t.clone(at::MemoryFormat::Contiguous);
}

// act = silu(x wg^T) * (x wu^T); a and b (the two products) are written where
// `save`, for the backward.
Tensor gate_up_forward(const Tensor &x, const Tensor &wg, const Tensor &wu, bool save, Tensor &a,
                       Tensor &b) {
  const int64_t m = x.size(0), d = x.size(1), h = wg.size(0);
  if (save) a = at::empty({m, h}, x.options());
  if (save) b = at::empty({m, h}, x.options());
  Tensor act = at::empty({m, h}, x.options());
  check(nf_gemm_swiglu(x.data_ptr(), x.stride(0), wg.data_ptr(), wg.stride(0), wu.data_ptr(),
                       wu.stride(0), ptr(a), ptr(b), act.data_ptr(), h, m, d, h, NF_DTYPE_BF16,
                       stream_of(x)),
        "nf_gemm_swiglu");
  return act;
}

struct GateUp : torch::autograd::Function<GateUp> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x_in, const Tensor &g_in,
                        const Tensor &u_in) {
    const c10::DeviceGuard guard(x_in.device());
    const Tensor x = rows_bf16(x_in), wg = rows_bf16(g_in), wu = rows_bf16(u_in);
    Tensor a, b;
    const Tensor act = gate_up_forward(x, wg, wu, true, a, b);
    ctx->save_for_backward({x, wg, wu, a, b});
    ctx->saved_data["dt"] = std::vector<int64_t>{(int64_t)x_in.scalar_type(),
                                                 (int64_t)g_in.scalar_type(),
                                                 (int64_t)u_in.scalar_type()};
    return act;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    Tensor x = s[0], wg = s[1], wu = s[2];
    const Tensor &a = s[3], &b = s[4];
    const c10::DeviceGuard guard(x.device());
    const at::NoGradGuard no_grad;
    const auto dt = ctx->saved_data["dt"].toIntVector();
    const Tensor dact = grads[0].to(at::kBFloat16).contiguous();
    TORCH_CHECK_VALUE(dact.device() == x.device(),
                      "fused_gate_up_swiglu backward: dact is not on the forward's device");
    const int64_t m = x.size(0), d = x.size(1), h = a.size(1);
    Tensor da = at::empty({m, h}, a.options()), db = at::empty({m, h}, a.options());
    void *const st = stream_of(x);
    check(nf_swiglu_bwd(dact.data_ptr(), a.data_ptr(), b.data_ptr(), da.data_ptr(),
                        db.data_ptr(), a.numel(), NF_DTYPE_BF16, st),
          "nf_swiglu_bwd");
    // both weight gradients leave the kernel in one type: theirs, or fp32 where
    // two are wanted and differ (neither may round the other's gradient)
    const auto tx = (at::ScalarType)dt[0], tg = (at::ScalarType)dt[1], tu = (at::ScalarType)dt[2];
    const bool need_g = ctx->needs_input_grad(1), need_u = ctx->needs_input_grad(2);
    const auto tw = need_g && need_u && tg != tu ? at::kFloat : need_g ? tg : tu;
    Tensor dx, dg, du;
    bool one_x = ctx->needs_input_grad(0), one_w = need_g || need_u;  // left to the one launch
    if (need_g) dg = at::empty({h, d}, x.options().dtype(tw));
    if (need_u) du = at::empty({h, d}, x.options().dtype(tw));
    if (tx == at::kBFloat16 && tg == tx && tu == tx &&
        !nf_gemm_swiglu_bwd_wins(m, d, h, one_w)) {
      if (one_x) {
        const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        dx = at::addmm(at::mm(da, wg), db, wu);
        one_x = false;
      }
      if (need_g && need_u) {
        const size_t nb = nf_gemm_swiglu_wgrad_workspace(m, d, h);
        Tensor ws = bytes(nb, x);
        check(nf_gemm_swiglu_wgrad(da.data_ptr(), db.data_ptr(), h, x.data_ptr(), x.stride(0),
                                   dg.data_ptr(), du.data_ptr(), d, m, d, h, NF_DTYPE_BF16,
                                   ws.data_ptr(), nb, st),
              "nf_gemm_swiglu_wgrad");
        one_w = false;
      }
    }
    if (one_x) dx = at::empty({m, d}, x.options().dtype(tx));
    if (one_x || one_w) {
      if (d % 8 == 0 && h % 8 == 0) {  // other widths are copied to padded rows in the call
        x = vector_rows(x);
        wg = vector_rows(wg);
        wu = vector_rows(wu);
      }
      void *const pg = one_w ? ptr(dg) : nullptr, *const pu = one_w ? ptr(du) : nullptr;
      const size_t nb = nf_gemm_swiglu_bwd_workspace(m, d, h, one_x, pg != nullptr, pu != nullptr);
      Tensor ws = bytes(nb, x);
      check(nf_gemm_swiglu_bwd(da.data_ptr(), db.data_ptr(), h, x.data_ptr(), x.stride(0),
                               wg.data_ptr(), wg.stride(0), wu.data_ptr(), wu.stride(0),
                               one_x ? dx.data_ptr() : nullptr, code_of(tx), pg, pu, code_of(tw),
                               m, d, h, NF_DTYPE_BF16, ws.data_ptr(), nb, st),
            "nf_gemm_swiglu_bwd");
    }
    return {dx, need_g ? dg.to(tg) : dg, need_u ? du.to(tu) : du};
  }
};

// ---------------------------------------------------------------------------
// chunked cross entropy
// ---------------------------------------------------------------------------
struct ChunkedCE : torch::autograd::Function<ChunkedCE> {
  static Tensor forward(AutogradContext *ctx, const Tensor &hidden, const Tensor &weight,
                        const Tensor &targets, int64_t chunk_rows, int64_t ignore_index,
                        int64_t compute) {
    const c10::DeviceGuard guard(hidden.device());
    const auto cdt = (at::ScalarType)compute;
    const int64_t m = hidden.size(0), d = hidden.size(1), v = weight.size(0);
    const int code = code_of(cdt);
    const Tensor h = hidden.to(cdt).contiguous(), w = weight.to(cdt).contiguous();
    const Tensor tg = targets.to(at::kLong).contiguous();
    Tensor loss = at::empty({}, hidden.options().dtype(at::kFloat));
    const size_t ns = nf_ce_state_bytes(m, d, v, chunk_rows, code);
    const size_t nw = nf_ce_fwd_workspace(m, d, v, chunk_rows, code);
    TORCH_CHECK_VALUE(ns && nw, "chunked_cross_entropy: shape M=", m, " D=", d, " V=", v,
                      " is beyond the kernels");
    Tensor state = bytes(ns, hidden), ws = bytes(nw, hidden);
    check(nf_ce_fwd(h.data_ptr(), w.data_ptr(), tg.data_ptr<int64_t>(), m, d, v, ignore_index,
                    chunk_rows, code, loss.data_ptr<float>(), nullptr, state.data_ptr(), ns,
                    ws.data_ptr(), nw, stream_of(hidden)),
          "nf_ce_fwd");
    ctx->save_for_backward({state});
    ctx->saved_data["s"] = std::vector<int64_t>{m, d, v, chunk_rows, code,
                                                (int64_t)hidden.scalar_type(),
                                                (int64_t)weight.scalar_type()};
    return loss;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &state = saved[0];
    const c10::DeviceGuard guard(state.device());
    const auto s = ctx->saved_data["s"].toIntVector();
    const int64_t m = s[0], d = s[1], v = s[2], chunk_rows = s[3];
    const int code = (int)s[4];
    const auto th = (at::ScalarType)s[5], tw = (at::ScalarType)s[6];
    const Tensor g = grads[0].to(at::kFloat).contiguous();
    TORCH_CHECK_VALUE(g.device() == state.device(),
                      "chunked_cross_entropy backward: grad_output is not on the forward's device");
    Tensor dh = at::empty({m, d}, state.options().dtype(th));
    Tensor dw = at::empty({v, d}, state.options().dtype(tw));
    const size_t nw = nf_ce_bwd_workspace(m, d, v, chunk_rows, code);
    Tensor ws = bytes(nw, state);
    check(nf_ce_bwd(m, d, v, chunk_rows, code, state.data_ptr(), (size_t)state.numel(),
                    g.data_ptr<float>(), dh.data_ptr(), code_of(th), dw.data_ptr(), code_of(tw),
                    ws.data_ptr(), nw, stream_of(state)),
          "nf_ce_bwd");
    return {dh, dw, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------------------
// entries
// ---------------------------------------------------------------------------
// The call's leading `n` arguments as tensors; false when one is not.
template <int N>
bool tensors(PyObject *const *args, Py_ssize_t nargs, Py_ssize_t want, Tensor (&t)[N]) {
  if (nargs != want) return false;
  for (int i = 0; i < N; ++i) {
    if (!THPVariable_CheckExact(args[i])) return false;  // a subclass may have its own rules
    t[i] = THPVariable_Unpack(args[i]);
  }
  return true;
}

// The call without the interpreter lock, which other threads take meanwhile (an
// allocation or a launch may wait); what calls into Python, such as a
// saved-tensor hook, takes it for itself.
template <class F>
auto unlocked(F &&f) {
  const pybind11::gil_scoped_release no_gil;
  return f();
}

PyObject *py_seam(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Tensor a[6];
  if (!tensors(args, nargs, 8, a) || !quiet()) Py_RETURN_NONE;
  const int64_t t = PyLong_Check(args[6]) ? PyLong_AsLongLong(args[6]) : 0;
  const double eps = PyFloat_AsDouble(args[7]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (!seam_plain(a[0], a[1], a[2], a[3], a[4], a[5], t)) Py_RETURN_NONE;
  const variable_list r =
      unlocked([&] { return Seam::apply(a[0], a[1], a[2], a[3], a[4], a[5], t, eps); });
  PyObject *h = THPVariable_Wrap(r[0]), *out = THPVariable_Wrap(r[1]);
  PyObject *pair = PyTuple_Pack(2, h, out);
  Py_XDECREF(h);
  Py_XDECREF(out);
  return pair;
  END_HANDLE_TH_ERRORS
}

PyObject *py_swiglu(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Tensor t[2];
  if (!tensors(args, nargs, 2, t) || !quiet()) Py_RETURN_NONE;
  const c10::Device dev = t[0].device();
  if (!plain(t[0], dev) || !plain(t[1], dev) || t[0].sizes() != t[1].sizes() ||
      t[0].scalar_type() != t[1].scalar_type() || code_of(t[0]) < 0 || t[0].numel() == 0)
    Py_RETURN_NONE;
  return THPVariable_Wrap(unlocked([&] { return SwiGLU::apply(t[0], t[1]); }));
  END_HANDLE_TH_ERRORS
}

// x [M, D], w_gate, w_up [H, D]
PyObject *py_gate_up(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Tensor t[3];
  if (!tensors(args, nargs, 3, t) || !quiet()) Py_RETURN_NONE;
  const c10::Device dev = t[0].device();
  for (const Tensor &v : t)
    if (!plain(v, dev) || code_of(v) < 0 || v.dim() != 2 || v.numel() == 0) Py_RETURN_NONE;
  if (t[1].sizes() != t[2].sizes() || t[0].size(1) != t[1].size(1)) Py_RETURN_NONE;
  if (!at::GradMode::is_enabled() ||
      !(t[0].requires_grad() || t[1].requires_grad() || t[2].requires_grad())) {
    // no backward: two of the three [M, H] outputs are not written
    return THPVariable_Wrap(unlocked([&] {
      const c10::DeviceGuard guard(dev);
      const at::NoGradGuard no_grad;
      Tensor a, b;
      return gate_up_forward(rows_bf16(t[0]), rows_bf16(t[1]), rows_bf16(t[2]), false, a, b);
    }));
  }
  return THPVariable_Wrap(unlocked([&] { return GateUp::apply(t[0], t[1], t[2]); }));
  END_HANDLE_TH_ERRORS
}

// hidden [M, D], lm_weight [V, D], targets [M], chunk rows, ignore index,
// compute type (0 fp32, 1 bf16)
PyObject *py_ce(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Tensor t[3];
  if (!tensors(args, nargs, 6, t) || !quiet()) Py_RETURN_NONE;
  int64_t v[3];
  for (int i = 0; i < 3; ++i) {
    if (!PyLong_Check(args[3 + i])) Py_RETURN_NONE;  // the general path converts it
    v[i] = PyLong_AsLongLong(args[3 + i]);
  }
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const c10::Device dev = t[0].device();
  for (const Tensor &x : t)
    if (!plain(x, dev)) Py_RETURN_NONE;
  if (t[0].dim() != 2 || t[1].dim() != 2 || t[0].size(1) != t[1].size(1) || t[0].numel() == 0 ||
      t[1].numel() == 0 || t[2].dim() != 1 || t[2].size(0) != t[0].size(0) ||
      code_of(t[0]) < 0 || code_of(t[1]) < 0 || t[2].scalar_type() != at::kLong || v[0] <= 0)
    Py_RETURN_NONE;
  const at::ScalarType cdt = v[2] == NF_DTYPE_BF16 ? at::kBFloat16 : at::kFloat;
  return THPVariable_Wrap(unlocked(
      [&] { return ChunkedCE::apply(t[0], t[1], t[2], v[0], v[1], (int64_t)cdt); }));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"seam", (PyCFunction)(void (*)(void))py_seam, METH_FASTCALL, nullptr},
    {"swiglu", (PyCFunction)(void (*)(void))py_swiglu, METH_FASTCALL, nullptr},
    {"gate_up", (PyCFunction)(void (*)(void))py_gate_up, METH_FASTCALL, nullptr},
    {"ce", (PyCFunction)(void (*)(void))py_ce, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&kModule); }
