// The eager entry points' host side: argument checks, output and workspace allocation, the C-ABI
// calls and the autograd nodes, in C++.  At the sizes of a decode step or a small training step the
// host is what an eager call waits for (a training step at B = 2, S = 128, D = 512 took 270 us of
// which the GPU worked 44): a ctypes call marshals 20-30 arguments, a Python autograd node costs
// 5 us forward and takes the GIL in the engine's thread backward.
//
// The nodes are the ones of mhc/_layer.py, mhc/ops.py and mhc/streams.py (their docstrings hold the
// reasoning): the same inputs, outputs and saved tensors in the same roles.  Every function returns
// None when a call is not the plain case -- a tensor subclass, a CPU tensor, mixed devices, an
// unsupported dtype or shape, a functorch transform, a torch-function or torch-dispatch mode,
// tracing, forward-mode tangents -- and the Python caller then takes those Python nodes, which
// handle or refuse it.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/mhc_abi.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

// ---------------------------------------------------------------------------
// Helpers
// ---------------------------------------------------------------------------

PyObject* g_error = nullptr;  // mhc._lib.MHCError

// Raises MHCError; also from the autograd engine's threads, which hold no GIL.
void check(int rc, const char* name) {
  if (rc == 0) return;
  const std::string msg =
      std::string("mhc: ") + name + " failed (status " + std::to_string(rc) + "): " + mhc_last_error();
  const PyGILState_STATE gil = PyGILState_Ensure();
  PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, msg.c_str());
  python_error e;
  e.persist();
  PyGILState_Release(gil);
  throw e;
}

int code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return MHC_DTYPE_F32;
    case at::kBFloat16: return MHC_DTYPE_BF16;
    case at::kHalf: return MHC_DTYPE_F16;
    default: return -1;
  }
}

void* stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const float* fptr(const Tensor& t) { return t.defined() ? static_cast<const float*>(t.data_ptr()) : nullptr; }
float* wptr(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }

Tensor f32(const Tensor& t) {
  if (!t.defined()) return t;
  return (t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)).contiguous();
}

Tensor in_dtype(const Tensor& t, at::ScalarType dt) {
  if (!t.defined()) return t;
  return t.contiguous().to(dt);
}

Tensor grad_like(const Tensor& g, const Tensor& p) {
  Tensor r = g.sizes() == p.sizes() ? g : g.reshape(p.sizes());
  return r.scalar_type() == p.scalar_type() ? r : r.to(p.scalar_type());
}

Tensor empty_f32(at::IntArrayRef sizes, const Tensor& like) {
  return at::empty(sizes, like.options().dtype(at::kFloat).requires_grad(false));
}

// What a node saved.  An unpack hook may hand back other strides, another dtype or another device: the
// backwards take each tensor through contiguous() or f32(), and a tensor that is not on the first
// one's GPU is refused here, as the Python nodes refuse it (_lib.require_gpu).
variable_list saved(AutogradContext* ctx) {
  variable_list s = ctx->get_saved_variables();
  for (const Tensor& t : s) {
    if (!t.defined()) continue;
    TORCH_CHECK(t.is_cuda(), "mhc: the HIP kernels need tensors on a ROCm GPU, got device '", t.device(),
                "' from a saved-tensor hook");
    TORCH_CHECK(t.device() == s[0].device(), "mhc: tensors on different devices (", s[0].device(), " and ", t.device(),
                ")");
  }
  return s;
}

// The f32 values of N <= 8 parameters: the parameters' own memory, or, where any is stored in another
// dtype, one buffer of them all, converted in one launch.  The forward keeps the buffer for the
// backward, which then reads nothing from the parameters.
template <int N>
struct Params {
  const float* p[N];
  Tensor buf;

  Params(const Tensor* t, const Tensor& have) : buf(f32(have)) {
    int64_t at[N], total = 0;
    bool own = !buf.defined();
    for (int i = 0; i < N; ++i) {
      at[i] = total;
      total += (t[i].numel() + 3) / 4 * 4;  // 16-byte aligned parts
      own = own && t[i].scalar_type() == at::kFloat && t[i].is_contiguous();
    }
    if (own) {
      for (int i = 0; i < N; ++i) p[i] = fptr(t[i]);
      return;
    }
    if (!buf.defined()) {
      buf = empty_f32({total}, t[0]);
      const void* src[N];
      void* dst[N];
      int sd[N], dd[N];
      int64_t count[N];
      Tensor hold[N];
      for (int i = 0; i < N; ++i) {
        hold[i] = (code(t[i]) < 0 ? t[i].to(at::kFloat) : t[i]).contiguous();
        src[i] = ptr(hold[i]);
        sd[i] = code(hold[i]);
        dst[i] = wptr(buf) + at[i];
        dd[i] = MHC_DTYPE_F32;
        count[i] = hold[i].numel();
      }
      check(mhc_convert(N, src, sd, dst, dd, count, stream(buf)), "convert");
    }
    for (int i = 0; i < N; ++i) p[i] = fptr(buf) + at[i];
  }
};

// The gradients of N parameters from f32 parts, each in its parameter's shape and dtype; those that
// are not f32 are converted in one launch.
template <int N>
void param_grads(const Tensor* prm, const Tensor* part, variable_list& out) {
  const void* src[N];
  void* dst[N];
  int sd[N], dd[N], n = 0;
  int64_t count[N];
  for (int i = 0; i < N; ++i) {
    const Tensor& p = prm[i];
    // a parameter of another size than the kernels' gradient: the reshape refuses it
    if (p.scalar_type() == at::kFloat || code(p) < 0 || p.numel() != part[i].numel()) {
      out.push_back(grad_like(part[i], p));
      continue;
    }
    Tensor g = at::empty(p.sizes(), p.options().requires_grad(false));
    src[n] = ptr(part[i]);
    sd[n] = MHC_DTYPE_F32;
    dst[n] = ptr(g);
    dd[n] = code(p);
    count[n++] = p.numel();
    out.push_back(std::move(g));
  }
  if (n) check(mhc_convert(n, src, sd, dst, dd, count, stream(part[0])), "convert");
}

struct Workspace {
  Tensor t;
  size_t bytes;
  Workspace(size_t n, const Tensor& like) : bytes(n) {
    if (n) t = at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false));
  }
  void* p() const { return ptr(t); }
};

// True when this thread runs plain eager calls: nothing that wants to see or rewrite them.
bool plain_thread() {
  using c10::DispatchKey;
  return !c10::impl::tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::tls_is_dispatch_key_included(DispatchKey::Tracer) && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

bool plain(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() &&
         !t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::Python) && !t._fw_grad(0).defined();
}

// args[0..n) as plain tensors on one GPU.
bool tensors(PyObject* const* args, int n, Tensor* out) {
  for (int i = 0; i < n; ++i) {
    if (!THPVariable_CheckExact(args[i])) return false;
    out[i] = THPVariable_Unpack(args[i]);
    if (!plain(out[i]) || out[i].device() != out[0].device()) return false;
  }
  return plain_thread();
}

bool number(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
  return *v >= 0 && *v <= INT32_MAX;
}

bool number(PyObject* o, double* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}

bool wants_grad(std::initializer_list<Tensor> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& t : ts)
    if (t.requires_grad()) return true;
  return false;
}

PyObject* none() { Py_RETURN_NONE; }

PyObject* tuple_of(const variable_list& ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  for (size_t i = 0; i < ts.size(); ++i) {
    PyObject* o = THPVariable_Wrap(ts[i]);
    if (!o) { Py_DECREF(r); return nullptr; }
    PyTuple_SET_ITEM(r, (Py_ssize_t)i, o);
  }
  return r;
}

struct ReleaseGil {
  PyThreadState* s = PyEval_SaveThread();
  ~ReleaseGil() { PyEval_RestoreThread(s); }
};

// ---------------------------------------------------------------------------
// HyperConnection: node A (dynamic fused, static) and the closure
// ---------------------------------------------------------------------------

struct Dims {
  int64_t B, S, D;
  explicit Dims(const Tensor& H) : B(H.size(0)), S(H.size(1)), D(H.size(3)) {}
};

// phi, H_pre_base, H_post_base, H_res_base, alpha_pre, alpha_post, alpha_res
constexpr int kDyn = 7;

struct DynOut { Tensor bi, x, w, aux, params; };

DynOut dynamic_forward(const Tensor& H, const Tensor* prm, int64_t iters, double eps, bool keep_x) {
  const c10::DeviceGuard guard(H.device());
  const Dims d(H);
  const Params<kDyn> q(prm, Tensor());
  const float* const* p = q.p;
  DynOut o;
  o.params = q.buf;
  o.bi = at::empty({d.B, d.S, d.D}, H.options().requires_grad(false));
  if (keep_x) o.x = empty_f32({d.B, 4 * d.D}, H);
  o.w = empty_f32({d.B, 24}, H);
  o.aux = empty_f32({d.B, 25}, H);
  const Workspace ws(mhc_layer_workspace_bytes(d.B, d.S, d.D, code(H)), H);
  check(mhc_layer_dynamic_forward(ptr(H), code(H), p[0], p[1], p[2], p[3], p[4], p[5], p[6], ptr(o.bi), wptr(o.x),
                                  wptr(o.w), wptr(o.aux), d.B, d.S, d.D, (int)iters, (float)eps, ws.p(), ws.bytes,
                                  stream(H)),
        "layer_dynamic_forward");
  return o;
}

Tensor post_link(const Tensor& w) { return at::empty({w.size(0), 4}, w.options()); }

Tensor d_bi_or_zeros(const Tensor& d_bi, const Tensor& H, const Dims& d) {
  if (!d_bi.defined()) return at::zeros({d.B, d.S, d.D}, H.options().requires_grad(false));
  return in_dtype(d_bi, H.scalar_type());
}

struct DynamicLayer : Function<DynamicLayer> {
  static variable_list forward(AutogradContext* ctx, const Tensor& H, const Tensor& phi, const Tensor& pre,
                               const Tensor& post, const Tensor& res, const Tensor& a_pre, const Tensor& a_post,
                               const Tensor& a_res, int64_t iters, double eps) {
    const Tensor prm[kDyn] = {phi, pre, post, res, a_pre, a_post, a_res};
    // at S = 1 the pooled rows are H's rows, which the backward reads from H
    DynOut o = dynamic_forward(H, prm, iters, eps, H.size(1) != 1);
    ctx->save_for_backward({H, o.x, o.w, o.aux, phi, pre, post, res, a_pre, a_post, a_res, o.params});
    ctx->saved_data["iters"] = iters;
    ctx->saved_data["eps"] = eps;
    ctx->set_materialize_grads(false);
    return {o.bi, o.w, H.view_as(H), post_link(o.w)};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = saved(ctx);
    const c10::DeviceGuard guard(s[0].device());
    const Tensor H = s[0].contiguous();
    const Tensor* prm = &s[4];
    const Dims d(H);
    const Tensor d_bi = d_bi_or_zeros(g[0], H, d);
    const Tensor dHn = in_dtype(g[2], H.scalar_type());
    const Tensor dpost = f32(g[3]);
    const Params<kDyn> q(prm, s[4 + kDyn]);
    const float* const* p = q.p;
    const Tensor x = f32(s[1]), w = f32(s[2]), aux = f32(s[3]);
    Tensor dH;
    if (ctx->needs_input_grad(0)) dH = at::empty(H.sizes(), H.options().requires_grad(false));
    const Tensor gphi = empty_f32({4 * d.D, 24}, H);
    const Tensor small = empty_f32({27}, H);  // grad_bias [24], grad_alpha [3]
    const Workspace ws(mhc_layer_workspace_bytes(d.B, d.S, d.D, code(H)), H);
    check(mhc_layer_dynamic_backward(ptr(H), code(H), ptr(d_bi), ptr(dHn), fptr(dpost), p[0], p[1], p[2], p[3], p[4],
                                     p[5], p[6], fptr(x), fptr(w), fptr(aux), ptr(dH), wptr(gphi), wptr(small),
                                     wptr(small) + 24, d.B, d.S, d.D, (int)ctx->saved_data["iters"].toInt(),
                                     (float)ctx->saved_data["eps"].toDouble(), ws.p(), ws.bytes, stream(H)),
          "layer_dynamic_backward");
    const Tensor part[kDyn] = {gphi,
                               small.narrow(0, 0, 4),
                               small.narrow(0, 4, 4),
                               small.narrow(0, 8, 16),
                               small.narrow(0, 24, 1),
                               small.narrow(0, 25, 1),
                               small.narrow(0, 26, 1)};
    variable_list out{dH};
    param_grads<kDyn>(prm, part, out);
    out.resize(kDyn + 3);  // iters, eps
    return out;
  }
};

PyObject* py_dynamic_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[8];
  int64_t iters;
  double eps;
  if (n != 10 || !tensors(a, 8, t) || !number(a[8], &iters) || !number(a[9], &eps)) return none();
  const Tensor& H = t[0];
  if (code(H) < 0 || H.dim() != 4 || !H.is_contiguous()) return none();
  for (int i = 5; i < 8; ++i)
    if (t[i].numel() != 1) return none();
  variable_list out;
  {
    ReleaseGil gil;
    if (wants_grad({t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7]})) {
      out = DynamicLayer::apply(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], iters, eps);
    } else {
      // no gradient can reach this forward: nothing is kept for one
      DynOut o = dynamic_forward(H, t + 1, iters, eps, false);
      out = {o.bi, o.w, H.detach(), o.w};
    }
  }
  return tuple_of(out);
  END_HANDLE_TH_ERRORS
}

struct StaticOut { Tensor bi, w, params; };

StaticOut static_forward(const Tensor& H, const Tensor* prm, int64_t iters) {
  const c10::DeviceGuard guard(H.device());
  const Dims d(H);
  const Params<3> q(prm, Tensor());
  StaticOut o;
  o.params = q.buf;
  o.bi = at::empty({d.B, d.S, d.D}, H.options().requires_grad(false));
  o.w = empty_f32({d.B, 24}, H);
  check(mhc_layer_static_forward(ptr(H), code(H), q.p[0], q.p[1], q.p[2], ptr(o.bi), wptr(o.w), d.B, d.S,
                                 d.D, (int)iters, stream(H)),
        "layer_static_forward");
  return o;
}

struct StaticLayer : Function<StaticLayer> {
  static variable_list forward(AutogradContext* ctx, const Tensor& H, const Tensor& pre, const Tensor& post,
                               const Tensor& res, int64_t iters) {
    const Tensor prm[3] = {pre, post, res};
    StaticOut o = static_forward(H, prm, iters);
    ctx->save_for_backward({H, o.w, pre, post, res, o.params});
    ctx->saved_data["iters"] = iters;
    ctx->set_materialize_grads(false);
    return {o.bi, o.w, H.view_as(H), post_link(o.w)};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = saved(ctx);
    const c10::DeviceGuard guard(s[0].device());
    const Tensor H = s[0].contiguous();
    const Tensor* prm = &s[2];
    const Dims d(H);
    const Tensor d_bi = d_bi_or_zeros(g[0], H, d);
    const Tensor dHn = in_dtype(g[2], H.scalar_type());
    const Tensor dpost = f32(g[3]), w = f32(s[1]);
    const Params<3> q(prm, s[5]);
    Tensor dH;
    if (ctx->needs_input_grad(0)) dH = at::empty(H.sizes(), H.options().requires_grad(false));
    const Tensor gb = empty_f32({24}, H);
    const Workspace ws(mhc_layer_workspace_bytes(d.B, d.S, d.D, code(H)), H);
    check(mhc_layer_static_backward(ptr(H), code(H), ptr(d_bi), ptr(dHn), fptr(dpost), q.p[0], q.p[1], q.p[2], fptr(w),
                                    ptr(dH), wptr(gb), d.B, d.S, d.D, (int)ctx->saved_data["iters"].toInt(), ws.p(),
                                    ws.bytes, stream(H)),
          "layer_static_backward");
    const Tensor part[3] = {gb.narrow(0, 0, 4), gb.narrow(0, 4, 4), gb.narrow(0, 8, 16)};
    variable_list out{dH};
    param_grads<3>(prm, part, out);
    out.resize(5);  // iters
    return out;
  }
};

PyObject* py_static_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[4];
  int64_t iters;
  if (n != 5 || !tensors(a, 4, t) || !number(a[4], &iters)) return none();
  const Tensor& H = t[0];
  if (code(H) < 0 || H.dim() != 4 || !H.is_contiguous()) return none();
  variable_list out;
  {
    ReleaseGil gil;
    if (wants_grad({t[0], t[1], t[2], t[3]})) {
      out = StaticLayer::apply(t[0], t[1], t[2], t[3], iters);
    } else {
      StaticOut o = static_forward(H, t + 1, iters);
      out = {o.bi, o.w, H.detach(), o.w};
    }
  }
  return tuple_of(out);
  END_HANDLE_TH_ERRORS
}

Tensor add_forward(const Tensor& link, const Tensor& branch_output, const Tensor& w_in) {
  const c10::DeviceGuard guard(link.device());
  const Dims d(link);
  const Tensor H = link.contiguous(), bo = branch_output.contiguous(), w = f32(w_in);
  const Tensor out = at::empty(H.sizes(), H.options().requires_grad(false));
  check(mhc_layer_add_forward(ptr(H), code(H), ptr(bo), code(bo), fptr(w), ptr(out), d.B, d.S, d.D, stream(H)),
        "layer_add_forward");
  return out;
}

struct LayerAdd : Function<LayerAdd> {
  static Tensor forward(AutogradContext* ctx, const Tensor& link, const Tensor& branch_output, const Tensor& w,
                        const Tensor& /*post_link*/) {
    const Tensor out = add_forward(link, branch_output, w);
    ctx->save_for_backward({branch_output, w});
    ctx->saved_data["h_dtype"] = (int64_t)link.scalar_type();
    return out;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = saved(ctx);
    const c10::DeviceGuard guard(g[0].device());
    const Tensor dHn = in_dtype(g[0], (at::ScalarType)ctx->saved_data["h_dtype"].toInt());
    const Dims d(dHn);
    const Tensor bo = s[0].contiguous(), w = f32(s[1]);
    const Tensor dbo = at::empty_like(bo);
    const Tensor dpost = empty_f32({d.B, 4}, dHn);
    const Workspace ws(mhc_layer_workspace_bytes(d.B, d.S, d.D, code(dHn)), dHn);
    check(mhc_layer_add_backward(ptr(dHn), code(dHn), ptr(bo), code(bo), fptr(w), ptr(dbo), wptr(dpost), d.B, d.S, d.D,
                                 ws.p(), ws.bytes, stream(dHn)),
          "layer_add_backward");
    return {ctx->needs_input_grad(0) ? dHn : Tensor(), dbo, Tensor(), ctx->needs_input_grad(3) ? dpost : Tensor()};
  }
};

PyObject* py_layer_add(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[4];
  if (n != 4 || !tensors(a, 4, t)) return none();
  const Tensor &H = t[0], &bo = t[1];
  if (code(H) < 0 || code(bo) < 0 || bo.dim() != 3 || bo.size(0) != H.size(0) || bo.size(1) != H.size(1) ||
      bo.size(2) != H.size(3))
    return none();
  Tensor out;
  {
    ReleaseGil gil;
    out = wants_grad({t[0], t[1], t[2], t[3]}) ? LayerAdd::apply(t[0], t[1], t[2], t[3]) : add_forward(H, bo, t[2]);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------
// The low-level ops
// ---------------------------------------------------------------------------

Tensor sinkhorn_forward(const Tensor& M_in, int64_t iters, double eps) {
  const c10::DeviceGuard guard(M_in.device());
  const Tensor M = M_in.contiguous();
  const Tensor out = at::empty(M.sizes(), M.options().requires_grad(false));
  check(mhc_sinkhorn_forward(ptr(M), ptr(out), M.numel() / 16, code(M), (int)iters, (float)eps, stream(M)),
        "sinkhorn_forward");
  return out;
}

struct Sinkhorn : Function<Sinkhorn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& M, int64_t iters, double eps) {
    const Tensor out = sinkhorn_forward(M, iters, eps);
    ctx->save_for_backward({M});
    ctx->saved_data["iters"] = iters;
    ctx->saved_data["eps"] = eps;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const Tensor M = saved(ctx)[0].contiguous();
    const c10::DeviceGuard guard(M.device());
    const Tensor dP = g[0].contiguous();
    const Tensor dM = at::empty(M.sizes(), M.options().requires_grad(false));
    check(mhc_sinkhorn_backward(ptr(M), code(M), ptr(dP), code(dP), ptr(dM), M.numel() / 16,
                                (int)ctx->saved_data["iters"].toInt(), (float)ctx->saved_data["eps"].toDouble(),
                                stream(M)),
          "sinkhorn_backward");
    return {dM, Tensor(), Tensor()};
  }
};

PyObject* py_sinkhorn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[1];
  int64_t iters;
  double eps;
  if (n != 3 || !tensors(a, 1, t) || !number(a[1], &iters) || !number(a[2], &eps)) return none();
  const Tensor& M = t[0];
  if (code(M) < 0 || M.dim() < 2 || M.size(-1) != 4 || M.size(-2) != 4) return none();
  Tensor out;
  {
    ReleaseGil gil;
    out = wants_grad({M}) ? Sinkhorn::apply(M, iters, eps) : sinkhorn_forward(M, iters, eps);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

variable_list stream_mix_forward(const Tensor& H_in, const Tensor& pre_in, const Tensor& res_in) {
  const c10::DeviceGuard guard(H_in.device());
  const Dims d(H_in);
  const Tensor H = H_in.contiguous(), pre = f32(pre_in), res = f32(res_in);
  const Tensor bi = at::empty({d.B, d.S, d.D}, H.options().requires_grad(false));
  const Tensor hr = at::empty(H.sizes(), H.options().requires_grad(false));
  check(mhc_stream_mix_forward(ptr(H), fptr(pre), fptr(res), ptr(bi), ptr(hr), d.B, d.S, d.D, code(H), stream(H)),
        "stream_mix_forward");
  return {bi, hr};
}

struct StreamMix : Function<StreamMix> {
  static variable_list forward(AutogradContext* ctx, const Tensor& H, const Tensor& pre, const Tensor& res) {
    variable_list out = stream_mix_forward(H, pre, res);
    ctx->save_for_backward({H, pre, res});
    return out;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = saved(ctx);
    const c10::DeviceGuard guard(s[0].device());
    const Tensor H = s[0].contiguous();
    const Dims d(H);
    const Tensor dbi = in_dtype(g[0], H.scalar_type()), dhr = in_dtype(g[1], H.scalar_type());
    const Tensor pre = f32(s[1]), res = f32(s[2]);
    const Tensor dH = at::empty(H.sizes(), H.options().requires_grad(false));
    const Tensor dpre = empty_f32({d.B, 4}, H), dres = empty_f32({d.B, 4, 4}, H);
    const Workspace ws(mhc_stream_mix_backward_workspace_bytes(d.B, d.S, d.D, code(H)), H);
    check(mhc_stream_mix_backward(ptr(dbi), ptr(dhr), ptr(H), fptr(pre), fptr(res), ptr(dH), wptr(dpre), wptr(dres),
                                  d.B, d.S, d.D, code(H), ws.p(), ws.bytes, stream(H)),
          "stream_mix_backward");
    return {dH, dpre.to(s[1].scalar_type()), dres.to(s[2].scalar_type())};
  }
};

PyObject* py_stream_mix(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[3];
  if (n != 3 || !tensors(a, 3, t)) return none();
  const Tensor& H = t[0];
  if (code(H) < 0 || H.dim() != 4 || H.size(2) != 4) return none();
  const int64_t B = H.size(0);
  if (t[1].sizes() != at::IntArrayRef({B, 4}) || t[2].sizes() != at::IntArrayRef({B, 4, 4})) return none();
  variable_list out;
  {
    ReleaseGil gil;
    out = wants_grad({t[0], t[1], t[2]}) ? StreamMix::apply(t[0], t[1], t[2]) : stream_mix_forward(t[0], t[1], t[2]);
  }
  return tuple_of(out);
  END_HANDLE_TH_ERRORS
}

Tensor add_residual_forward(const Tensor& hr_in, const Tensor& bo_in, const Tensor& post_in) {
  const c10::DeviceGuard guard(hr_in.device());
  const Dims d(hr_in);
  const Tensor hr = hr_in.contiguous(), bo = bo_in.contiguous(), post = f32(post_in);
  const Tensor out = at::empty(hr.sizes(), hr.options().requires_grad(false));
  check(mhc_add_residual_forward(ptr(hr), code(hr), ptr(bo), code(bo), fptr(post), ptr(out), d.B, d.S, d.D, stream(hr)),
        "add_residual_forward");
  return out;
}

struct AddResidual : Function<AddResidual> {
  static Tensor forward(AutogradContext* ctx, const Tensor& hr, const Tensor& bo, const Tensor& post) {
    const Tensor out = add_residual_forward(hr, bo, post);
    ctx->save_for_backward({bo, post});
    return out;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = saved(ctx);
    const c10::DeviceGuard guard(g[0].device());
    const Tensor dHn = g[0].contiguous(), bo = s[0].contiguous(), post = f32(s[1]);
    const Dims d(dHn);
    const Tensor dbo = at::empty_like(bo);
    const Tensor dpost = empty_f32({d.B, 4}, dHn);
    const Workspace ws(mhc_add_residual_backward_workspace_bytes(d.B, d.S, d.D, code(dHn)), dHn);
    check(mhc_add_residual_backward(ptr(dHn), code(dHn), ptr(bo), code(bo), fptr(post), ptr(dbo), wptr(dpost), d.B,
                                    d.S, d.D, ws.p(), ws.bytes, stream(dHn)),
          "add_residual_backward");
    return {dHn, dbo, dpost.to(s[1].scalar_type())};
  }
};

PyObject* py_add_residual(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[3];
  if (n != 3 || !tensors(a, 3, t)) return none();
  const Tensor &hr = t[0], &bo = t[1];
  if (code(hr) < 0 || code(bo) < 0 || hr.dim() != 4 || hr.size(2) != 4) return none();
  if (bo.sizes() != at::IntArrayRef({hr.size(0), hr.size(1), hr.size(3)}) ||
      t[2].sizes() != at::IntArrayRef({hr.size(0), 4}))
    return none();
  Tensor out;
  {
    ReleaseGil gil;
    out = wants_grad({t[0], t[1], t[2]}) ? AddResidual::apply(t[0], t[1], t[2])
                                         : add_residual_forward(t[0], t[1], t[2]);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// x, phi, bias, alpha_pre, alpha_post, alpha_res
constexpr int kDw = 6;

struct DwOut { Tensor pre, post, res, aux, params; };

DwOut dynamic_weights_forward(const Tensor* t, int64_t iters, double eps) {
  const c10::DeviceGuard guard(t[0].device());
  const Tensor x = t[0].contiguous();
  const int64_t R = x.size(0), K = x.size(1);
  const Params<kDw - 1> q(t + 1, Tensor());
  const float* const* p = q.p;
  DwOut o{empty_f32({R, 4}, x), empty_f32({R, 4}, x), empty_f32({R, 4, 4}, x), empty_f32({R, 25}, x), q.buf};
  const Workspace ws(mhc_dynamic_weights_workspace_bytes(R, K), x);
  check(mhc_dynamic_weights_forward(ptr(x), code(x), p[0], p[1], p[2], p[3], p[4], wptr(o.pre), wptr(o.post),
                                    wptr(o.res), wptr(o.aux), R, K, (int)iters, (float)eps, ws.p(), ws.bytes,
                                    stream(x)),
        "dynamic_weights_forward");
  return o;
}

struct DynamicWeights : Function<DynamicWeights> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& phi, const Tensor& bias,
                               const Tensor& a_pre, const Tensor& a_post, const Tensor& a_res, int64_t iters,
                               double eps) {
    const Tensor t[kDw] = {x, phi, bias, a_pre, a_post, a_res};
    DwOut o = dynamic_weights_forward(t, iters, eps);
    ctx->save_for_backward({x, phi, bias, a_pre, a_post, a_res, o.pre, o.aux, o.params});
    ctx->saved_data["iters"] = iters;
    ctx->saved_data["eps"] = eps;
    ctx->set_materialize_grads(false);
    return {o.pre, o.post, o.res};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = saved(ctx);
    const c10::DeviceGuard guard(s[0].device());
    const Tensor x = s[0].contiguous();
    const int64_t R = x.size(0), K = x.size(1);
    const Params<kDw - 1> q(&s[1], s[8]);
    const float* const* p = q.p;
    const Tensor pre = f32(s[6]), aux = f32(s[7]);
    const Tensor g0 = f32(g[0]), g1 = f32(g[1]), g2 = f32(g[2]);
    const Tensor gx = at::empty(x.sizes(), x.options().requires_grad(false));
    const Tensor gphi = empty_f32({K, 24}, x), small = empty_f32({27}, x);
    const Workspace ws(mhc_dynamic_weights_backward_workspace_bytes(R, K), x);
    check(mhc_dynamic_weights_backward(ptr(x), code(x), p[0], p[1], p[2], p[3], p[4], fptr(aux), fptr(pre), fptr(g0),
                                       fptr(g1), fptr(g2), ptr(gx), wptr(gphi), wptr(small), wptr(small) + 24, R, K,
                                       (int)ctx->saved_data["iters"].toInt(),
                                       (float)ctx->saved_data["eps"].toDouble(), ws.p(), ws.bytes, stream(x)),
          "dynamic_weights_backward");
    const Tensor part[kDw - 1] = {gphi, small.narrow(0, 0, 24), small.narrow(0, 24, 1), small.narrow(0, 25, 1),
                                  small.narrow(0, 26, 1)};
    variable_list out{gx};
    param_grads<kDw - 1>(&s[1], part, out);
    out.resize(kDw + 2);  // iters, eps
    return out;
  }
};

PyObject* py_dynamic_weights(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[kDw];
  int64_t iters;
  double eps;
  if (n != 8 || !tensors(a, kDw, t) || !number(a[6], &iters) || !number(a[7], &eps)) return none();
  const Tensor& x = t[0];
  if (code(x) < 0 || x.dim() != 2 || t[1].sizes() != at::IntArrayRef({x.size(1), 24}) ||
      t[2].sizes() != at::IntArrayRef({24}))
    return none();
  for (int i = 3; i < kDw; ++i)
    if (t[i].numel() != 1) return none();
  variable_list out;
  {
    ReleaseGil gil;
    if (wants_grad({t[0], t[1], t[2], t[3], t[4], t[5]})) {
      out = DynamicWeights::apply(t[0], t[1], t[2], t[3], t[4], t[5], iters, eps);
    } else {
      DwOut o = dynamic_weights_forward(t, iters, eps);
      out = {o.pre, o.post, o.res};
    }
  }
  return tuple_of(out);
  END_HANDLE_TH_ERRORS
}

Tensor expand(const Tensor& x_in, double scale, at::ScalarType dt) {
  const c10::DeviceGuard guard(x_in.device());
  const Tensor x = x_in.contiguous();
  const int64_t B = x.size(0), S = x.size(1), D = x.size(2);
  const Tensor H = at::empty({B, S, 4, D}, x.options().dtype(dt).requires_grad(false));
  check(mhc_stream_expand(ptr(x), code(x), ptr(H), code(H), B, S, D, (float)scale, stream(x)), "stream_expand");
  return H;
}

Tensor collapse(const Tensor& H_in, double scale, at::ScalarType dt) {
  const c10::DeviceGuard guard(H_in.device());
  const Tensor H = H_in.contiguous();
  const Dims d(H);
  const Tensor y = at::empty({d.B, d.S, d.D}, H.options().dtype(dt).requires_grad(false));
  check(mhc_stream_collapse(ptr(H), code(H), ptr(y), code(y), d.B, d.S, d.D, (float)scale, stream(H)),
        "stream_collapse");
  return y;
}

template <bool EXPAND>
struct Ends : Function<Ends<EXPAND>> {
  static Tensor forward(AutogradContext* ctx, const Tensor& t, double scale) {
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["dtype"] = (int64_t)t.scalar_type();
    return EXPAND ? expand(t, scale, t.scalar_type()) : collapse(t, scale, t.scalar_type());
  }

  // each is the other's adjoint
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const double scale = ctx->saved_data["scale"].toDouble();
    const auto dt = (at::ScalarType)ctx->saved_data["dtype"].toInt();
    return {EXPAND ? collapse(g[0], scale, dt) : expand(g[0], scale, dt), Tensor()};
  }
};

template <bool EXPAND>
PyObject* py_ends(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[1];
  double scale;
  if (n != 2 || !tensors(a, 1, t) || !number(a[1], &scale)) return none();
  if (code(t[0]) < 0 || t[0].dim() != (EXPAND ? 3 : 4) || (!EXPAND && t[0].size(2) != 4)) return none();
  Tensor out;
  {
    ReleaseGil gil;
    if (wants_grad({t[0]})) out = Ends<EXPAND>::apply(t[0], scale);
    else out = EXPAND ? expand(t[0], scale, t[0].scalar_type()) : collapse(t[0], scale, t[0].scalar_type());
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* py_set_error(PyObject*, PyObject* cls) {
  Py_INCREF(cls);
  Py_XDECREF(g_error);
  g_error = cls;
  Py_RETURN_NONE;
}

#define FAST(f) (PyCFunction)(void (*)(void)) f, METH_FASTCALL, nullptr

PyMethodDef methods[] = {
    {"dynamic_layer", FAST(py_dynamic_layer)},   {"static_layer", FAST(py_static_layer)},
    {"layer_add", FAST(py_layer_add)},           {"sinkhorn", FAST(py_sinkhorn)},
    {"stream_mix", FAST(py_stream_mix)},         {"add_residual", FAST(py_add_residual)},
    {"dynamic_weights", FAST(py_dynamic_weights)}, {"expand", FAST(py_ends<true>)},
    {"collapse", FAST(py_ends<false>)},          {"set_error", py_set_error, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  return PyModule_Create(&module);
}
