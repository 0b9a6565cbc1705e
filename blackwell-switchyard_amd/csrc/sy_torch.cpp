// The autograd operators as native torch functions over the C ABI: what the Python
// functions of hip_op.py, table_op.py and stats_op.py do on their ordinary inputs,
// without the interpreter. A small forward + backward is bound by the host: the
// Python bodies and their ctypes calls take 16 + 19 us, and twice that when autograd
// alternates between the caller's thread and its own. Forward + backward, N=4 T=256
// D=512 fp32 (14 us on the device): 122-133 us, here 40-59; N=9 T=4096 D=2048 bf16
// 135, here 88 (the device's time); a forward of 8 tokens 15.0, here 6.3.
//
// Every function here returns nullopt (None) instead of a result for a call that is
// not ordinary -- anything its checks refuse, no tokens, transforms, modes, tracing,
// forward-mode tangents -- and the caller then takes the Python path, which raises or
// handles it. Nothing is cached between calls.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <optional>
#include <vector>

#include "../../include/switchyard.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

int code_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return SY_F32;
    case at::kHalf: return SY_F16;
    case at::kBFloat16: return SY_BF16;
    default: return -1;
  }
}

void check(int64_t rc, const char* what) {
  if (rc != 0)
    throw std::runtime_error(std::string(what) + " failed (" + std::to_string(rc) +
                             "): " + sy_strerror((int)rc));
}

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// A dense GPU tensor of a supported dtype that nothing intercepts: no tensor subclass
// with its own dispatch, no transform's wrapper, no lazy negation or conjugation, no
// forward-mode tangent.
bool plain(const Tensor& t) {
  using c10::DispatchKey;
  constexpr c10::DispatchKeySet wrapped{DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                        DispatchKey::Batched, DispatchKey::Functionalize};
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && code_of(t) >= 0 &&
         !t.unsafeGetTensorImpl()->is_python_dispatch() && !t.key_set().has_any(wrapped) && !t.is_neg() &&
         !t.is_conj() && !t._fw_grad(0).defined();
}

// No function transform (vmap, grad, jvp), torch dispatch or function mode, nor tracer
// is active on this thread.
bool ordinary() {
  return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
         !torch::jit::tracer::isTracing();
}

Tensor dense(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }

// A dense copy in `like`'s dtype where the gradient is not already that.
Tensor grad_like(const Tensor& g, const Tensor& like) {
  return dense(g.scalar_type() == like.scalar_type() ? g : g.to(like.scalar_type()));
}

bool needs_grad(const Tensor& a, const Tensor& b) {
  return at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad());
}

at::TensorOptions f32_on(const Tensor& t) { return t.options().dtype(at::kFloat).requires_grad(false); }

// Sizes of stacked sources; `ok` false where the Python path has to see the call.
struct Stacked {
  int64_t n = 0, b = 0, t = 0, d = 0, tok = 0;
  bool ok = false;
};
Stacked sizes_of(const Tensor& v, const Tensor& w, int64_t w_dim) {
  Stacked s;
  if (!plain(v) || !plain(w) || v.dim() != 4 || w.dim() != w_dim || w.device() != v.device()) return s;
  s.n = v.size(0), s.b = v.size(1), s.t = v.size(2), s.d = v.size(3), s.tok = s.b * s.t;
  s.ok = w.size(w_dim - 1) == s.d && s.n > 0 && s.tok > 0 && s.d > 0 && ordinary();
  return s;
}

Tensor bwd_workspace(const Tensor& like, int64_t n, int64_t tok, int64_t d, int vt, int wt) {
  const int64_t bytes = sy_bwd_workspace_bytes(n, tok, d, vt, wt);
  if (bytes < 0) check(bytes, "sy_bwd_workspace_bytes");
  return at::empty({std::max<int64_t>(1, (bytes + 3) / 4)}, f32_on(like));
}

// ------------------------------------------------------------------ operator

Tensor operator_forward(const Tensor& v, const Tensor& w, const Stacked& s, double eps, Tensor* stats) {
  const c10::DeviceGuard guard(v.device());
  Tensor out = at::empty({s.b, s.t, s.d}, v.options().requires_grad(false));
  if (stats != nullptr) *stats = at::empty({2, s.n, s.tok}, f32_on(v));
  check(sy_fwd(v.data_ptr(), w.data_ptr(), out.data_ptr(),
               stats != nullptr ? stats->data_ptr<float>() : nullptr, s.n, s.tok, s.d, s.tok * s.d,
               code_of(v), code_of(w), (float)eps, stream_of(v)),
        "sy_fwd");
  return out;
}

// (dv, dw) of the operator from dense v and w and the forward's statistics.
variable_list operator_backward(const Tensor& v, const Tensor& w, const Tensor& stats, const Tensor& grad,
                                double eps) {
  const c10::DeviceGuard guard(v.device());
  const int64_t n = v.size(0), d = v.size(3), tok = v.size(1) * v.size(2);
  const int vt = code_of(v), wt = code_of(w);
  const Tensor g = grad_like(grad, v);
  Tensor dv = at::empty(v.sizes(), v.options().requires_grad(false));
  Tensor dw = at::empty({d}, w.options().requires_grad(false));
  const Tensor ws = bwd_workspace(v, n, tok, d, vt, wt);
  check(sy_bwd(v.data_ptr(), w.data_ptr(), g.data_ptr(), stats.data_ptr<float>(), dv.data_ptr(),
               dw.data_ptr(), ws.data_ptr(), ws.numel() * 4, n, tok, d, tok * d, vt, wt, (float)eps,
               stream_of(v)),
        "sy_bwd");
  return {dv, dw};
}

struct BlockAttnResHIP : torch::autograd::Function<BlockAttnResHIP> {
  static Tensor forward(AutogradContext* ctx, const Tensor& v_in, const Tensor& w_in, double eps) {
    const Tensor v = dense(v_in), w = dense(w_in);
    Stacked s{v.size(0), v.size(1), v.size(2), v.size(3), v.size(1) * v.size(2), true};
    Tensor stats;
    Tensor out = operator_forward(v, w, s, eps, &stats);
    ctx->save_for_backward({v, w, stats});
    ctx->saved_data["eps"] = eps;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    auto r = operator_backward(saved[0], saved[1], saved[2], grads[0], ctx->saved_data["eps"].toDouble());
    return {r[0], r[1], Tensor()};
  }
};

std::optional<Tensor> block_attn_res(const Tensor& v, const Tensor& w, double eps) {
  const Stacked s = sizes_of(v, w, 1);
  if (!s.ok) return std::nullopt;
  if (needs_grad(v, w)) return BlockAttnResHIP::apply(v, w, eps);
  return operator_forward(dense(v), dense(w), s, eps, nullptr);
}

// ------------------------------------------- the module: a query and its gain

Tensor gain_forward(const Tensor& v, const Tensor& w, const Tensor& g, double eps, Tensor* stats) {
  const c10::DeviceGuard guard(v.device());
  const int64_t n = v.size(0), b = v.size(1), t = v.size(2), d = v.size(3), tok = b * t;
  Tensor out = at::empty({b, t, d}, v.options().requires_grad(false));
  if (stats != nullptr) *stats = at::empty({2, n, tok}, f32_on(v));
  check(sy_fwd_gain(v.data_ptr(), w.data_ptr(), g.data_ptr(), out.data_ptr(),
                    stats != nullptr ? stats->data_ptr<float>() : nullptr, n, tok, d, tok * d, code_of(v),
                    code_of(w), (float)eps, stream_of(v)),
        "sy_fwd_gain");
  return out;
}

struct BlockAttnResGain : torch::autograd::Function<BlockAttnResGain> {
  static Tensor forward(AutogradContext* ctx, const Tensor& v_in, const Tensor& w_in, const Tensor& g_in,
                        double eps) {
    const Tensor v = dense(v_in), w = dense(w_in), g = dense(g_in);
    Tensor stats;
    Tensor out = gain_forward(v, w, g, eps, &stats);
    ctx->save_for_backward({v, w, g, stats});
    ctx->saved_data["eps"] = eps;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &v = saved[0], &w = saved[1];
    const c10::DeviceGuard guard(v.device());
    if (at::GradMode::is_enabled()) {
      // Recorded: the product's own gradients are torch operations, through which the
      // factors can be differentiated again (the operator's carry no graph).
      const Tensor wf = w.to(at::kFloat), gf = saved[2].to(at::kFloat);
      const auto r = operator_backward(v, (wf * gf).detach(), saved[3], grads[0],
                                       ctx->saved_data["eps"].toDouble());
      return {r[0], (r[1] * gf).to(w.scalar_type()), (r[1] * wf).to(w.scalar_type()), Tensor()};
    }
    const int64_t n = v.size(0), d = v.size(3), tok = v.size(1) * v.size(2);
    const int vt = code_of(v), wt = code_of(w);
    const Tensor go = grad_like(grads[0], v);
    Tensor dv = at::empty(v.sizes(), v.options().requires_grad(false));
    Tensor dw = at::empty({d}, w.options().requires_grad(false));
    Tensor dg = at::empty({d}, w.options().requires_grad(false));
    const Tensor ws = bwd_workspace(v, n, tok, d, vt, wt);
    check(sy_bwd_gain(v.data_ptr(), w.data_ptr(), saved[2].data_ptr(), go.data_ptr(),
                      saved[3].data_ptr<float>(), dv.data_ptr(), dw.data_ptr(), dg.data_ptr(), ws.data_ptr(),
                      ws.numel() * 4, n, tok, d, tok * d, vt, wt, (float)ctx->saved_data["eps"].toDouble(),
                      stream_of(v)),
          "sy_bwd_gain");
    return {dv, dw, dg, Tensor()};
  }
};

std::optional<Tensor> block_attn_res_gain(const Tensor& v, const Tensor& w, const Tensor& g, double eps) {
  if (!sizes_of(v, w, 1).ok || !plain(g) || g.sizes() != w.sizes() || g.scalar_type() != w.scalar_type() ||
      g.device() != w.device())
    return std::nullopt;
  if (needs_grad(v, w) || (at::GradMode::is_enabled() && g.requires_grad()))
    return BlockAttnResGain::apply(v, w, g, eps);
  return gain_forward(dense(v), dense(w), dense(g), eps, nullptr);
}

// --------------------------------------------------- sources as separate tensors

struct BlockAttnResSources : torch::autograd::Function<BlockAttnResSources> {
  static Tensor forward(AutogradContext* ctx, const Tensor& w_in, double eps, at::TensorList sources);
  static variable_list backward(AutogradContext* ctx, variable_list grads);
};

Tensor sources_forward(const Tensor& w, const variable_list& rows, double eps, Tensor* stats) {
  const Tensor& first = rows[0];
  const c10::DeviceGuard guard(first.device());
  const int64_t n = (int64_t)rows.size(), d = first.size(2), tok = first.size(0) * first.size(1);
  Tensor out = at::empty(first.sizes(), first.options().requires_grad(false));
  if (stats != nullptr) *stats = at::empty({2, n, tok}, f32_on(first));
  const void* p[SY_MAX_TABLE_ROWS];
  for (int64_t k = 0; k < n; ++k) p[k] = rows[k].data_ptr();
  check(sy_fwd_table(p, w.data_ptr(), out.data_ptr(), stats != nullptr ? stats->data_ptr<float>() : nullptr,
                     n, tok, d, code_of(first), code_of(w), (float)eps, stream_of(first)),
        "sy_fwd_table");
  return out;
}

Tensor BlockAttnResSources::forward(AutogradContext* ctx, const Tensor& w_in, double eps,
                                    at::TensorList sources) {
  const Tensor w = dense(w_in);
  variable_list rows;
  rows.reserve(sources.size() + 2);
  for (const Tensor& s : sources) rows.push_back(dense(s));
  Tensor stats;
  Tensor out = sources_forward(w, rows, eps, &stats);
  rows.push_back(w);
  rows.push_back(stats);
  ctx->save_for_backward(std::move(rows));
  ctx->saved_data["eps"] = eps;
  return out;
}

variable_list BlockAttnResSources::backward(AutogradContext* ctx, variable_list grads) {
  const auto saved = ctx->get_saved_variables();
  const int64_t n = (int64_t)saved.size() - 2;
  const Tensor &first = saved[0], &w = saved[n], &stats = saved[n + 1];
  const c10::DeviceGuard guard(first.device());
  const int64_t d = first.size(2), tok = first.size(0) * first.size(1);
  const int vt = code_of(first), wt = code_of(w);
  const Tensor g = grad_like(grads[0], first);
  // One allocation; each source's gradient is a slice of it.
  const variable_list dvs =
      at::empty({n, first.size(0), first.size(1), d}, first.options().requires_grad(false)).unbind(0);
  Tensor dw = at::empty({d}, w.options().requires_grad(false));
  const Tensor ws = bwd_workspace(first, n, tok, d, vt, wt);
  const void* p[SY_MAX_TABLE_ROWS];
  void* q[SY_MAX_TABLE_ROWS];
  for (int64_t k = 0; k < n; ++k) {
    p[k] = saved[k].data_ptr();
    q[k] = dvs[k].data_ptr();
  }
  check(sy_bwd_table(p, w.data_ptr(), g.data_ptr(), stats.data_ptr<float>(), q, dw.data_ptr(),
                     ws.data_ptr(), ws.numel() * 4, n, tok, d, vt, wt,
                     (float)ctx->saved_data["eps"].toDouble(), stream_of(first)),
        "sy_bwd_table");
  variable_list r{dw, Tensor()};
  r.insert(r.end(), dvs.begin(), dvs.end());
  return r;
}

std::optional<Tensor> block_attn_res_sources(const std::vector<Tensor>& sources, const Tensor& w,
                                             double eps) {
  if (sources.empty() || sources.size() > SY_MAX_TABLE_ROWS || !ordinary()) return std::nullopt;
  const Tensor& first = sources[0];
  if (!plain(first) || !plain(w) || first.dim() != 3 || first.numel() == 0 || w.dim() != 1 ||
      w.size(0) != first.size(2) || w.device() != first.device())
    return std::nullopt;
  bool grad = w.requires_grad();
  for (const Tensor& s : sources) {
    if (!plain(s) || s.sizes() != first.sizes() || s.device() != first.device() ||
        s.scalar_type() != first.scalar_type())
      return std::nullopt;
    grad = grad || s.requires_grad();
  }
  if (grad && at::GradMode::is_enabled()) return BlockAttnResSources::apply(w, eps, at::TensorList(sources));
  variable_list rows;
  for (const Tensor& s : sources) rows.push_back(dense(s));
  return sources_forward(dense(w), rows, eps, nullptr);
}

// ----------------------------------------------------------------- two phases

Tensor two_phase_forward(const Tensor& v, const Tensor& w, int64_t split, double eps, Tensor* stats) {
  const c10::DeviceGuard guard(v.device());
  const int64_t n = v.size(0), b = v.size(1), t = v.size(2), d = v.size(3), tok = b * t;
  Tensor out = at::empty({b, t, d}, v.options().requires_grad(false));
  if (stats != nullptr) *stats = at::empty({2, n, tok}, f32_on(v));
  const Tensor o1 = at::empty_like(out), ml = at::empty({4, tok}, f32_on(v));
  check(sy_two_phase(v.data_ptr(), w.data_ptr(), o1.data_ptr(), ml.data_ptr<float>(), out.data_ptr(),
                     stats != nullptr ? stats->data_ptr<float>() : nullptr, n, split, tok, d, tok * d,
                     code_of(v), code_of(w), (float)eps, stream_of(v)),
        "sy_two_phase");
  return out;
}

struct TwoPhase : torch::autograd::Function<TwoPhase> {
  static Tensor forward(AutogradContext* ctx, const Tensor& v_in, const Tensor& w_in, int64_t split,
                        double eps) {
    const Tensor v = dense(v_in), w = dense(w_in);
    Tensor stats;
    Tensor out = two_phase_forward(v, w, split, eps, &stats);
    ctx->save_for_backward({v, w, stats});
    ctx->saved_data["eps"] = eps;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    auto r = operator_backward(saved[0], saved[1], saved[2], grads[0], ctx->saved_data["eps"].toDouble());
    return {r[0], r[1], Tensor(), Tensor()};
  }
};

std::optional<Tensor> block_attn_res_two_phase(const Tensor& v, const Tensor& w, int64_t split, double eps) {
  const Stacked s = sizes_of(v, w, 1);
  if (!s.ok || split < 1 || split >= s.n) return std::nullopt;
  if (needs_grad(v, w)) return TwoPhase::apply(v, w, split, eps);
  return two_phase_forward(dense(v), dense(w), split, eps, nullptr);
}

// -------------------------------------------------------------------- batched

Tensor batched_forward(const Tensor& v, const Tensor& q, double eps) {
  const c10::DeviceGuard guard(v.device());
  const int64_t n = v.size(0), b = v.size(1), t = v.size(2), d = v.size(3), s = q.size(0);
  Tensor out = at::empty({s, b, t, d}, v.options().requires_grad(false));
  check(sy_fwd_batched(v.data_ptr(), q.data_ptr(), out.data_ptr(), n, s, b * t, d, b * t * d, code_of(v),
                       (float)eps, stream_of(v)),
        "sy_fwd_batched");
  return out;
}

struct BlockAttnResBatched : torch::autograd::Function<BlockAttnResBatched> {
  static Tensor forward(AutogradContext* ctx, const Tensor& v_in, const Tensor& q_in, double eps) {
    const Tensor v = dense(v_in), q = dense(q_in);
    ctx->save_for_backward({v, q});
    ctx->saved_data["eps"] = eps;
    return batched_forward(v, q, eps);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &v = saved[0], &q = saved[1];
    const c10::DeviceGuard guard(v.device());
    const int64_t n = v.size(0), d = v.size(3), tok = v.size(1) * v.size(2), s = q.size(0);
    const int dt = code_of(v);
    const Tensor g = grad_like(grads[0], v);
    Tensor dv = at::empty(v.sizes(), v.options().requires_grad(false));
    Tensor dq = at::empty(q.sizes(), q.options().requires_grad(false));
    const int64_t bytes = sy_bwd_batched_workspace_bytes(n, s, tok, d, dt);
    if (bytes < 0) check(bytes, "sy_bwd_batched_workspace_bytes");
    const Tensor ws = at::empty({std::max<int64_t>(1, (bytes + 3) / 4)}, f32_on(v));
    check(sy_bwd_batched(v.data_ptr(), q.data_ptr(), g.data_ptr(), dv.data_ptr(), dq.data_ptr(),
                         ws.data_ptr(), ws.numel() * 4, n, s, tok, d, tok * d, dt,
                         (float)ctx->saved_data["eps"].toDouble(), stream_of(v)),
          "sy_bwd_batched");
    return {dv, dq, Tensor()};
  }
};

bool batched_ok(const Tensor& v, const Tensor& q) {
  return sizes_of(v, q, 2).ok && q.size(0) > 0 && v.scalar_type() == q.scalar_type();
}

std::optional<Tensor> block_attn_res_batched(const Tensor& v, const Tensor& q, double eps) {
  if (!batched_ok(v, q) || v.requires_grad() || q.requires_grad()) return std::nullopt;
  return batched_forward(dense(v), dense(q), eps);
}

std::optional<Tensor> block_attn_res_batched_train(const Tensor& v, const Tensor& q, double eps) {
  if (!batched_ok(v, q)) return std::nullopt;
  if (needs_grad(v, q)) return BlockAttnResBatched::apply(v, q, eps);
  return batched_forward(dense(v), dense(q), eps);
}

// ------------------------------------------------------------ decoder sublayers

bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
int64_t chunk(const Tensor& t) { return 16 / (int64_t)t.element_size(); }

// Whether a backward may launch its kernel. A recorded one (create_graph) may not, as
// the kernels' results carry no graph, nor one inside a transform or mode or given a
// wrapped gradient (is_grads_batched): those evaluate the same gradient from torch
// operations in fp32.
bool kernel_backward(const variable_list& grads) {
  if (at::GradMode::is_enabled() || !ordinary()) return false;
  for (const Tensor& g : grads)
    if (!plain(g)) return false;
  return true;
}

Tensor norm_forward(const Tensor& x, const Tensor& w, double eps, Tensor* rinv) {
  const c10::DeviceGuard guard(x.device());
  const int64_t d = w.size(0), tok = x.numel() / d;
  Tensor out = at::empty(x.sizes(), x.options().requires_grad(false));
  if (rinv != nullptr) *rinv = at::empty({tok}, f32_on(x));
  check(sy_rms_norm(x.data_ptr(), w.data_ptr(), out.data_ptr(),
                    rinv != nullptr ? rinv->data_ptr<float>() : nullptr, tok, d, code_of(x), (float)eps,
                    stream_of(x)),
        "sy_rms_norm");
  return out;
}

struct RmsNorm : torch::autograd::Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    Tensor rinv;
    Tensor out = norm_forward(x, w, eps, &rinv);
    ctx->save_for_backward({x, w, rinv});
    ctx->saved_data["eps"] = eps;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1];
    const c10::DeviceGuard guard(x.device());
    if (!kernel_backward(grads)) {
      const Tensor xf = x.to(at::kFloat), gf = grads[0].to(at::kFloat), gw = gf * w.to(at::kFloat);
      const Tensor r = xf.square().mean(-1, /*keepdim=*/true).add(ctx->saved_data["eps"].toDouble()).rsqrt();
      const Tensor dx = r * gw - xf * (r.pow(3) * (gw * xf).mean(-1, /*keepdim=*/true));
      const Tensor dw = (gf * xf * r).reshape({-1, w.size(0)}).sum(0);
      return {dx.to(x.scalar_type()), dw.to(w.scalar_type()), Tensor()};
    }
    const int64_t d = w.size(0), tok = x.numel() / d;
    Tensor g = grad_like(grads[0], x);
    if (!aligned16(g)) g = g.clone();
    Tensor dx = at::empty(x.sizes(), x.options().requires_grad(false));
    Tensor dw = at::empty({d}, w.options().requires_grad(false));
    const int64_t bytes = sy_rms_norm_bwd_bytes(tok, d);
    if (bytes < 0) check(bytes, "sy_rms_norm_bwd_bytes");
    const Tensor ws = at::empty({std::max<int64_t>(1, bytes / 4)}, f32_on(x));
    check(sy_rms_norm_bwd(x.data_ptr(), w.data_ptr(), g.data_ptr(), saved[2].data_ptr<float>(), dx.data_ptr(),
                          dw.data_ptr(), ws.data_ptr(), ws.numel() * 4, tok, d, code_of(x), stream_of(x)),
          "sy_rms_norm_bwd");
    return {dx, dw, Tensor()};
  }
};

std::optional<Tensor> rms_norm(const Tensor& x, const Tensor& w, double eps) {
  if (!ordinary() || !plain(x) || !plain(w) || w.dim() != 1 || x.dim() < 1 || x.numel() == 0 ||
      x.size(-1) != w.size(0) || x.scalar_type() != w.scalar_type() || x.device() != w.device() ||
      !x.is_contiguous() || !w.is_contiguous() || !aligned16(x) || !aligned16(w) ||
      w.size(0) % chunk(x) != 0 || w.size(0) / chunk(x) > 512)
    return std::nullopt;
  if (needs_grad(x, w)) return RmsNorm::apply(x, w, eps);
  return norm_forward(x, w, eps, nullptr);
}

variable_list rope_forward(const Tensor& qkv, const Tensor& cosv, const Tensor& sinv) {
  const c10::DeviceGuard guard(qkv.device());
  const int64_t b = qkv.size(0), t = qkv.size(1), h = qkv.size(3), hd = qkv.size(4);
  variable_list r;
  for (int k = 0; k < 3; ++k) r.push_back(at::empty({b, h, t, hd}, qkv.options().requires_grad(false)));
  check(sy_rope_qkv(qkv.data_ptr(), r[0].data_ptr(), r[1].data_ptr(), r[2].data_ptr(),
                    cosv.data_ptr<float>(), sinv.data_ptr<float>(), b * t, t, h, hd, code_of(qkv), 0,
                    stream_of(qkv)),
        "sy_rope_qkv");
  return r;
}

struct RopeQkv : torch::autograd::Function<RopeQkv> {
  static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& cosv,
                               const Tensor& sinv) {
    ctx->save_for_backward({cosv, sinv});
    return rope_forward(qkv, cosv, sinv);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    if (!kernel_backward(grads)) {  // the kernel's inverse rotation
      const int64_t t = grads[0].size(2), half = grads[0].size(3) / 2;
      const Tensor c = saved[0].reshape({-1, half}).slice(0, 0, t), s = saved[1].reshape({-1, half}).slice(0, 0, t);
      variable_list d;
      for (int k = 0; k < 3; ++k) {
        Tensor g = grads[k];
        if (k < 2) {
          const auto p = g.to(at::kFloat).chunk(2, -1);
          g = at::cat({p[0] * c + p[1] * s, p[1] * c - p[0] * s}, -1).to(g.scalar_type());
        }
        d.push_back(g.transpose(1, 2));
      }
      return {at::stack(d, 2), Tensor(), Tensor()};
    }
    for (Tensor& g : grads) {
      g = dense(g);
      if (!aligned16(g)) g = g.clone();
    }
    const Tensor& q = grads[0];
    const c10::DeviceGuard guard(q.device());
    const int64_t b = q.size(0), h = q.size(1), t = q.size(2), hd = q.size(3);
    Tensor dqkv = at::empty({b, t, 3, h, hd}, q.options().requires_grad(false));
    check(sy_rope_qkv(dqkv.data_ptr(), q.data_ptr(), grads[1].data_ptr(), grads[2].data_ptr(),
                      saved[0].data_ptr<float>(), saved[1].data_ptr<float>(), b * t, t, h, hd, code_of(q), 1,
                      stream_of(q)),
          "sy_rope_qkv");
    return {dqkv, Tensor(), Tensor()};
  }
};

// qkv [B, T, 3, H, hd], tables [>= T, 1, hd/2] -> (q, k, v), each [B, H, T, hd].
std::optional<variable_list> rope_qkv(const Tensor& qkv, const Tensor& cosv, const Tensor& sinv) {
  if (!ordinary() || !plain(qkv) || !plain(cosv) || !plain(sinv) || qkv.dim() != 5 || qkv.size(2) != 3 ||
      qkv.numel() == 0 || !qkv.is_contiguous() || !aligned16(qkv) || qkv.size(4) % (2 * chunk(qkv)) != 0 ||
      qkv.size(3) > 0xffff || qkv.size(4) > 0xffff)
    return std::nullopt;
  for (const Tensor* t : {&cosv, &sinv})
    if (t->scalar_type() != at::kFloat || t->device() != qkv.device() || !t->is_contiguous() ||
        t->requires_grad() || t->dim() != 3 || t->size(1) != 1 || t->size(2) != qkv.size(4) / 2 ||
        t->size(0) < qkv.size(1))
      return std::nullopt;
  if (at::GradMode::is_enabled() && qkv.requires_grad()) return RopeQkv::apply(qkv, cosv, sinv);
  return rope_forward(qkv, cosv, sinv);
}

struct SwiGlu : torch::autograd::Function<SwiGlu> {
  static Tensor run(const Tensor& gu) {
    const c10::DeviceGuard guard(gu.device());
    auto sizes = gu.sizes().vec();
    const int64_t f = sizes.back() / 2;
    sizes.back() = f;
    Tensor out = at::empty(sizes, gu.options().requires_grad(false));
    check(sy_swiglu(gu.data_ptr(), out.data_ptr(), out.numel() / f, f, code_of(gu), stream_of(gu)), "sy_swiglu");
    return out;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& gu) {
    ctx->save_for_backward({gu});
    return run(gu);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor gu = ctx->get_saved_variables()[0];
    const c10::DeviceGuard guard(gu.device());
    if (!kernel_backward(grads)) {
      const auto p = gu.to(at::kFloat).chunk(2, -1);
      const Tensor gf = grads[0].to(at::kFloat), s = at::sigmoid(p[0]);
      return {at::cat({gf * p[1] * s * (1 + p[0] * (1 - s)), gf * p[0] * s}, -1).to(gu.scalar_type())};
    }
    Tensor g = grad_like(grads[0], gu);
    if (!aligned16(g)) g = g.clone();
    Tensor d = at::empty(gu.sizes(), gu.options().requires_grad(false));
    const int64_t f = gu.size(-1) / 2;
    check(sy_swiglu_bwd(gu.data_ptr(), g.data_ptr(), d.data_ptr(), g.numel() / f, f, code_of(gu),
                        stream_of(gu)),
          "sy_swiglu_bwd");
    return {d};
  }
};

std::optional<Tensor> swiglu(const Tensor& gu) {
  if (!ordinary() || !plain(gu) || gu.dim() < 1 || gu.numel() == 0 || !gu.is_contiguous() || !aligned16(gu) ||
      gu.size(-1) % (2 * chunk(gu)) != 0)
    return std::nullopt;
  if (at::GradMode::is_enabled() && gu.requires_grad()) return SwiGlu::apply(gu);
  return SwiGlu::run(gu);
}

}  // namespace

// The interpreter's lock is released during a call, as ctypes does.
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  const auto free_lock = py::call_guard<py::gil_scoped_release>();
  m.def("block_attn_res", &block_attn_res, free_lock);
  m.def("block_attn_res_gain", &block_attn_res_gain, free_lock);
  m.def("block_attn_res_sources", &block_attn_res_sources, free_lock);
  m.def("block_attn_res_two_phase", &block_attn_res_two_phase, free_lock);
  m.def("block_attn_res_batched", &block_attn_res_batched, free_lock);
  m.def("block_attn_res_batched_train", &block_attn_res_batched_train, free_lock);
  m.def("rms_norm", &rms_norm, free_lock);
  m.def("rope_qkv", &rope_qkv, free_lock);
  m.def("swiglu", &swiglu, free_lock);
}
