// Native host side of the Python entry points: argument checks, output
// allocation, kernel launches and the autograd nodes of their common calls.
//
// A small call of these ops is bound by the host, not by its kernels (a
// training step's loss over 64 x 512 logits takes 115 us through Python and
// ctypes, 61 us through these functions, and has about 20 us of kernels; an
// inference scan 21 and 5 us, a norm's forward and backward 250 and 43-90 us,
// since a backward in Python also waits for autograd's thread). Every function
// here takes the plain form of one entry point (dense tensors of the kernels'
// types on the current GPU) and returns nothing for any other form, or when
// something that wants to see the single steps is in force (a dispatch or
// function mode, a functorch transform): the Python code then takes the call,
// with its conversions and its errors. The kernels come from the C library,
// whose path the loader passes in, so there is one copy of them in the process.
#include <dlfcn.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/engine.h>
#include <torch/extension.h>

#include "autokernel_mi355x.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using Maybe = std::optional<Tensor>;

#define AK_ENTRIES(X)                                                                              \
  X(ak_last_error) X(ak_rmsnorm_fwd) X(ak_fused_add_rmsnorm_fwd) X(ak_rmsnorm_bwd_workspace_bytes) \
  X(ak_fused_add_rmsnorm_bwd_gw) X(ak_softmax_fwd) X(ak_ce_fwd) X(ak_ce_bwd_tiny)   \
  X(ak_ce_count_valid) X(ak_ce_mean) X(ak_scale_inplace) X(ak_diag_scan_fwd)                       \
  X(ak_diag_scan_bwd_workspace_bytes) X(ak_diag_scan_bwd) X(ak_selective_scan_fwd_ws) X(ak_selective_scan_fwd_workspace_bytes)                 \
  X(ak_selective_scan_bwd_workspace_bytes) X(ak_selective_scan_bwd)                                \
  X(ak_lmhead_ce_workspace_bytes) X(ak_lmhead_ce_fwd_denom) X(ak_lmhead_ce_bwd_range)                    \
  X(ak_lmhead_grad_workspace_bytes) X(ak_lmhead_grad_hidden) X(ak_lmhead_grad_weight)

#define AK_FIELD(n) decltype(&::n) n = nullptr;
struct Api { AK_ENTRIES(AK_FIELD) } api;
#undef AK_FIELD

void init(const std::string& path) {
  void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(h, "cannot open ", path, ": ", dlerror());
  Api a;
#define AK_LOAD(n)                                                  \
  a.n = reinterpret_cast<decltype(&::n)>(dlsym(h, #n));             \
  TORCH_CHECK(a.n, #n " is missing from ", path);
  AK_ENTRIES(AK_LOAD)
#undef AK_LOAD
  api = a;
}

void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed (", rc, "): ", api.ak_last_error());
}

int code_of(at::ScalarType t) {
  return t == at::kFloat ? AK_DTYPE_F32 : t == at::kHalf ? AK_DTYPE_F16 : t == at::kBFloat16 ? AK_DTYPE_BF16 : -1;
}

// A dense GPU tensor that nothing wraps (no subclass with its own dispatch, no
// functorch level, no lazy conjugate or negative).
bool plain(const Tensor& t) {
  static const uint64_t known =
      (c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
       c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA))
          .raw_repr();
  return t.defined() && t.is_cuda() && (t.key_set().raw_repr() & ~known) == 0 &&
         !t._fw_grad(0).defined();
}

// (function modes are the loader's to look at: a default device is one, too)
bool quiet() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// Whether a call on `first` and the others (all of one GPU, the current one) is ours.
template <typename... Ts>
bool ours(const Tensor& first, const Ts&... rest) {
  if (!api.ak_last_error || !quiet() || !plain(first) || first.get_device() != c10::hip::current_device()) return false;
  return ((plain(rest) && rest.get_device() == first.get_device()) && ...);
}

bool ours_if(const Maybe& t, const Tensor& first) {
  return !t || (plain(*t) && t->get_device() == first.get_device());
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* f32p(const Tensor& t) { return static_cast<float*>(ptr(t)); }
Tensor f32_like(const Tensor& t, at::IntArrayRef size) { return at::empty(size, t.options().dtype(at::kFloat)); }
Tensor bytes_like(const Tensor& t, size_t n) { return at::empty({(int64_t)n}, t.options().dtype(at::kByte)); }

// A saved tensor as a kernel takes it: saved-tensor hooks may hand back another
// layout or type.
Tensor saved_as(const Tensor& t, at::ScalarType type) { return t.defined() ? t.to(type).contiguous() : t; }

// t as rows of cols elements the row kernels take (last dimension contiguous,
// rows that do not overlap), copied only if it is not; ld gets the row pitch.
Tensor rows_of(const Tensor& t, int64_t cols, int64_t& ld) {
  ld = cols;
  if (t.is_contiguous()) return t;
  Tensor r = t.reshape({-1, cols});
  if ((cols > 1 && r.stride(1) != 1) || (r.size(0) > 1 && r.stride(0) < cols)) r = r.contiguous();
  if (r.size(0) > 1) ld = r.stride(0);
  return r;
}

bool records(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// The torch formulas that stand in for the norm and diagonal-scan backward
// kernels where those are switched off (a Python callable per op).
bool hip_backward = true;
std::map<std::string, py::object>* formulas = new std::map<std::string, py::object>();  // never destroyed

void set_hip_backward(bool on) { hip_backward = on; }
void set_formula(const std::string& op, py::object fn) { (*formulas)[op] = std::move(fn); }

variable_list by_formula(const char* op, const variable_list& args, double eps) {
  py::gil_scoped_acquire gil;
  py::tuple a(args.size());
  for (size_t i = 0; i < args.size(); ++i) a[i] = args[i].defined() ? py::cast(args[i]) : py::none();
  variable_list out;
  for (py::handle h : formulas->at(op)(a, eps)) out.push_back(h.is_none() ? Tensor() : h.cast<Tensor>());
  return out;
}

// ---------------------------------------------------------------------------
// Norms and softmax
// ---------------------------------------------------------------------------
bool norm_args(const Tensor& x, const Tensor& w) {
  return x.dim() >= 1 && w.dim() == 1 && x.is_contiguous() && w.is_contiguous() && x.scalar_type() == w.scalar_type() &&
         code_of(x.scalar_type()) >= 0 && w.size(0) == x.size(-1) && x.numel() > 0;
}

Tensor run_rmsnorm(const Tensor& x, const Tensor& w, double eps) {
  Tensor y = at::empty(x.sizes(), x.options());
  const int64_t cols = x.size(-1);
  check(api.ak_rmsnorm_fwd(x.data_ptr(), w.data_ptr(), y.data_ptr(), x.numel() / cols, cols, cols, cols, (float)eps,
                           code_of(x.scalar_type()), stream_of(x)), "ak_rmsnorm_fwd");
  return y;
}

Maybe rmsnorm(const Tensor& x, const Tensor& w, double eps) {
  if (!ours(x, w) || !norm_args(x, w)) return std::nullopt;
  return run_rmsnorm(x, w, eps);
}

void run_add_rmsnorm(const Tensor& x, const Tensor& r, const Tensor& w, double eps, const Tensor& h, const Tensor& y) {
  const int64_t cols = x.size(-1);
  check(api.ak_fused_add_rmsnorm_fwd(x.data_ptr(), r.data_ptr(), w.data_ptr(), ptr(h), y.data_ptr(), x.numel() / cols,
                                     cols, cols, cols, cols, cols, (float)eps, code_of(x.scalar_type()), stream_of(x)),
        "ak_fused_add_rmsnorm_fwd");
}

bool add_norm_args(const Tensor& x, const Tensor& r, const Tensor& w) {
  return norm_args(x, w) && r.scalar_type() == x.scalar_type() && r.sizes() == x.sizes() && r.is_contiguous();
}

Maybe add_rmsnorm(const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
  if (!ours(x, r, w) || !add_norm_args(x, r, w)) return std::nullopt;
  Tensor y = at::empty(x.sizes(), x.options());
  run_add_rmsnorm(x, r, w, eps, Tensor(), y);
  return y;
}

using Pair = std::optional<std::tuple<Tensor, Tensor>>;

Pair add_rmsnorm_dual(const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
  if (!ours(x, r, w) || !add_norm_args(x, r, w)) return std::nullopt;
  Tensor h = at::empty(x.sizes(), x.options()), y = at::empty(x.sizes(), x.options());
  run_add_rmsnorm(x, r, w, eps, h, y);
  return std::make_tuple(h, y);
}

// (grad_x, grad_w) of the norm of h; gh: the gradient that reaches h beside it, if any.
std::pair<Tensor, Tensor> norm_backward(const Tensor& h, const Tensor& w, const Tensor& gh, const Tensor& gy, double eps) {
  const int64_t cols = h.size(-1), rows = h.numel() / cols;
  int64_t ld_y = cols, ld_h = cols;
  Tensor y = rows_of(gy.to(h.scalar_type()), cols, ld_y), g;
  if (gh.defined()) g = rows_of(gh.to(h.scalar_type()), cols, ld_h);
  Tensor gx = at::empty(h.sizes(), h.options()), gw = at::empty({cols}, w.options());
  const size_t bytes = api.ak_rmsnorm_bwd_workspace_bytes(rows, cols);
  Tensor ws = bytes_like(h, bytes);
  check(api.ak_fused_add_rmsnorm_bwd_gw(h.data_ptr(), w.data_ptr(), ptr(g), y.data_ptr(), gx.data_ptr(), gw.data_ptr(),
                                        ws.data_ptr(), bytes, rows, cols, cols, ld_h, ld_y, cols, (float)eps,
                                        code_of(h.scalar_type()), stream_of(h)), "ak_fused_add_rmsnorm_bwd_gw");
  return {gx, gw};
}

struct RmsNorm : torch::autograd::Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    ctx->save_for_backward({x, w});
    ctx->saved_data["eps"] = eps;
    return run_rmsnorm(x, w, eps);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const double eps = ctx->saved_data["eps"].toDouble();
    if (!hip_backward) {
      variable_list r = by_formula("rmsnorm", {s[0], s[1], g[0]}, eps);
      return {r[0], r[1], Tensor()};
    }
    const Tensor x = s[0].contiguous(), w = saved_as(s[1], x.scalar_type());
    auto [gx, gw] = norm_backward(x, w, Tensor(), g[0], eps);
    return {gx, gw, Tensor()};
  }
};

struct AddRmsNorm : torch::autograd::Function<AddRmsNorm> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
    Tensor h = at::empty(x.sizes(), x.options()), y = at::empty(x.sizes(), x.options());
    run_add_rmsnorm(x, r, w, eps, h, y);
    ctx->save_for_backward({h, w});
    ctx->saved_data["eps"] = eps;
    ctx->set_materialize_grads(false);
    return {h, y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const double eps = ctx->saved_data["eps"].toDouble();
    if (!g[1].defined()) {  // only the sum was used, or neither output's gradient came
      Tensor gx = g[0].defined() ? g[0].to(s[0].scalar_type()) : at::zeros_like(s[0]);
      return {gx, gx, at::zeros_like(s[1]), Tensor()};
    }
    if (!hip_backward) {
      variable_list r = by_formula("fused_res_rmsnorm", {s[0], s[1], g[0], g[1]}, eps);
      return {r[0], r[1], r[2], Tensor()};
    }
    const Tensor h = s[0].contiguous(), w = saved_as(s[1], h.scalar_type());
    auto [gx, gw] = norm_backward(h, w, g[0], g[1], eps);
    return {gx, gx, gw, Tensor()};
  }
};

// The registered ops: with autograd where it records, otherwise the plain call.
Maybe rmsnorm_op(const Tensor& x, const Tensor& w, double eps) {
  if (!ours(x, w) || !norm_args(x, w)) return std::nullopt;
  return records({&x, &w}) ? RmsNorm::apply(x, w, eps) : run_rmsnorm(x, w, eps);
}

Pair add_rmsnorm_op(const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
  if (!records({&x, &r, &w})) return add_rmsnorm_dual(x, r, w, eps);
  if (!ours(x, r, w) || !add_norm_args(x, r, w)) return std::nullopt;
  variable_list v = AddRmsNorm::apply(x, r, w, eps);
  return std::make_tuple(v[0], v[1]);
}

Maybe softmax(const Tensor& x) {
  if (!ours(x) || x.dim() < 1 || !x.is_contiguous() || x.numel() == 0 || code_of(x.scalar_type()) < 0) return std::nullopt;
  Tensor y = at::empty(x.sizes(), x.options());
  const int64_t cols = x.size(-1);
  check(api.ak_softmax_fwd(x.data_ptr(), y.data_ptr(), x.numel() / cols, cols, cols, cols, code_of(x.scalar_type()),
                           stream_of(x)), "ak_softmax_fwd");
  return y;
}

// ---------------------------------------------------------------------------
// Cross-entropy over logits
// ---------------------------------------------------------------------------
bool ce_args(const Tensor& x, const Tensor& t) {
  return x.dim() == 2 && x.is_contiguous() && x.size(0) > 0 && x.size(1) > 0 && code_of(x.scalar_type()) >= 0 &&
         t.scalar_type() == at::kLong && t.is_contiguous() && t.numel() == x.size(0);
}

const int64_t* i64p(const Tensor& t) { return static_cast<const int64_t*>(t.data_ptr()); }

// Whether the running backward frees the graph as it goes, so that nothing it
// has saved is asked for again (a captured backward may be replayed).
bool last_backward(const Tensor& t) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  const auto s = c10::hip::getCurrentHIPStream(t.get_device()).stream();
  return !torch::autograd::get_current_graph_task_keep_graph() &&
         hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone;
}

struct CrossEntropy : torch::autograd::Function<CrossEntropy> {
  // need: a gradient will be asked for; own: nobody but the graph holds what it
  // saves. lse_out: the row statistics, which have no gradient and are no output
  // of the node (compiled autograd takes no C++ node with one that is marked so).
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& t, double softcap, int64_t ignore,
                        double smoothing, bool fused, double zw, bool need, bool own, Tensor* lse_out) {
    const int64_t n = x.size(0), v = x.size(1);
    const int code = code_of(x.scalar_type());
    void* s = stream_of(x);
    Tensor loss = f32_like(x, {}), lse = f32_like(x, {n});
    // [max(1, #counted rows), its reciprocal], losses, and (tiny) row maxima and sums
    Tensor rest = f32_like(x, {2 + (fused ? 1 : 3) * n});
    float* denom = f32p(rest);
    float *losses = denom + 2, *mx = fused ? nullptr : losses + n, *sm = fused ? nullptr : mx + n;
    Tensor grad;
    if (need && fused) {
      check(api.ak_ce_count_valid(i64p(t), n, ignore, denom, s), "ak_ce_count_valid");
      grad = at::empty(x.sizes(), x.options());
    }
    check(api.ak_ce_fwd(x.data_ptr(), i64p(t), losses, f32p(lse), mx, sm, ptr(grad), n, v, v, v, (float)softcap, ignore,
                        (float)smoothing, 1.0f, (float)zw, grad.defined() ? denom + 1 : nullptr, code, s), "ak_ce_fwd");
    check(api.ak_ce_mean(losses, f32p(lse), i64p(t), n, ignore, (float)zw, f32p(loss), nullptr, s), "ak_ce_mean");
    *lse_out = lse;
    if (need) {
      if (fused) ctx->save_for_backward({grad});
      else ctx->save_for_backward({x, t, rest});
      ctx->saved_data["p"] = std::vector<double>{softcap, smoothing, zw};
      ctx->saved_data["i"] = std::vector<int64_t>{ignore, fused, own};
    }
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto p = ctx->saved_data["p"].toDoubleVector();
    const auto i = ctx->saved_data["i"].toIntVector();
    const auto saved = ctx->get_saved_variables();
    Tensor up = g[0].detach().to(at::kFloat);
    variable_list out(10);
    if (i[1]) {
      // The saved gradient carries 1 / #counted rows already. The upstream
      // gradient scales it in place where this backward is the graph's last: 1
      // (a plain loss.backward()) then costs a scalar read, where the product
      // is a pass over the gradient (4096 x 32768 bf16: 96 us).
      Tensor grad = saved[0];
      if (i[2] && grad.is_contiguous() && last_backward(grad)) {
        check(api.ak_scale_inplace(grad.data_ptr(), grad.numel(), f32p(up), code_of(grad.scalar_type()), stream_of(grad)),
              "ak_scale_inplace");
      } else {
        grad = grad * up.to(grad.scalar_type());
      }
      out[0] = grad;
    } else {
      Tensor x = saved[0].contiguous(), t = saved_as(saved[1], at::kLong), rest = saved_as(saved[2], at::kFloat);
      const int64_t n = x.size(0), v = x.size(1);
      float* denom = f32p(rest);
      float* mx = denom + 2 + n;
      check(api.ak_ce_count_valid(i64p(t), n, i[0], denom, stream_of(x)), "ak_ce_count_valid");
      Tensor scale = up * rest.select(0, 1);
      Tensor grad = at::empty(x.sizes(), x.options());
      check(api.ak_ce_bwd_tiny(x.data_ptr(), i64p(t), mx, mx + n, grad.data_ptr(), n, v, v, v, (float)p[0], i[0], (float)p[1],
                               1.0f, (float)p[2], f32p(scale), code_of(x.scalar_type()), stream_of(x)), "ak_ce_bwd_tiny");
      out[0] = grad;
    }
    return out;
  }
};

Pair ce_full(const Tensor& x, const Tensor& t, double softcap, int64_t ignore, double smoothing, bool fused, double zw,
             bool own) {
  if (!ours(x, t) || !ce_args(x, t)) return std::nullopt;
  const bool need = records({&x});
  Tensor lse;
  const Tensor loss = CrossEntropy::apply(x, t, softcap, ignore, smoothing, fused, zw, need, own, &lse);
  return std::make_tuple(loss, lse);
}

// ---------------------------------------------------------------------------
// Diagonal scan
// ---------------------------------------------------------------------------
bool dense_f32(const Tensor& t) { return t.scalar_type() == at::kFloat && t.is_contiguous(); }

bool diag_args(const Tensor& dA, const Tensor& dBx, const Tensor& C, const Tensor& D, const Tensor& x) {
  return dA.dim() == 3 && dA.numel() > 0 && dense_f32(dA) && dense_f32(dBx) && dense_f32(C) && dense_f32(D) && dense_f32(x) &&
         dBx.sizes() == dA.sizes() && C.sizes() == dA.sizes() && x.sizes() == dA.sizes() && D.dim() == 1 && D.numel() == dA.size(2);
}

Tensor run_diag(const Tensor& dA, const Tensor& dBx, const Tensor& C, const Tensor& D, const Tensor& x) {
  Tensor y = at::empty(dA.sizes(), dA.options());
  check(api.ak_diag_scan_fwd(f32p(dA), f32p(dBx), f32p(C), f32p(D), f32p(x), f32p(y), dA.size(0), dA.size(1), dA.size(2),
                             stream_of(dA)), "ak_diag_scan_fwd");
  return y;
}

struct DiagScan : torch::autograd::Function<DiagScan> {
  static Tensor forward(AutogradContext* ctx, const Tensor& dA, const Tensor& dBx, const Tensor& C, const Tensor& D,
                        const Tensor& x) {
    ctx->save_for_backward({dA, dBx, C, D, x});
    return run_diag(dA, dBx, C, D, x);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    if (!hip_backward) return by_formula("selective_scan", {s[0], s[1], s[2], s[3], s[4], g[0]}, 0.0);
    variable_list in;
    for (const Tensor& t : s) in.push_back(saved_as(t, at::kFloat));
    Tensor gy = g[0].to(at::kFloat).contiguous();
    variable_list out;
    for (const Tensor& t : in) out.push_back(at::empty(t.sizes(), t.options()));
    const int64_t b = in[0].size(0), l = in[0].size(1), d = in[0].size(2);
    const size_t bytes = api.ak_diag_scan_bwd_workspace_bytes(b, d);
    Tensor ws = bytes_like(gy, bytes);
    check(api.ak_diag_scan_bwd(f32p(in[0]), f32p(in[1]), f32p(in[2]), f32p(in[3]), f32p(in[4]), f32p(gy), f32p(out[0]),
                               f32p(out[1]), f32p(out[2]), f32p(out[3]), f32p(out[4]), ws.data_ptr(), bytes, b, l, d,
                               stream_of(gy)), "ak_diag_scan_bwd");
    return out;
  }
};

Maybe diag_scan(const Tensor& dA, const Tensor& dBx, const Tensor& C, const Tensor& D, const Tensor& x) {
  if (!ours(dA, dBx, C, D, x) || !diag_args(dA, dBx, C, D, x)) return std::nullopt;
  return run_diag(dA, dBx, C, D, x);
}

Maybe diag_scan_op(const Tensor& dA, const Tensor& dBx, const Tensor& C, const Tensor& D, const Tensor& x) {
  if (!records({&dA, &dBx, &C, &D, &x})) return diag_scan(dA, dBx, C, D, x);
  if (!ours(dA, dBx, C, D, x) || !diag_args(dA, dBx, C, D, x)) return std::nullopt;
  return DiagScan::apply(dA, dBx, C, D, x);
}

// ---------------------------------------------------------------------------
// Mamba-1 selective scan (real A, input-dependent B / C)
// ---------------------------------------------------------------------------
constexpr int64_t kStep = 16;  // steps between the states that training keeps

bool last_dense(const Tensor& t) { return t.stride(-1) == 1; }

struct ScanDims {
  int64_t b, d, l, n, g;
};

bool scan_args(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C, const Maybe& D,
               const Maybe& z, const Maybe& bias, ScanDims& k) {
  if (u.dim() != 3 || A.dim() != 2 || u.numel() == 0 || code_of(u.scalar_type()) < 0) return false;
  k = {u.size(0), u.size(1), u.size(2), A.size(1), B.dim() == 4 ? B.size(1) : 1};
  const auto half = [&](const Tensor& t) { return t.scalar_type() == u.scalar_type() || t.scalar_type() == at::kFloat; };
  const auto vec = [&](const Maybe& t) { return !t || (dense_f32(*t) && t->dim() == 1 && t->numel() == k.d); };
  const auto bc = [&](const Tensor& t) {
    if (t.dim() == 3) return t.size(0) == k.b && t.size(1) == k.n && t.size(2) == k.l;
    return t.dim() == 4 && t.size(0) == k.b && t.size(1) > 0 && k.d % t.size(1) == 0 && t.size(2) == k.n && t.size(3) == k.l;
  };
  return k.n > 0 && last_dense(u) && delta.sizes() == u.sizes() && last_dense(delta) && half(delta) && A.size(0) == k.d &&
         A.scalar_type() == at::kFloat && A.stride(1) == 1 && bc(B) && C.sizes() == B.sizes() && half(B) &&
         C.scalar_type() == B.scalar_type() && last_dense(B) && last_dense(C) && vec(D) && vec(bias) &&
         (!z || (z->sizes() == u.sizes() && z->scalar_type() == u.scalar_type() && last_dense(*z)));
}

struct BcStride {
  int64_t b, g, n;
};
BcStride bc_stride(const Tensor& t) {
  if (t.dim() == 4) return {t.stride(0), t.stride(1), t.stride(2)};
  return {t.stride(0), 0, t.stride(1)};
}

void run_scan(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C, const Tensor& D,
              const Tensor& z, const Tensor& bias, bool softplus, const ScanDims& k, const Tensor& out, const Tensor& last,
              const Tensor& prez, const Tensor& ckpt) {
  const BcStride sb = bc_stride(B), sc = bc_stride(C);
  const size_t bytes = api.ak_selective_scan_fwd_workspace_bytes(k.b, k.d, k.l, k.n, k.g, 0);
  const Tensor ws = bytes ? bytes_like(u, bytes) : Tensor();
  check(api.ak_selective_scan_fwd_ws(
            u.data_ptr(), delta.data_ptr(), f32p(A), B.data_ptr(), C.data_ptr(), f32p(D), ptr(z), f32p(bias), out.data_ptr(),
            f32p(last), ptr(prez), nullptr, f32p(ckpt), k.b, k.d, k.l, k.n, k.g, u.stride(0), u.stride(1), delta.stride(0),
            delta.stride(1), A.stride(0), sb.b, sb.g, sb.n, sc.b, sc.g, sc.n, z.defined() ? z.stride(0) : 0,
            z.defined() ? z.stride(1) : 0, out.stride(0), out.stride(1), softplus, 0, code_of(u.scalar_type()),
            code_of(delta.scalar_type()), code_of(B.scalar_type()), AK_DTYPE_F32, ptr(ws), bytes, stream_of(u)), "ak_selective_scan_fwd");
}

struct SelectiveScan : torch::autograd::Function<SelectiveScan> {
  // last_out: takes the last state where it is wanted (no output of the node, as in CrossEntropy)
  static Tensor forward(AutogradContext* ctx, const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B,
                        const Tensor& C, const Maybe& D_, const Maybe& z_, const Maybe& bias_, bool softplus,
                        Tensor* last_out, bool keep) {
    const Tensor D = D_.value_or(Tensor()), z = z_.value_or(Tensor()), bias = bias_.value_or(Tensor());
    const ScanDims k{u.size(0), u.size(1), u.size(2), A.size(1), B.dim() == 4 ? B.size(1) : 1};
    Tensor out = at::empty(u.sizes(), u.options()), last, prez, ckpt;
    if (last_out) last = *last_out = f32_like(u, {k.b, k.d, k.n});
    if (keep) {
      if (z.defined()) prez = at::empty(u.sizes(), u.options());
      ckpt = f32_like(u, {k.b, (k.l + kStep - 1) / kStep, k.d, k.n});
    }
    run_scan(u, delta, A, B, C, D, z, bias, softplus, k, out, last, prez, ckpt);
    ctx->save_for_backward({u, delta, A, B, C, D, z, bias, ckpt, prez});
    ctx->saved_data["softplus"] = softplus;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const bool softplus = ctx->saved_data["softplus"].toBool();
    // the kernels take rows at any pitch; saved-tensor hooks may hand back another layout or type
    const auto rows = [](const Tensor& t) { return !t.defined() || last_dense(t) ? t : t.contiguous(); };
    const Tensor u = rows(s[0]), delta = rows(s[1]), B = rows(s[3]), C = rows(s[4].to(B.scalar_type()));
    const Tensor A = rows(s[2].to(at::kFloat)), z = s[6].defined() ? rows(s[6].to(u.scalar_type())) : s[6];
    const Tensor D = saved_as(s[5], at::kFloat), bias = saved_as(s[7], at::kFloat), ckpt = saved_as(s[8], at::kFloat);
    const Tensor prez = saved_as(s[9], u.scalar_type());
    Tensor dout = rows(grads[0].to(u.scalar_type()));
    const ScanDims k{u.size(0), u.size(1), u.size(2), A.size(1), B.dim() == 4 ? B.size(1) : 1};
    Tensor du = at::empty(u.sizes(), u.options()), ddelta = at::empty(u.sizes(), delta.options());
    Tensor dA = at::empty(A.sizes(), A.options()), dB = at::empty(B.sizes(), B.options()), dC = at::empty(C.sizes(), C.options());
    Tensor dD, dz, dbias;
    if (D.defined()) dD = at::empty(D.sizes(), D.options());
    if (z.defined()) dz = at::empty(z.sizes(), z.options());
    if (bias.defined()) dbias = at::empty(bias.sizes(), bias.options());
    const size_t bytes = api.ak_selective_scan_bwd_workspace_bytes(k.b, k.d, k.l, k.n, k.g, 0);
    Tensor ws = bytes_like(u, bytes);
    const BcStride sb = bc_stride(B), sc = bc_stride(C);
    check(api.ak_selective_scan_bwd(
              u.data_ptr(), delta.data_ptr(), f32p(A), B.data_ptr(), C.data_ptr(), f32p(D), ptr(z), f32p(bias), dout.data_ptr(),
              du.data_ptr(), ddelta.data_ptr(), f32p(dA), dB.data_ptr(), dC.data_ptr(), f32p(dD), ptr(dz), f32p(dbias), f32p(ckpt),
              ptr(prez), ws.data_ptr(), bytes, k.b, k.d, k.l, k.n, k.g, u.stride(0), u.stride(1), delta.stride(0), delta.stride(1),
              A.stride(0), sb.b, sb.g, sb.n, sc.b, sc.g, sc.n, z.defined() ? z.stride(0) : 0, z.defined() ? z.stride(1) : 0,
              dout.stride(0), dout.stride(1), softplus, 0, code_of(u.scalar_type()), code_of(delta.scalar_type()),
              code_of(B.scalar_type()), AK_DTYPE_F32, stream_of(u)), "ak_selective_scan_bwd");
    return {du, ddelta, dA, dB, dC, dD, dz, dbias, Tensor(), Tensor(), Tensor()};
  }
};

// (out, last state or nothing). save: training keeps its states; max_bytes: up to this size.
std::optional<std::vector<Tensor>> selective_scan(const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B,
                                                  const Tensor& C, const Maybe& D, const Maybe& z, const Maybe& bias,
                                                  bool softplus, bool want_last, bool save, double max_bytes) {
  ScanDims k;
  if (!ours(u, delta, A, B, C) || !ours_if(D, u) || !ours_if(z, u) || !ours_if(bias, u) ||
      !scan_args(u, delta, A, B, C, D, z, bias, k))
    return std::nullopt;
  const Tensor d = D.value_or(Tensor()), zz = z.value_or(Tensor()), bb = bias.value_or(Tensor());
  Tensor out, last;
  if (records({&u, &delta, &A, &B, &C, &d, &zz, &bb})) {
    const double bytes = 4.0 * k.b * k.d * k.n * ((k.l + kStep - 1) / kStep);
    out = SelectiveScan::apply(u, delta, A, B, C, D, z, bias, softplus, want_last ? &last : nullptr, save && bytes <= max_bytes);
  } else {
    out = at::empty(u.sizes(), u.options());
    if (want_last) last = f32_like(u, {k.b, k.d, k.n});
    run_scan(u, delta, A, B, C, d, zz, bb, softplus, k, out, last, Tensor(), Tensor());
  }
  std::vector<Tensor> r{out};
  if (want_last) r.push_back(last);
  return r;
}

// ---------------------------------------------------------------------------
// lm-head + cross-entropy
// ---------------------------------------------------------------------------
bool at16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
bool dense16(const Tensor& t) { return t.dim() == 2 && t.is_contiguous() && at16(t); }
Tensor realigned(const Tensor& t) { return at16(t) ? t : t.clone(); }

struct LmHead : torch::autograd::Function<LmHead> {
  static Tensor forward(AutogradContext* ctx, const Tensor& h, const Tensor& w, const Tensor& t, int64_t ignore, double cap,
                        double smoothing) {
    const int64_t n = h.size(0), d = h.size(1), v = w.size(0);
    Tensor loss = f32_like(h, {}), lse = f32_like(h, {n});
    const size_t bytes = api.ak_lmhead_ce_workspace_bytes(n, v);
    Tensor ws = bytes_like(h, bytes);
    Tensor denom = f32_like(h, {1});
    check(api.ak_lmhead_ce_fwd_denom(h.data_ptr(), w.data_ptr(), i64p(t), f32p(loss), f32p(lse), nullptr, nullptr, f32p(denom),
                                     ws.data_ptr(), bytes, n, v, d, d, d, ignore, (float)cap, (float)smoothing,
                                     code_of(h.scalar_type()), stream_of(h)), "ak_lmhead_ce_fwd");
    ctx->save_for_backward({h, w, t, lse, denom});
    ctx->saved_data["ignore"] = ignore;
    ctx->saved_data["p"] = std::vector<double>{cap, smoothing};
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const int64_t ignore = ctx->saved_data["ignore"].toInt();
    const auto p = ctx->saved_data["p"].toDoubleVector();
    const bool need_h = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1);
    // (saved-tensor hooks may hand back any address too, where the tile kernels need 16-byte rows)
    const Tensor h = realigned(s[0].contiguous()), w = realigned(saved_as(s[1], h.scalar_type()));
    const Tensor t = saved_as(s[2], at::kLong);
    const Tensor lse = saved_as(s[3], at::kFloat), denom = saved_as(s[4], at::kFloat);  // denom: max(1, #counted rows)
    const Tensor up = g[0].detach().to(at::kFloat).contiguous();
    const int64_t n = h.size(0), d = h.size(1), v = w.size(0);
    const int code = code_of(h.scalar_type());
    void* st = stream_of(h);
    // dlogits: the pitch covers whole 64-column K blocks and stays off powers
    // of two, whose rows would all start in the same memory channels
    const int64_t padded = (v + 63) / 64 * 64;
    const int64_t pitch = (padded & (padded - 1)) == 0 ? padded + 64 : padded;
    Tensor gl = at::empty({n, pitch}, h.options());
    check(api.ak_lmhead_ce_bwd_range(h.data_ptr(), w.data_ptr(), i64p(t), f32p(lse), f32p(up), f32p(denom), gl.data_ptr(), pitch,
                                     n, v, 0, v, d, d, d, ignore, (float)p[0], (float)p[1], code, st), "ak_lmhead_ce_bwd_range");
    const size_t bytes = api.ak_lmhead_grad_workspace_bytes(n, v, d);
    Tensor ws = bytes ? bytes_like(h, bytes) : Tensor();
    Tensor gh, gw;
    if (need_w) {
      gw = at::empty(w.sizes(), w.options());
      check(api.ak_lmhead_grad_weight(gl.data_ptr(), pitch, h.data_ptr(), d, gw.data_ptr(), d, n, v, d, 0, ptr(ws), bytes, code,
                                      st), "ak_lmhead_grad_weight");
    }
    if (need_h) {
      // the K padding meets weight rows that load as zeros, but NaN x 0 is NaN
      if (padded > v) gl.slice(1, v, padded).zero_();
      gh = at::empty(h.sizes(), h.options());
      check(api.ak_lmhead_grad_hidden(gl.data_ptr(), pitch, w.data_ptr(), d, gh.data_ptr(), d, n, v, d, 0, ptr(ws), bytes, code,
                                      st), "ak_lmhead_grad_hidden");
    }
    return {gh, gw, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// budget: the bytes of dlogits that the backward may hold at once.
Maybe lmhead_ce(const Tensor& h, const Tensor& w, const Tensor& t, int64_t ignore, double cap, double smoothing, double budget) {
  if (!ours(h, w, t) || !dense16(h) || !dense16(w) || h.scalar_type() != w.scalar_type() || h.size(0) == 0 || w.size(0) == 0 ||
      (h.scalar_type() != at::kHalf && h.scalar_type() != at::kBFloat16) || h.size(1) != w.size(1) || h.size(1) == 0 ||
      h.size(1) % 64 || t.scalar_type() != at::kLong || t.dim() != 1 || !t.is_contiguous() || t.size(0) != h.size(0))
    return std::nullopt;
  if (records({&h, &w}) && 2.0 * h.size(0) * ((w.size(0) + 255) / 256 * 256) > budget) return std::nullopt;  // vocab ranges
  return LmHead::apply(h, w, t, ignore, cap, smoothing);
}

}  // namespace

PYBIND11_MODULE(_host_ops, m) {
  using nogil = py::call_guard<py::gil_scoped_release>;
  m.def("init", &init);
  m.def("set_hip_backward", &set_hip_backward);
  m.def("set_formula", &set_formula);
  m.def("rmsnorm", &rmsnorm, nogil());
  m.def("add_rmsnorm", &add_rmsnorm, nogil());
  m.def("add_rmsnorm_dual", &add_rmsnorm_dual, nogil());
  m.def("rmsnorm_op", &rmsnorm_op, nogil());
  m.def("add_rmsnorm_op", &add_rmsnorm_op, nogil());
  m.def("softmax", &softmax, nogil());
  m.def("ce_full", &ce_full, nogil());
  m.def("diag_scan", &diag_scan, nogil());
  m.def("diag_scan_op", &diag_scan_op, nogil());
  m.def("selective_scan", &selective_scan, nogil());
  m.def("lmhead_ce", &lmhead_ce, nogil());
}
