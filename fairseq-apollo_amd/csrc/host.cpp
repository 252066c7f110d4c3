// Host side of the calls whose device work is shorter than their Python would be: allocation of the results, argument
// checks and the C ABI call in native code, one Python call per composite step.  Tensors in, tensors out; the launch
// stream's raw handle comes from the caller (ops._stream).  No device code and no state in here.
#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <Python.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mega_hip.h"

namespace {

using at::Tensor;

// One Python argument, read while the interpreter lock is held.  Tensors stay where they are: the caller's frame holds
// them until the call returns.
struct Value {
  enum Kind { kOther, kNone, kTensor, kInt, kFloat } kind = kOther;
  const Tensor* t = nullptr;
  int64_t i = 0;
  double d = 0.0;
};
// false: a Python error is set
bool read(PyObject* o, Value* v) {
  if (o == Py_None) {
    v->kind = Value::kNone;
  } else if (THPVariable_Check(o)) {
    v->kind = Value::kTensor;
    v->t = &THPVariable_Unpack(o);
  } else if (!PyFloat_Check(o) && PyIndex_Check(o)) {
    PyObject* n = PyNumber_Index(o);
    if (!n) return false;
    v->i = PyLong_AsLongLong(n);
    Py_DECREF(n);
    if (v->i == -1 && PyErr_Occurred()) return false;
    v->kind = Value::kInt;
    v->d = (double)v->i;
  } else if (PyNumber_Check(o)) {
    v->d = PyFloat_AsDouble(o);
    if (v->d == -1.0 && PyErr_Occurred()) return false;
    v->kind = Value::kFloat;
  }
  return true;
}

struct Args {
  const Value* a;
  Py_ssize_t n;
  const char* who;
  void want(Py_ssize_t k) const {
    if (n != k) throw std::runtime_error(std::string(who) + ": " + std::to_string(k) + " arguments expected");
  }
  [[noreturn]] void bad(int i, const char* what) const {
    throw std::runtime_error(std::string(who) + ": argument " + std::to_string(i) + " must be " + what);
  }
  bool none(int i) const { return a[i].kind == Value::kNone; }
  const Tensor& t(int i) const {
    if (a[i].kind != Value::kTensor) bad(i, "a tensor");
    return *a[i].t;
  }
  // a contiguous tensor of the given type, size and device
  const Tensor& t(int i, at::ScalarType dt, int64_t numel, const at::Device& dev) const {
    const Tensor& x = t(i);
    if (x.scalar_type() != dt || x.numel() != numel || x.device() != dev || !x.is_contiguous())
      throw std::runtime_error(std::string(who) + ": argument " + std::to_string(i) + " must be a contiguous tensor of " +
                               std::to_string(numel) + " elements of " + at::toString(dt) + " on the input's device");
    return x;
  }
  const void* p(int i, at::ScalarType dt, int64_t numel, const at::Device& dev) const { return t(i, dt, numel, dev).data_ptr(); }
  const void* opt(int i, at::ScalarType dt, int64_t numel, const at::Device& dev) const {
    return none(i) ? nullptr : p(i, dt, numel, dev);
  }
  // a weight matrix [rows, cols]
  const void* mat(int i, at::ScalarType dt, int64_t rows, int64_t cols, const at::Device& dev) const {
    shape(i, {rows, cols});
    return p(i, dt, rows * cols, dev);
  }
  // the kernels take every size from one operand: the others must have it
  void shape(int i, at::IntArrayRef sizes) const {
    if (!none(i) && t(i).sizes() != sizes) {
      std::string want;
      for (int64_t s : sizes) want += (want.empty() ? "" : ", ") + std::to_string(s);
      throw std::runtime_error(std::string(who) + ": argument " + std::to_string(i) + " must be [" + want + "]");
    }
  }
  double d(int i) const {
    if (a[i].kind != Value::kInt && a[i].kind != Value::kFloat) bad(i, "a number");
    return a[i].d;
  }
  int64_t i64(int i) const {
    if (a[i].kind != Value::kInt) bad(i, "an integer");
    return a[i].i;
  }
  bool flag(int i) const { return i64(i) != 0; }
  void* stream(int i) const { return (void*)(uintptr_t)i64(i); }
};

int dtype_code(const Tensor& x) {
  switch (x.scalar_type()) {
    case at::kFloat: return MEGA_F32;
    case at::kBFloat16: return MEGA_BF16;
    case at::kHalf: return MEGA_F16;
    default: throw std::runtime_error("unsupported activation dtype (float32, bfloat16, float16)");
  }
}

void check(int rc, const char* who) {
  if (rc != 0) throw std::runtime_error(std::string(who) + ": " + mega_last_error() + " (code " + std::to_string(rc) + ")");
}

// what an entry returns: one tensor, or a tuple of them (undefined: None)
struct Result {
  Tensor t[10];
  int n = 0;
  bool one = false;
};
Result wrap(Tensor t) {
  Result r;
  r.t[0] = std::move(t);
  r.n = 1;
  r.one = true;
  return r;
}
template <size_t N>
Result tuple(Tensor (&ts)[N]) {
  static_assert(N <= 10, "Result holds ten tensors");
  Result r;
  for (size_t i = 0; i < N; ++i) r.t[i] = std::move(ts[i]);
  r.n = (int)N;
  return r;
}

Tensor empty(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dt) {
  return at::empty(sizes, like.options().dtype(dt));
}

// (x [B, 1, D], mask [B] bytes | None, count, mean, var, h | None, keys | None, values | None, keep, norm gamma, norm beta,
//  norm eps, groups, p, q, gamma, omega, v weight, v bias, mx weight, mx bias, h weight, gamma, beta, move act,
//  move weight | None, move eps, cis, heads, stream) -> (out [B, 1, D], count, mean, var, h', keys' | None, values' | None)
Result token_gated_attention(const Args& A) {
  A.want(30);
  const Tensor& x = A.t(0);
  const at::Device dev = x.device();
  const at::ScalarType T = x.scalar_type();
  if (x.dim() != 3 || x.size(1) != 1 || !x.is_contiguous() || !x.is_cuda())
    throw std::runtime_error("token_gated_attention: x must be a contiguous [B, 1, D] device tensor");
  const int64_t B = x.size(0), D = x.size(2);
  const Tensor &p = A.t(13), &hw = A.t(21), &gm = A.t(22);
  if (p.dim() != 2 || hw.dim() != 2 || gm.dim() != 2) throw std::runtime_error("token_gated_attention: weight shapes");
  const int64_t N = p.size(1), hidden = hw.size(1), S = gm.size(1), G = A.i64(12), Nh = A.i64(28);
  const int64_t W = 2 * D + S + hidden;
  if (G <= 0 || D % G || Nh <= 0) throw std::runtime_error("token_gated_attention: groups / heads");
  int64_t n = 0;
  if (!A.none(6)) {
    const Tensor& k = A.t(6);
    if (k.dim() != 3 || k.size(0) != B || k.size(2) != S) throw std::runtime_error("token_gated_attention: cached keys must be [B, n, S]");
    n = k.size(1);
  }
  MegaTokenAttention a = {};
  a.dtype = dtype_code(x); a.B = B; a.D = D; a.S = S; a.hidden = hidden; a.heads = Nh; a.groups = G; a.states = N;
  a.context = n;
  a.x = x.data_ptr();
  a.mask = (const uint8_t*)A.opt(1, at::kByte, B, dev);
  a.prev_count = (const int64_t*)A.p(2, at::kLong, B, dev);
  a.prev_mean = (const float*)A.p(3, at::kFloat, B * G, dev);
  a.prev_var = (const float*)A.p(4, at::kFloat, B * G, dev);
  a.h_in = (const float*)A.opt(5, at::kComplexFloat, B * D * N, dev);
  if (n > 0) {                       // keys straight from a prompt are a strided half of the q / k map's result
    const Tensor& k = A.t(6);
    if (k.scalar_type() != T || k.device() != dev || k.stride(2) != 1)
      throw std::runtime_error("token_gated_attention: cached keys must be rows of the activation type");
    a.k_old = k.data_ptr();
    a.k_row = k.stride(1);
    a.k_batch = k.stride(0);
  }
  a.v_old = A.opt(7, T, B * n * hidden, dev);
  const bool keep = A.flag(8);
  a.norm_gamma = (const float*)A.p(9, at::kFloat, D, dev);
  a.norm_beta = (const float*)A.p(10, at::kFloat, D, dev);
  a.norm_eps = A.d(11);
  a.p = (const float*)A.p(13, at::kFloat, D * N, dev);
  a.q = (const float*)A.p(14, at::kFloat, D * N * 2, dev);
  a.ema_gamma = (const float*)A.p(15, at::kFloat, D * N * 2, dev);
  a.omega = (const float*)A.p(16, at::kFloat, D, dev);
  a.v_weight = A.mat(17, T, hidden, D, dev);
  a.v_bias = A.p(18, T, hidden, dev);
  a.mx_weight = A.mat(19, T, W, D, dev);
  a.mx_bias = A.p(20, T, W, dev);
  a.h_weight = A.mat(21, T, D, hidden, dev);
  a.gamma = A.mat(22, T, 2, S, dev);
  a.beta = A.mat(23, T, 2, S, dev);
  a.move_act = A.i64(24);
  a.move_norm_weight = A.opt(25, T, D, dev);
  a.move_norm_eps = A.d(26);
  const Tensor& cis = A.t(27);
  if (cis.scalar_type() != at::kComplexFloat || cis.dim() != 2 || cis.size(0) <= n || cis.size(1) * 2 * Nh != S ||
      !cis.is_contiguous() || cis.device() != dev)
    throw std::runtime_error("token_gated_attention: the rotation table must cover the new position");
  a.cis = (const float*)cis.data_ptr();
  Tensor r[7];
  r[0] = at::empty({B, 1, D}, x.options());
  r[1] = empty({B}, x, at::kLong);
  r[2] = empty({B, G}, x, at::kFloat);
  r[3] = empty({B, G}, x, at::kFloat);
  r[4] = empty({B, D, N}, x, at::kComplexFloat);
  if (keep) {
    r[5] = at::empty({B, n + 1, S}, x.options());
    r[6] = at::empty({B, n + 1, hidden}, x.options());
    a.k_out = r[5].data_ptr();
    a.v_out = r[6].data_ptr();
  }
  a.out = r[0].data_ptr();
  a.count = (int64_t*)r[1].data_ptr();
  a.mean = (float*)r[2].data_ptr();
  a.var = (float*)r[3].data_ptr();
  a.h_out = (float*)r[4].data_ptr();
  const int64_t nws = (int64_t)mega_token_attention_workspace_bytes(B, n, D, S, hidden, Nh);
  Tensor ws = empty({nws}, x, at::kByte);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = nws;
  check(mega_token_gated_attention(&a, A.stream(29)), A.who);
  return tuple(r);
}

// (x [B, 1, D], norm kind, norm weight | None, norm bias | None, eps, fc1 weight, fc1 bias, fc2 weight, layer scale | None,
//  stream) -> x + scale fc2(silu(fc1(norm(x))))
Result token_ffn(const Args& A) {
  A.want(10);
  const Tensor& x = A.t(0);
  const at::Device dev = x.device();
  const at::ScalarType T = x.scalar_type();
  const Tensor& w1 = A.t(5);
  if (x.dim() != 3 || x.size(1) != 1 || !x.is_contiguous() || !x.is_cuda() || w1.dim() != 2)
    throw std::runtime_error("token_ffn: x must be a contiguous [B, 1, D] device tensor");
  const int64_t B = x.size(0), D = x.size(2), H = w1.size(0);
  Tensor hid = at::empty({B, H}, x.options()), rows = at::empty({B, D}, x.options()), out[1] = {at::empty({B, 1, D}, x.options())};
  MegaTokenLinear f1 = {}, f2 = {};
  f1.prologue = (int)A.i64(1);
  f1.scratch = rows.data_ptr();
  f1.norm_weight = A.opt(2, T, D, dev);
  f1.norm_bias = A.opt(3, T, D, dev);
  f1.eps = (float)A.d(4);
  f1.weight = A.mat(5, T, H, D, dev);
  f1.bias = A.p(6, T, H, dev);
  f1.x = x.data_ptr(); f1.x_stride = D; f1.out = hid.data_ptr(); f1.out_stride = H; f1.N = H; f1.K = D;
  f1.epilogue = MEGA_TOKEN_SILU;
  f2.weight = A.mat(7, T, D, H, dev);
  f2.scale = A.opt(8, T, D, dev);
  f2.x = hid.data_ptr(); f2.x_stride = H; f2.out = out[0].data_ptr(); f2.out_stride = D; f2.N = D; f2.K = H;
  f2.epilogue = MEGA_TOKEN_RESIDUAL; f2.residual = x.data_ptr(); f2.residual_stride = D;
  const int dt = dtype_code(x);
  void* s = A.stream(9);
  check(mega_token_linear(&f1, dt, B, s), A.who);
  check(mega_token_linear(&f2, dt, B, s), A.who);
  return wrap(out[0]);
}

// (tokens [B, 1], table [V, D], scale | None, pad | None) -> (x [B, 1, D], mask [B, 1] bool | None): torch's own lookup, which
// knows what to do with an index outside the table
Result token_embed(const Args& A) {
  A.want(4);
  const Tensor& tok = A.t(0);
  Tensor r[2] = {at::embedding(A.t(1), tok), Tensor()};
  if (!A.none(2)) r[0].mul_(A.d(2));
  if (!A.none(3)) r[1] = tok.eq(A.i64(3));
  return tuple(r);
}

// (x [B, 1, D], mask [B] bytes | None, count, mean, var, gamma, beta, eps, groups, stream) -> (xn, count, mean, var)
Result token_norm(const Args& A) {
  A.want(10);
  const Tensor& x = A.t(0);
  const at::Device dev = x.device();
  if (x.dim() != 3 || x.size(1) != 1 || !x.is_contiguous() || !x.is_cuda())
    throw std::runtime_error("token_norm: x must be a contiguous [B, 1, D] device tensor");
  const int64_t B = x.size(0), D = x.size(2), G = A.i64(8);
  Tensor r[4] = {at::empty({B, 1, D}, x.options()), empty({B}, x, at::kLong), empty({B, G}, x, at::kFloat),
                 empty({B, G}, x, at::kFloat)};
  check(mega_norm_token(x.data_ptr(), r[0].data_ptr(), dtype_code(x), (const uint8_t*)A.opt(1, at::kByte, B, dev),
                        (const int64_t*)A.p(2, at::kLong, B, dev), (const float*)A.p(3, at::kFloat, B * G, dev),
                        (const float*)A.p(4, at::kFloat, B * G, dev), (int64_t*)r[1].data_ptr(), (float*)r[2].data_ptr(),
                        (float*)r[3].data_ptr(), (const float*)A.p(5, at::kFloat, D, dev),
                        (const float*)A.p(6, at::kFloat, D, dev), A.d(7), B, D, G, A.stream(9)),
        A.who);
  return tuple(r);
}

// (x [B, 1, K], weight [N, K], bias | None, stream) -> [B, 1, N]
Result token_linear(const Args& A) {
  A.want(4);
  const Tensor &x = A.t(0), &w = A.t(1);
  if (x.dim() != 3 || x.size(1) != 1 || !x.is_contiguous() || !x.is_cuda() || w.dim() != 2)
    throw std::runtime_error("token_linear: x must be a contiguous [B, 1, K] device tensor");
  const int64_t B = x.size(0), K = x.size(2), N = w.size(0);
  Tensor out = at::empty({B, 1, N}, x.options());
  MegaTokenLinear f = {};
  f.weight = A.mat(1, x.scalar_type(), N, K, x.device());
  f.bias = A.opt(2, x.scalar_type(), N, x.device());
  f.x = x.data_ptr(); f.x_stride = K; f.out = out.data_ptr(); f.out_stride = N; f.N = N; f.K = K;
  check(mega_token_linear(&f, dtype_code(x), B, A.stream(3)), A.who);
  return wrap(out);
}

// (x [B, D] in any shape, count, next count, mean, var, norm weight, norm bias, eps, p, q, gamma, complex, omega, h, groups,
//  stream) -> (xn, y) in x's shape; count / mean / var / h are the step's own buffers, updated in place (next count takes the new count)
Result norm_ema_step(const Args& A) {
  A.want(16);
  Tensor x = A.t(0).detach().contiguous();
  const at::Device dev = x.device();
  const Tensor& p = A.t(8);
  if (!x.is_cuda() || p.dim() != 2) throw std::runtime_error("norm_ema_step: x must be a device tensor");
  const int64_t B = A.t(1).numel(), D = p.size(0), N = p.size(1), G = A.i64(14);
  if (x.numel() != B * D) throw std::runtime_error("norm_ema_step: x must hold [B, D] values, the streams' and channels' of the state");
  Tensor r[2] = {at::empty_like(x), at::empty_like(x)};
  float* mean = (float*)A.p(3, at::kFloat, B * G, dev);
  float* var = (float*)A.p(4, at::kFloat, B * G, dev);
  float* h = (float*)A.p(13, at::kFloat, B * D * N * 2, dev);
  check(mega_norm_ema_step(x.data_ptr(), r[0].data_ptr(), r[1].data_ptr(), dtype_code(x), (const int64_t*)A.p(1, at::kLong, B, dev),
                           mean, var, (int64_t*)A.p(2, at::kLong, B, dev), mean, var, (const float*)A.p(5, at::kFloat, D, dev),
                           (const float*)A.p(6, at::kFloat, D, dev), A.d(7), (const float*)A.p(8, at::kFloat, D * N, dev),
                           (const float*)A.p(9, at::kFloat, D * N * 2, dev), (const float*)A.p(10, at::kFloat, D * N * 2, dev),
                           (int)A.i64(11), (const float*)A.p(12, at::kFloat, D, dev), h, h, B, D, G, N, A.stream(15)),
        A.who);
  return tuple(r);
}

// ---- training: TimestepNorm -> moving average, and the moving average alone, from the stored parameters
struct EmaIn {
  MegaEmaParams e = {};
  at::Device dev = at::kCPU;
};
// alpha, delta, third, gamma, omega at a[i..i+4]
EmaIn ema_params(const Args& A, int i, bool is_complex, bool two_sided) {
  EmaIn r;
  const Tensor& alpha = A.t(i);
  if (alpha.dim() < 2 || !alpha.is_cuda()) throw std::runtime_error(std::string(A.who) + ": alpha must be [K, N, 1] on the device");
  r.dev = alpha.device();
  const at::ScalarType T = alpha.scalar_type();
  MegaEmaParams& e = r.e;
  e.dtype = dtype_code(alpha);
  e.is_complex = is_complex;
  e.K = alpha.size(0);
  e.N = alpha.size(1);
  e.D = two_sided ? e.K / 2 : e.K;
  e.alpha = A.p(i, T, e.K * e.N, r.dev);
  e.delta = A.p(i + 1, T, e.K * e.N, r.dev);
  e.third = A.p(i + 2, T, is_complex ? e.K : e.K * e.N, r.dev);
  e.gamma = A.p(i + 3, T, e.K * e.N * (is_complex ? 2 : 1), r.dev);
  e.omega = A.p(i + 4, T, e.D, r.dev);
  return r;
}

// (alpha, delta, third, gamma, omega, is_complex, two_sided, shift, activations (a tensor of their type),
//  weight | None, bias, prior mean, prior log-variance, prior count, batch, stream)
//   -> (p, q, gamma, omega, image, norm gamma, norm beta, prior mean [B, G], prior var [B, G], count [B])
Result train_prepare(const Args& A) {
  A.want(16);
  const bool cplx = A.flag(5), two = A.flag(6);
  const EmaIn in = ema_params(A, 0, cplx, two);
  const MegaEmaParams& e = in.e;
  const Tensor& like = A.t(0);
  Tensor r[10];
  r[0] = empty({e.K, e.N}, like, at::kFloat);
  r[1] = empty({e.K, e.N, 2}, like, at::kFloat);
  r[2] = empty({e.K, e.N, 2}, like, at::kFloat);
  r[3] = empty({e.D}, like, at::kFloat);
  const int64_t nimg = (int64_t)mega_ema_image_bytes(e.D, e.N, two ? 1 : 0);
  if (nimg <= 0) throw std::runtime_error("train_prepare: more than 16 states have no operand image");
  r[4] = empty({nimg}, like, at::kByte);
  MegaNormParams n = {};
  const bool norm = !A.none(9);
  if (norm) {
    const Tensor &w = A.t(9), &pm = A.t(11);
    n.dtype = dtype_code(w);
    n.prior_dtype = dtype_code(pm);
    n.H = w.numel();
    n.G = pm.numel();
    n.B = A.i64(14);
    n.weight = A.p(9, w.scalar_type(), n.H, in.dev);
    n.bias = A.p(10, w.scalar_type(), n.H, in.dev);
    n.prior_mean = A.p(11, pm.scalar_type(), n.G, in.dev);
    n.prior_logv = A.p(12, pm.scalar_type(), n.G, in.dev);
    n.prior_count = (const int64_t*)A.p(13, at::kLong, 1, in.dev);
    r[5] = empty({n.H}, like, at::kFloat);
    r[6] = empty({n.H}, like, at::kFloat);
    r[7] = empty({n.B, n.G}, like, at::kFloat);
    r[8] = empty({n.B, n.G}, like, at::kFloat);
    r[9] = empty({n.B}, like, at::kLong);
    n.gamma = (float*)r[5].data_ptr();
    n.beta = (float*)r[6].data_ptr();
    n.prev_mean = (float*)r[7].data_ptr();
    n.prev_var = (float*)r[8].data_ptr();
    n.prev_count = (int64_t*)r[9].data_ptr();
  }
  check(mega_train_prepare(&e, norm ? &n : nullptr, dtype_code(A.t(8)), A.flag(7), (float*)r[0].data_ptr(),
                           (float*)r[1].data_ptr(), (float*)r[2].data_ptr(), (float*)r[3].data_ptr(), r[4].data_ptr(), nimg,
                           A.stream(15)),
        A.who);
  return tuple(r);
}

// (x [B, L, D], mask bytes | None, count, mean, var, norm gamma, norm beta, eps, p, q, gamma, omega, image, is_complex,
//  y in x's layout, norm workspace, stream) -> (xn, y [B, D, L], count, cummean, cumrstd)
Result norm_move_forward(const Args& A) {
  A.want(17);
  const Tensor& x = A.t(0);
  const at::Device dev = x.device();
  if (x.dim() != 3 || !x.is_contiguous() || !x.is_cuda()) throw std::runtime_error("norm_move_forward: x must be a contiguous [B, L, D] device tensor");
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2), N = A.t(8).size(1), G = A.t(3).numel() / (B > 0 ? B : 1);
  if (G <= 0 || D % G) throw std::runtime_error("norm_move_forward: groups");
  const bool input = A.flag(14);
  Tensor r[5] = {at::empty_like(x), input ? at::empty({B, L, D}, x.options()).transpose(1, 2) : at::empty({B, D, L}, x.options()),
                 empty({B}, x, at::kLong), empty({B, L, G}, x, at::kFloat), empty({B, L, G}, x, at::kFloat)};
  Tensor stats = empty({2, B, G}, x, at::kFloat);
  const int64_t nsc = (int64_t)mega_norm_ema_fwd_scratch_bytes(B, L, D, G, N);
  Tensor sc = empty({nsc}, x, at::kByte);
  const Tensor &ws = A.t(15), &img = A.t(12);
  check(mega_norm_ema_fwd_train(
            x.data_ptr(), r[0].data_ptr(), r[1].data_ptr(), dtype_code(x), r[1].stride(0), r[1].stride(1), r[1].stride(2),
            (const int64_t*)A.p(2, at::kLong, B, dev), (const float*)A.p(3, at::kFloat, B * G, dev),
            (const float*)A.p(4, at::kFloat, B * G, dev), (const float*)A.p(5, at::kFloat, D, dev),
            (const float*)A.p(6, at::kFloat, D, dev), (const uint8_t*)A.opt(1, at::kByte, B * L, dev), A.d(7),
            (int64_t*)r[2].data_ptr(), (float*)stats.data_ptr(), (float*)stats.data_ptr() + B * G, (float*)r[3].data_ptr(),
            (float*)r[4].data_ptr(), (const float*)A.p(8, at::kFloat, D * N, dev), (const float*)A.p(9, at::kFloat, D * N * 2, dev),
            (const float*)A.p(10, at::kFloat, D * N * 2, dev), A.flag(13), (const float*)A.p(11, at::kFloat, D, dev), nullptr,
            nullptr, B, L, D, G, N, img.data_ptr(), ws.data_ptr(), ws.numel(), sc.data_ptr(), nsc, A.stream(16)),
        A.who);
  return tuple(r);
}

// The gradient with respect to the moving average's input, [B, L, D] memory: the layer run backwards in time on the
// output's gradient (which already lies time-major)
Tensor adjoint(const Tensor& g, const float* p, const float* q, const float* gamma, const float* omega, const void* image,
               int cplx, int two, int shift, int64_t N, void* stream, const char* who) {
  const int64_t B = g.size(0), L = g.size(1), D = g.size(2), es = g.element_size();
  Tensor dx = at::empty_like(g);
  const int64_t nws = (int64_t)mega_ema_fwd_workspace_bytes(B, D, N, L, two, 0);
  Tensor ws = empty({nws}, g, at::kByte);
  const int64_t back = (L - 1) * D * es;
  check(mega_ema_fwd((const char*)g.data_ptr() + back, (char*)dx.data_ptr() + back, dtype_code(g), L * D, 1, -D, L * D, 1, -D,
                     p, q, gamma, cplx, omega, nullptr, nullptr, nullptr, B, D, N, L, two, 0, shift, image, ws.data_ptr(), nws,
                     stream),
        who);
  return dx;
}

struct ParamGrads {
  Tensor r[5];
  MegaEmaParamGrads g;
  explicit ParamGrads(const Args& A, int i) {
    void** out[5] = {&g.alpha, &g.delta, &g.third, &g.gamma, &g.omega};
    for (int k = 0; k < 5; ++k) {
      r[k] = at::empty_like(A.t(i + k));
      *out[k] = r[k].data_ptr();
    }
  }
};

// (xn gradient | None, y gradient [B, D, L], x, xn, mask bytes | None, prior mean, count, cummean, cumrstd, norm gamma, p, q,
//  gamma, omega, image, weight, prior log-variance, prior needs gradients, alpha, delta, third, gamma, omega, is_complex,
//  stream) -> (x gradient, weight, bias, prior mean | None, prior log-variance | None, alpha, delta, third, gamma, omega)
Result norm_move_backward(const Args& A) {
  A.want(25);
  const Tensor &x = A.t(2), &xn = A.t(3);
  const at::Device dev = x.device();
  const at::ScalarType T = x.scalar_type();
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2), N = A.t(10).size(1);
  if (B <= 0 || L <= 0) throw std::runtime_error("norm_move_backward: empty input");
  const int64_t G = A.t(5).numel() / B;
  const int cplx = A.flag(23), dt = dtype_code(x);
  void* s = A.stream(24);
  const EmaIn in = ema_params(A, 18, cplx, false);
  Tensor g = A.t(1).detach();
  if (g.scalar_type() != T) g = g.to(T);
  if (g.dim() != 3 || g.size(0) != B || g.size(1) != D || g.size(2) != L) throw std::runtime_error("norm_move_backward: y gradient must be [B, D, L]");
  g = g.transpose(1, 2).contiguous();                          // free when it already lies time-major
  const float *p = (const float*)A.p(10, at::kFloat, D * N, dev), *q = (const float*)A.p(11, at::kFloat, D * N * 2, dev);
  // The padding mask plays no part here: xn is zero at padding, so the sums over time see the masked input as it is, and
  // what flows back to a padded token ends in the norm, which hands no gradient through it.
  Tensor dxn = adjoint(g, p, q, (const float*)A.p(12, at::kFloat, D * N * 2, dev), (const float*)A.p(13, at::kFloat, D, dev),
                       A.t(14).data_ptr(), cplx, 0, 1, N, s, A.who);
  Tensor sums = empty({B * D * N * 4 + B * D}, x, at::kFloat);
  float *sp = (float*)sums.data_ptr(), *dyx = sp + B * D * N * 4;
  check(mega_ema_param_sums(g.data_ptr(), xn.data_ptr(), dt, L * D, 1, D, L * D, 1, D, q, nullptr, B, D, N, L, 0, 0, sp, dyx, s), A.who);
  // the norm's backward pass on the sum of both gradients of xn
  Tensor other;
  if (!A.none(0)) {
    other = A.t(0).detach();
    if (other.scalar_type() != T) other = other.to(T);
    other = other.contiguous();
    if (!mega_timestep_norm_bwd_adds(dt, B, L, D, G) || (uintptr_t)other.data_ptr() % 16 || (uintptr_t)x.data_ptr() % 16) {
      dxn.add_(other);
      other = Tensor();
    }
  }
  Tensor dx = at::empty_like(x), ng = empty({2, D}, x, at::kFloat), pg = empty({2, B, G}, x, at::kFloat);
  const int64_t nws = (int64_t)mega_timestep_norm_bwd_workspace_bytes(dt, B, L, D, G);
  Tensor ws = empty({nws}, x, at::kByte);
  float *dg = (float*)ng.data_ptr(), *dpm = (float*)pg.data_ptr();
  check(mega_group_timestep_norm_bwd_add(
            dxn.data_ptr(), other.defined() ? other.data_ptr() : nullptr, nullptr, nullptr, x.data_ptr(), dt,
            (const float*)A.p(5, at::kFloat, B * G, dev), (const int64_t*)A.p(6, at::kLong, B, dev), nullptr,
            (const float*)A.p(7, at::kFloat, B * L * G, dev), (const float*)A.p(8, at::kFloat, B * L * G, dev),
            (const float*)A.p(9, at::kFloat, D, dev), (const uint8_t*)A.opt(4, at::kByte, B * L, dev), B, L, D, G, dx.data_ptr(),
            dpm, dpm + B * G, dg, dg + D, ws.data_ptr(), nws, s),
        A.who);
  const Tensor &w = A.t(15), &pl = A.t(16);
  Tensor r[10];
  MegaNormParamGrads n = {};
  n.gamma_grad = dg; n.beta_grad = dg + D; n.mean_grad = dpm; n.var_grad = dpm + B * G;
  n.prior_logv = pl.data_ptr();
  n.dtype = dtype_code(w); n.prior_dtype = dtype_code(pl); n.H = D; n.G = G;
  r[0] = dx;
  r[1] = at::empty_like(w);
  r[2] = at::empty_like(w);
  n.weight = r[1].data_ptr();
  n.bias = r[2].data_ptr();
  if (A.flag(17)) {
    r[3] = at::empty_like(pl);
    r[4] = at::empty_like(pl);
    n.prior_mean = r[3].data_ptr();
    n.prior_logv_grad = r[4].data_ptr();
  }
  ParamGrads eg(A, 18);
  check(mega_ema_param_finish(sp, dyx, &in.e, B, &eg.g, &n, s), A.who);
  for (int k = 0; k < 5; ++k) r[5 + k] = eg.r[k];
  return tuple(r);
}

// (y gradient, x, both with any strides of [B, D, L], mask bytes | None, q, alpha, delta, third, gamma, omega, is_complex,
//  two_sided, shift, stream) -> gradients of (alpha, delta, third, gamma, omega)
Result ema_param_backward(const Args& A) {
  A.want(13);
  const Tensor &g = A.t(0), &x = A.t(1);
  const int cplx = A.flag(9), two = A.flag(10), shift = A.flag(11);
  void* s = A.stream(12);
  const EmaIn in = ema_params(A, 4, cplx, two);
  const int64_t B = x.size(0), D = x.size(1), L = x.size(2), N = in.e.N;
  if (x.dim() != 3 || g.sizes() != x.sizes() || g.scalar_type() != x.scalar_type() || D != in.e.D || B <= 0 || L <= 0 ||
      x.device() != in.dev || g.device() != in.dev)
    throw std::runtime_error("ema_param_backward: shapes");
  const float* q = (const float*)A.p(3, at::kFloat, in.e.K * N * 2, in.dev);
  const uint8_t* mask = (const uint8_t*)A.opt(2, at::kByte, B * L, in.dev);
  const int halves = two ? 2 : 1;
  Tensor sums = empty({halves * (B * D * N * 4 + B * D)}, x, at::kFloat);
  float* dyx = (float*)sums.data_ptr() + halves * B * D * N * 4;
  for (int h = 0; h < halves; ++h)
    check(mega_ema_param_sums(g.data_ptr(), x.data_ptr(), dtype_code(x), g.stride(0), g.stride(1), g.stride(2), x.stride(0),
                              x.stride(1), x.stride(2), q + h * D * N * 2, mask, B, D, N, L, h, h && shift ? 1 : 0,
                              (float*)sums.data_ptr() + h * B * D * N * 4, dyx + h * B * D, s),
          A.who);
  ParamGrads eg(A, 4);
  check(mega_ema_param_finish((const float*)sums.data_ptr(), dyx, &in.e, B, &eg.g, nullptr, s), A.who);
  return tuple(eg.r);
}

// ---- training: the layer around its norm, moving average and attention, forwards and backwards in few calls.  The
// products (by size, order and type) and what lies between them run in libmega_hip.
// Activations and weights share one type.
Tensor rows2(const Tensor& t) { return t.reshape({-1, t.size(-1)}); }

// A matrix whose elements follow each other along one of its axes: that axis and the other one's stride
struct Matrix {
  int64_t ld;
  bool first;                                   // the contiguous axis is the first one
};
bool matrix(const Tensor& t, Matrix* m) {
  if (t.dim() != 2) return false;
  const int64_t r = t.size(0), c = t.size(1), sr = t.stride(0), sc = t.stride(1);
  if ((sc == 1 || c == 1) && (sr >= c || r == 1)) return *m = {r == 1 ? c : sr, false}, true;
  if ((sr == 1 || r == 1) && (sc >= r || c == 1)) return *m = {c == 1 ? r : sc, true}, true;
  return false;
}

// a [M, K] b [K, N] (+ bias) (+ residual) on the library's own products, silu of it with the value before in `pre`; `out`
// (optional) receives the result and may be the residual.  Rows of whole 16-byte pieces, at the sizes where mega_gemm_f32 and
// mega_gemm16 are worth a call (their own rules).  False: not of this kind.
bool product(const Tensor& a, const Tensor& b, const Tensor& bias, const Tensor& residual, bool silu, Tensor* pre, Tensor* out,
             void* s, const char* who) {
  Matrix ma, mb, mr = {0, false};
  const at::ScalarType dt = a.scalar_type();
  const bool wide = dt == at::kFloat;
  if ((!wide && dt != at::kBFloat16 && dt != at::kHalf) || b.scalar_type() != dt || !a.is_cuda() || a.device() != b.device() ||
      !matrix(a, &ma) || !matrix(b, &mb) || a.size(1) != b.size(0) || a.numel() == 0 || b.numel() == 0)
    return false;
  const int64_t M = a.size(0), K = a.size(1), N = b.size(1);
  auto fits = [&](const Tensor& t) { return t.scalar_type() == dt && t.device() == a.device(); };
  if (bias.defined() && (!fits(bias) || bias.numel() != N || !bias.is_contiguous())) return false;
  if (residual.defined() && (!fits(residual) || !matrix(residual, &mr) || mr.first || residual.size(0) != M || residual.size(1) != N)) return false;
  auto on16 = [](const Tensor& t) { return !t.defined() || (uintptr_t)t.data_ptr() % 16 == 0; };
  const int64_t vec = 16 / a.element_size(), far = ((int64_t)1 << 32) / a.element_size() / 128;
  if (!(wide ? mega_gemm_f32_pays : silu ? mega_gemm16_silu_pays : mega_gemm16_pays)(M, N, K, ma.first, !mb.first) || ma.ld % vec || mb.ld % vec || (ma.first ? M : K) % vec ||
      (mb.first ? K : N) % vec || ma.ld >= far || mb.ld >= far)
    return false;
  if (!wide && (N % vec || mr.ld % vec || !on16(bias) || !on16(residual) || !on16(*out))) return false;
  // a gradient that starts off 16 bytes gives what the same gradient on 16 bytes gives: from a copy of it
  auto aligned = [&](const Tensor& t, Matrix* m) {
    if (on16(t)) return t;
    const Tensor c = (m->first ? t.t() : t).clone(at::MemoryFormat::Contiguous);
    m->ld = c.size(1);
    return m->first ? c.t() : c;
  };
  const Tensor a16 = aligned(a, &ma), b16 = aligned(b, &mb);
  if (!out->defined()) *out = at::empty({M, N}, a.options());
  if (pre) *pre = at::empty({M, N}, a.options());
  MegaGemm g = {};
  g.a = a16.data_ptr(); g.b = b16.data_ptr(); g.c = out->data_ptr();
  g.bias = bias.defined() ? bias.data_ptr() : nullptr;
  g.residual = residual.defined() ? residual.data_ptr() : nullptr;
  g.pre = pre ? pre->data_ptr() : nullptr;
  g.lda = ma.ld; g.a_kmajor = ma.first;
  g.ldb = mb.ld; g.b_kmajor = !mb.first;
  g.ldc = N; g.ldr = mr.ld;
  g.M = M; g.N = N; g.K = K; g.batch = g.inner = 1;
  g.silu = silu; g.alpha = 1.f;
  const int64_t nws = (int64_t)(wide ? mega_gemm_workspace_bytes(M, N, K, 1) : mega_gemm16_workspace_bytes(M, N, K));
  Tensor ws;
  if (nws) ws = at::empty({nws}, a.options().dtype(at::kByte));
  void* w = nws ? ws.data_ptr() : nullptr;
  check(wide ? mega_gemm_f32(&g, w, (size_t)nws, s) : mega_gemm16(&g, dtype_code(a), w, (size_t)nws, s), who);
  return true;
}

Tensor mm(const Tensor& a, const Tensor& b, void* s, const char* who) {
  Tensor out;
  return product(a, b, Tensor(), Tensor(), false, nullptr, &out, s, who) ? out : at::mm(a, b);
}
// a b + c, c a row of biases or a whole matrix
Tensor addmm(const Tensor& c, const Tensor& a, const Tensor& b, void* s, const char* who) {
  Tensor out;
  const bool row = c.dim() == 1;
  return product(a, b, row ? c : Tensor(), row ? Tensor() : c, false, nullptr, &out, s, who) ? out : at::addmm(c, a, b);
}
// silu(a b + bias) and the value before
std::pair<Tensor, Tensor> silu_mm(const Tensor& bias, const Tensor& a, const Tensor& b, void* s, const char* who);

const void* ptr_or_null(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
Tensor opt_t(const Args& A, int i) { return A.none(i) ? Tensor() : A.t(i); }
void same_type(const Args& A, std::initializer_list<int> at, const Tensor& x) {
  for (int i : at)
    if (!A.none(i) && (A.t(i).scalar_type() != x.scalar_type() || A.t(i).device() != x.device() || !A.t(i).is_contiguous()))
      throw std::runtime_error(std::string(A.who) + ": argument " + std::to_string(i) + " must be contiguous, of the activations' type and on their device");
}

// A gradient as the row kernels read it: of x's type, contiguous, on 16 bytes (autograd also hands out views that start
// anywhere in a buffer, behind a concatenation for instance)
Tensor rows16(const Tensor& t, const Tensor& x) {
  Tensor r = t.to(x.scalar_type()).contiguous();
  return (uintptr_t)r.data_ptr() % 16 ? r.clone() : r;
}

// a row norm's parameters hold one value per column: the kernels read (and in the backward pass write) that many
void norm_width(const Tensor& x, const Tensor& w, const Tensor& b, const char* who) {
  for (const Tensor* p : {&w, &b})
    if (p->defined() && (p->dim() != 1 || p->numel() != x.size(-1)))
      throw std::runtime_error(std::string(who) + ": norm parameters of " + std::to_string(p->numel()) + " values on rows of " +
                               std::to_string(x.size(-1)));
}

Tensor row_norm(const Tensor& x, const Tensor& w, const Tensor& b, int kind, double eps, void* s, const char* who) {
  norm_width(x, w, b, who);
  Tensor y = at::empty_like(x);
  if (x.numel()) check(mega_row_norm_fwd(x.data_ptr(), x.size(-1), ptr_or_null(w), ptr_or_null(b), y.data_ptr(), dtype_code(x), kind, x.numel() / x.size(-1), x.size(-1), eps, s), who);
  return y;
}

// (dx, dw, db); dw / db undefined where there is no parameter
std::tuple<Tensor, Tensor, Tensor> row_norm_back(const Tensor& dy, const Tensor& x, const Tensor& w, const Tensor& b,
                                                 const Tensor& add, int kind, double eps, void* s, const char* who) {
  norm_width(x, w, b, who);
  if (dy.numel() != x.numel() || dy.size(-1) != x.size(-1)) throw std::runtime_error(std::string(who) + ": the gradient must have the rows' shape");
  Tensor dx = at::empty_like(x), dw, db;
  if (w.defined()) dw = at::empty_like(w);
  if (b.defined()) db = at::empty_like(b);
  const int64_t D = x.size(-1), T = x.numel() / D;
  const int64_t nws = (int64_t)mega_row_norm_bwd_workspace_bytes(T, D);
  Tensor ws = empty({nws}, x, at::kByte);
  check(mega_row_norm_bwd(dy.data_ptr(), x.data_ptr(), D, ptr_or_null(w), ptr_or_null(add), dx.data_ptr(),
                          dw.defined() ? dw.data_ptr() : nullptr, db.defined() ? db.data_ptr() : nullptr, dtype_code(x), kind, T,
                          D, eps, ws.data_ptr(), nws, s),
        who);
  return {dx, dw, db};
}

// dx = dy silu'(x) and its sum over the tokens (x undefined: the sum of dy alone)
std::pair<Tensor, Tensor> sum_rows(const Tensor& dy, const Tensor& x, void* s, const char* who) {
  const int64_t W = dy.size(-1), T = dy.numel() / W;
  Tensor dx, out = at::empty({W}, dy.options());
  if (x.defined()) dx = at::empty_like(x);
  const int64_t nws = (int64_t)mega_sum_rows_workspace_bytes(dtype_code(dy), T, W);
  Tensor ws = empty({nws}, dy, at::kByte);
  check(mega_sum_rows(dy.data_ptr(), W, ptr_or_null(x), dx.defined() ? dx.data_ptr() : nullptr, dtype_code(dy), T, W, out.data_ptr(),
                      ws.data_ptr(), nws, s),
        who);
  return {dx, out};
}

Tensor silu(const Tensor& x, void* s, const char* who) {
  Tensor y = at::empty_like(x);
  check(mega_silu_fwd(x.data_ptr(), y.data_ptr(), dtype_code(x), x.numel(), s), who);
  return y;
}

std::pair<Tensor, Tensor> silu_mm(const Tensor& bias, const Tensor& a, const Tensor& b, void* s, const char* who) {
  Tensor pre, out;
  if (!product(a, b, bias, Tensor(), true, &pre, &out, s, who)) {
    pre = at::addmm(bias, a, b);
    out = silu(pre, s, who);
  }
  return {pre, out};
}

// a linear layer outside training: (x [.., K] contiguous, weight [N, K], bias | None, residual [.., N] | None, silu,
// the residual's memory may take the result, stream) -> [.., N], or None where the product is left to the GEMM library
Result linear_own(const Args& A) {
  A.want(7);
  const Tensor &x = A.t(0), &w = A.t(1);
  same_type(A, {0, 1, 2, 3}, x);
  auto sizes = x.sizes().vec();
  if (w.dim() != 2 || sizes.back() != w.size(1)) throw std::runtime_error("linear_own: rows of another width than the weight's");
  sizes.back() = w.size(0);
  A.shape(2, {w.size(0)});
  A.shape(3, sizes);
  const Tensor r = A.none(3) ? Tensor() : rows2(A.t(3));
  Tensor out = !A.none(3) && A.flag(5) ? r : Tensor();
  if (!product(rows2(x), w.t(), opt_t(A, 2), r, A.flag(4), nullptr, &out, A.stream(6), A.who)) return wrap(Tensor());
  return wrap(out.view(sizes));
}

// Batched fp32 products over the positions and heads of attention: (a, b, c, M, N, K, batch, heads, a's row stride, batch
// stride, head stride, reduction along its rows, the same four of b, c's row, batch and head stride, causal, alpha, a's rows
// are padded to whole pieces of four, stream)
Result attention_product(const Args& A) {
  A.want(23);
  MegaGemm g = {};
  const Tensor& a = A.t(0);
  same_type(A, {0, 1, 2}, a);
  if (a.scalar_type() != at::kFloat || !a.is_cuda()) throw std::runtime_error("attention_product: fp32 device tensors expected");
  g.a = a.data_ptr(); g.b = A.t(1).data_ptr(); g.c = A.t(2).data_ptr();
  g.M = A.i64(3); g.N = A.i64(4); g.K = A.i64(5); g.batch = A.i64(6) * A.i64(7); g.inner = A.i64(7);
  g.lda = A.i64(8); g.sa = A.i64(9); g.sai = A.i64(10); g.a_kmajor = A.flag(11);
  g.ldb = A.i64(12); g.sb = A.i64(13); g.sbi = A.i64(14); g.b_kmajor = A.flag(15);
  g.ldc = A.i64(16); g.sc = A.i64(17); g.sci = A.i64(18);
  g.causal = (int)A.i64(19); g.alpha = (float)A.d(20); g.a_padded = A.flag(21);
  auto inside = [&](const Tensor& t, int64_t rows, int64_t cols, int64_t ld, int64_t sb, int64_t si) {
    return ld >= 0 && sb >= 0 && si >= 0 &&
           (A.i64(6) - 1) * sb + (g.inner - 1) * si + (rows - 1) * ld + cols <= t.numel();
  };
  if (g.a_padded && g.lda % 4) throw std::runtime_error("attention_product: padded rows are whole pieces");
  if (g.M < 1 || g.N < 1 || g.K < 1 || A.i64(6) < 1 || g.inner < 1 ||
      !inside(a, g.a_kmajor ? g.K : g.M, g.a_padded ? g.lda : g.a_kmajor ? g.M : g.K, g.lda, g.sa, g.sai) ||
      !inside(A.t(1), g.b_kmajor ? g.K : g.N, g.b_kmajor ? g.N : g.K, g.ldb, g.sb, g.sbi) || !inside(A.t(2), g.M, g.N, g.ldc, g.sc, g.sci))
    throw std::runtime_error("attention_product: sizes beyond an operand");
  const int64_t nws = (int64_t)mega_gemm_workspace_bytes(g.M, g.N, g.K, g.batch);
  Tensor ws;
  if (nws) ws = at::empty({nws}, a.options().dtype(at::kByte));
  check(mega_gemm_f32(&g, nws ? ws.data_ptr() : nullptr, (size_t)nws, A.stream(22)), A.who);
  return Result();
}

// Operations are only being run, not looked at: no tracing, function transform or dispatch mode, which see torch's own
// operations and nothing that happens in here.
bool eager() {
  return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer) &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::dispatch_mode_enabled();
}

// Values of its own in memory and no forward-mode tangent beside them.
bool plain(const Tensor& t) { return !at::isTensorSubclassLike(t) && !t._fw_grad(0).defined(); }

// (x, kind, weight | None, bias | None, eps, stream) -> y
Result row_norm_forward(const Args& A) {
  A.want(6);
  same_type(A, {0, 2, 3}, A.t(0));
  return wrap(row_norm(A.t(0), opt_t(A, 2), opt_t(A, 3), (int)A.i64(1), A.d(4), A.stream(5), A.who));
}

// (dy, x, kind, weight | None, bias | None, eps, stream) -> (dx, dw, db)
Result row_norm_backward(const Args& A) {
  A.want(7);
  same_type(A, {1, 3, 4}, A.t(1));
  auto [dx, dw, db] = row_norm_back(rows16(A.t(0), A.t(1)), A.t(1), opt_t(A, 3), opt_t(A, 4), Tensor(), (int)A.i64(2), A.d(5), A.stream(6), A.who);
  Tensor r[3] = {dx, dw, db};
  return tuple(r);
}

// x + fc2(silu(fc1(norm(x)))): (x, kind, norm weight | None, norm bias | None, eps, fc1 weight, fc1 bias, fc2 weight, stream)
//   -> (out, n, pre, h)
Result ffn_forward(const Args& A) {
  A.want(9);
  const Tensor& x = A.t(0);
  same_type(A, {0, 2, 3, 5, 6, 7}, x);
  void* s = A.stream(8);
  Tensor n = row_norm(x, opt_t(A, 2), opt_t(A, 3), (int)A.i64(1), A.d(4), s, A.who);
  auto [pre, h] = silu_mm(A.t(6), rows2(n), A.t(5).t(), s, A.who);
  Tensor out = addmm(rows2(x), h, A.t(7).t(), s, A.who).view(x.sizes());
  Tensor r[4] = {out, n, pre, h};
  return tuple(r);
}

// Which gradients a backward pass is asked for (bit i: input i of the autograd function): the products behind the others are
// left out, and their places in the result are None.
struct Wanted {
  int64_t bits;
  bool any(int64_t m) const { return (bits & m) != 0; }
  bool operator()(int i) const { return any((int64_t)1 << i); }
};

// (dout, x, n, pre, h, kind, norm weight | None, norm bias | None, eps, fc1 weight, fc2 weight, stream, wanted)
//   -> (dx, d norm weight, d norm bias, d fc1 weight, d fc1 bias, d fc2 weight)
Result ffn_backward(const Args& A) {
  A.want(13);
  const Wanted want{A.i64(12)};               // x, norm weight, norm bias, fc1 weight, fc1 bias, fc2 weight
  const Tensor &x = A.t(1), &n = A.t(2), &pre = A.t(3), &h = A.t(4);
  const Tensor dout = rows16(A.t(0), x);
  same_type(A, {1, 2, 3, 4, 6, 7, 9, 10}, x);
  void* s = A.stream(11);
  A.shape(4, pre.sizes());
  if (dout.numel() != x.numel() || n.numel() != x.numel() || pre.numel() != x.numel() / x.size(-1) * A.t(10).size(1))
    throw std::runtime_error("ffn_backward: gradients and saved operands of other sizes than the forward's");
  const Tensor d2 = rows2(dout);
  Tensor dx, dnw, dnb, dw1, db1, dw2;
  if (want(5)) dw2 = mm(d2.t(), h, s, A.who);
  if (want.any(0x1f)) {
    Tensor dpre;
    std::tie(dpre, db1) = sum_rows(mm(d2, A.t(10), s, A.who), pre, s, A.who);
    if (want(3)) dw1 = mm(dpre.t(), rows2(n), s, A.who);
    if (want.any(7))
      std::tie(dx, dnw, dnb) = row_norm_back(mm(dpre, A.t(9), s, A.who), x, opt_t(A, 6), opt_t(A, 7), dout, (int)A.i64(5), A.d(8), s, A.who);
  }
  Tensor r[6] = {dx, dnw, dnb, dw1, db1, dw2};
  return tuple(r);
}

// W2 (silu(W1 n) * W3 n) + residual: (n, residual | None, W1, W3, W2, stream) -> (out, a, b, g)
Result swiglu_forward(const Args& A) {
  A.want(6);
  const Tensor& n = A.t(0);
  same_type(A, {0, 1, 2, 3, 4}, n);
  void* s = A.stream(5);
  const Tensor n2 = rows2(n);
  A.shape(3, A.t(2).sizes());
  Tensor a = mm(n2, A.t(2).t(), s, A.who), b = mm(n2, A.t(3).t(), s, A.who), g = at::empty_like(a);
  check(mega_swiglu_fwd(a.data_ptr(), b.data_ptr(), g.data_ptr(), dtype_code(n), a.numel(), s), A.who);
  Tensor out = A.none(1) ? mm(g, A.t(4).t(), s, A.who) : addmm(rows2(A.t(1)), g, A.t(4).t(), s, A.who);
  auto sizes = n.sizes().vec();
  sizes.back() = A.t(4).size(0);
  Tensor r[4] = {out.view(sizes), a, b, g};
  return tuple(r);
}

// (dout, n, a, b, g, W1, W3, W2, stream, wanted) -> (dn, dW1, dW3, dW2)
Result swiglu_backward(const Args& A) {
  A.want(10);
  const Wanted want{A.i64(9)};                // n, residual, W1, W3, W2
  const Tensor &n = A.t(1), &a = A.t(2), &b = A.t(3), &g = A.t(4);
  same_type(A, {1, 2, 3, 4, 5, 6, 7}, n);
  void* s = A.stream(8);
  A.shape(3, a.sizes());
  A.shape(4, a.sizes());
  const Tensor d2 = rows2(A.t(0).to(n.scalar_type()).contiguous()), n2 = rows2(n);
  Tensor dn, dw1, dw3, dw2;
  if (want(4)) dw2 = mm(d2.t(), g, s, A.who);
  if (want.any(0xd)) {
    const Tensor dg = mm(d2, A.t(7), s, A.who);
    const Tensor da = at::empty_like(a), db = at::empty_like(b);
    check(mega_swiglu_bwd(dg.data_ptr(), a.data_ptr(), b.data_ptr(), da.data_ptr(), db.data_ptr(), dtype_code(n), a.numel(), s), A.who);
    if (want(2)) dw1 = mm(da.t(), n2, s, A.who);
    if (want(3)) dw3 = mm(db.t(), n2, s, A.who);
    if (want(0)) {                            // both branches into one gradient: no third pass to add them
      Tensor both = mm(da, A.t(5), s, A.who), out = both;
      if (!product(db, A.t(6), Tensor(), both, false, nullptr, &out, s, A.who)) both.addmm_(db, A.t(6));
      dn = both.view(n.sizes());
    }
  }
  Tensor r[4] = {dn, dw1, dw3, dw2};
  return tuple(r);
}

// The gated attention between its norm / moving average and the attention product.
// (xn [B, L, D], mx [B, D, L] view of time-major memory, v weight, v bias, mx weight, mx bias, gamma, beta, freqs, heads,
//  chunk, move act, move weight | None, move eps, stream) -> (vp, v, mx (time-major), act, base, q, k)
Result mix_forward(const Args& A) {
  A.want(15);
  const Tensor& xn = A.t(0);
  same_type(A, {0, 2, 3, 4, 5, 6, 7, 12}, xn);
  void* s = A.stream(14);
  const int dt = dtype_code(xn);
  const int64_t D = xn.size(2), S = A.t(6).size(1), E = A.t(2).size(0), heads = A.i64(9), chunk = A.i64(10);
  const int64_t T = xn.numel() / D, W = 2 * D + S + E;
  A.shape(2, {E, D});
  A.shape(4, {W, D});
  A.shape(6, {2, S});
  A.shape(7, {2, S});
  A.shape(12, {D});
  const Tensor mx = A.t(1).transpose(1, 2).contiguous();
  if (mx.scalar_type() != xn.scalar_type() || mx.sizes() != xn.sizes()) throw std::runtime_error("mix_forward: mx must be [B, D, L]");
  auto [vp, v] = silu_mm(A.t(3), rows2(xn), A.t(2).t(), s, A.who);
  const int act_kind = (int)A.i64(11);
  Tensor act = act_kind == MEGA_TOKEN_RMSNORM ? row_norm(mx, opt_t(A, 12), Tensor(), act_kind, A.d(13), s, A.who) : silu(mx, s, A.who);
  Tensor base = addmm(A.t(5), rows2(act), A.t(4).t(), s, A.who);
  Tensor q = at::empty({T, S}, xn.options()), k = at::empty({T, S}, xn.options());
  check(mega_gate_qk_fwd_raw((const char*)base.data_ptr() + D * xn.element_size(), W, A.t(6).data_ptr(), A.t(7).data_ptr(),
                             (const float*)A.p(8, at::kFloat, S / heads / 2, xn.device()), q.data_ptr(), k.data_ptr(), dt, T, S, heads,
                             chunk, 0, 1e-5, s),
        A.who);
  Tensor r[7] = {vp, v, mx, act, base, q, k};
  return tuple(r);
}

// (residual [B, L, D], base, attention [T, E], h weight, S, stream) -> (out, gated, hp)
Result mix_out_forward(const Args& A) {
  A.want(6);
  const Tensor &x = A.t(0), &base = A.t(1), &attn = A.t(2);
  same_type(A, {0, 1, 2, 3}, x);
  void* s = A.stream(5);
  const int dt = dtype_code(x);
  const int64_t D = x.size(2), E = attn.size(-1), S = A.i64(4), W = base.size(1), T = x.numel() / D, es = x.element_size();
  A.shape(1, {T, 2 * D + S + E});
  A.shape(3, {D, E});
  if (attn.numel() != T * E) throw std::runtime_error("mix_out_forward: attention must be [tokens, E]");
  const char* b = (const char*)base.data_ptr();
  Tensor gated = at::empty({T, E}, x.options());
  check(mega_gate_mul_fwd(attn.data_ptr(), E, b + (D + S) * es, W, gated.data_ptr(), dt, T, E, s), A.who);
  Tensor hp = mm(gated, A.t(3).t(), s, A.who);
  Tensor out = at::empty_like(x);
  check(mega_gate_out_fwd(x.data_ptr(), D, b, W, b + (D + S + E) * es, W, hp.data_ptr(), D, out.data_ptr(), dt, T, D, s), A.who);
  Tensor r[3] = {out, gated, hp};
  return tuple(r);
}

// (dout, residual, base, attention [T, E], gated, hp, h weight, S, stream, wanted) -> (d residual, d base (u, r, hx slots), d attention, d h weight)
Result mix_out_backward(const Args& A) {
  A.want(10);
  const Wanted want{A.i64(9)};                // residual, base, attention, h weight
  const Tensor &x = A.t(1), &base = A.t(2), &attn = A.t(3), &gated = A.t(4), &hp = A.t(5), &hw = A.t(6);
  same_type(A, {1, 2, 3, 4, 5, 6}, x);
  const Tensor dout = A.t(0).to(x.scalar_type()).contiguous();
  void* s = A.stream(8);
  const int dt = dtype_code(x);
  const int64_t D = x.size(2), E = attn.size(-1), S = A.i64(7), W = base.size(1), T = x.numel() / D, es = x.element_size();
  if (dout.numel() != x.numel() || attn.numel() != T * E) throw std::runtime_error("mix_out_backward: the gradient must have the residual's shape, attention [tokens, E]");
  A.shape(2, {T, 2 * D + S + E});
  A.shape(4, {T, E});
  A.shape(5, {T, D});
  A.shape(6, {D, E});
  const char* b = (const char*)base.data_ptr();
  Tensor dbase = at::empty_like(base), dres = at::empty_like(x);
  // Autograd holds the whole buffer as a gradient before mix_backward fills q's and k's slice: whoever looks at it
  // (anomaly detection, a hook on the node) must find no stale memory there.  8192 tokens x 512 columns in bf16: 4.6 us.
  dbase.narrow(1, D, S).zero_();
  char* db = (char*)dbase.data_ptr();
  check(mega_gate_out_bwd_strided(dout.data_ptr(), x.data_ptr(), D, b, W, b + (D + S + E) * es, W, hp.data_ptr(), D, dres.data_ptr(), db,
                                  W, db + (D + S + E) * es, W, dt, T, D, s),
        A.who);
  const Tensor dh = dbase.narrow(1, D + S + E, D);
  Tensor dattn, dhw;
  if (want(3)) dhw = mm(dh.t(), gated, s, A.who);
  if (want.any(6)) {
    const Tensor dgated = mm(dh, hw, s, A.who);
    dattn = at::empty_like(attn);
    check(mega_gate_mul_bwd_strided(dgated.data_ptr(), attn.data_ptr(), E, b + (D + S) * es, W, dattn.data_ptr(), db + (D + S) * es, W,
                                    dt, T, E, s),
          A.who);
  }
  Tensor r[4] = {dres, want(1) ? dbase : Tensor(), dattn, dhw};
  return tuple(r);
}

// (dq [T, S], dk, dv [T, E], dbase, xn, vp, mx, act, base, v weight, mx weight, gamma, freqs, heads, chunk, move act,
//  move weight | None, move eps, stream, wanted)
//   -> (d xn, d mx (time-major), d v weight, d v bias, d mx weight, d mx bias, d gamma, d beta, d move weight)
Result mix_backward(const Args& A) {
  A.want(20);
  const Wanted want{A.i64(19)};               // xn, mx, v weight, v bias, mx weight, mx bias, gamma, beta, freqs, move weight
  const Tensor &dbase = A.t(3), &xn = A.t(4), &vp = A.t(5), &mx = A.t(6), &act = A.t(7), &base = A.t(8);
  same_type(A, {3, 4, 5, 6, 7, 8, 9, 10, 11, 16}, xn);
  void* s = A.stream(18);
  const int dt = dtype_code(xn);
  const Tensor dq = rows16(A.t(0), xn), dk = rows16(A.t(1), xn), dv = rows16(A.t(2), xn);
  const int64_t D = xn.size(2), S = A.t(11).size(1), heads = A.i64(13), chunk = A.i64(14), T = xn.numel() / D;
  const int64_t W = base.size(1), es = xn.element_size(), E = vp.size(-1);
  if (dq.numel() != T * S || dk.numel() != T * S || dv.numel() != T * E || act.numel() != T * D || mx.numel() != T * D ||
      mx.size(-1) != D || act.size(-1) != D || W != 2 * D + S + E)
    throw std::runtime_error("mix_backward: gradients and saved operands of other sizes than the forward's");
  A.shape(3, {T, W});
  A.shape(5, {T, E});
  A.shape(8, {T, W});
  A.shape(9, {E, D});
  A.shape(10, {W, D});
  A.shape(11, {2, S});
  A.shape(16, {D});
  Tensor dgamma = at::empty_like(A.t(11)), dbeta = at::empty_like(A.t(11));
  {
    const int64_t nws = (int64_t)mega_gate_qk_bwd_workspace_bytes(T, S);
    Tensor ws = empty({nws}, xn, at::kByte);
    check(mega_gate_qk_bwd_raw(dq.data_ptr(), dk.data_ptr(), (const char*)base.data_ptr() + D * es, W, A.t(11).data_ptr(),
                               (const float*)A.p(12, at::kFloat, S / heads / 2, xn.device()), (char*)dbase.data_ptr() + D * es, W,
                               dgamma.data_ptr(), dbeta.data_ptr(), dt, T, S, heads, chunk, 0, 1e-5, ws.data_ptr(), nws, s),
          A.who);
  }
  Tensor dxn, dmx, dvw, dvb, dmxw, dmxb, dmw;
  if (want(4)) dmxw = mm(dbase.t(), rows2(act), s, A.who);
  if (want(5)) dmxb = sum_rows(dbase, Tensor(), s, A.who).second;
  if (want.any(0x202)) {
    const Tensor dact = mm(dbase, A.t(10), s, A.who).view(mx.sizes());
    const int act_kind = (int)A.i64(15);
    if (act_kind == MEGA_TOKEN_RMSNORM) {
      Tensor none;
      std::tie(dmx, dmw, none) = row_norm_back(dact, mx, opt_t(A, 16), Tensor(), Tensor(), act_kind, A.d(17), s, A.who);
    } else {
      dmx = at::empty_like(mx);
      check(mega_silu_bwd(dact.data_ptr(), mx.data_ptr(), dmx.data_ptr(), dt, mx.numel(), s), A.who);
    }
  }
  if (want.any(0xd)) {
    Tensor dvp;
    std::tie(dvp, dvb) = sum_rows(dv.view(vp.sizes()), vp, s, A.who);
    if (want(2)) dvw = mm(dvp.t(), rows2(xn), s, A.who);
    if (want(0)) dxn = mm(dvp, A.t(9), s, A.who).view(xn.sizes());
  }
  Tensor r[9] = {dxn, dmx, dvw, dvb, dmxw, dmxb, dgamma, dbeta, dmw};
  return tuple(r);
}

// ---- questions about Python objects and tensors: short, nothing is launched, the interpreter lock is held
struct Held {
  PyObject* const* a;
  Py_ssize_t n;
};

// (x, tensor | None, ...) -> bool: x is a GPU activation and every tensor is contiguous, of its type and device, on 16
// bytes; `graph`: and every one asks for its gradient (the composites' backward passes form all of them)
PyObject* same_storage(const Held& A, bool graph) {
  Value v[32];
  if (A.n < 1 || A.n > 32) throw std::runtime_error("uniform / trainable: 1 to 32 tensors");
  for (Py_ssize_t i = 0; i < A.n; ++i) {
    if (A.a[i] != Py_None && !THPVariable_Check(A.a[i])) throw std::runtime_error("uniform / trainable: tensors expected");
    read(A.a[i], &v[i]);
  }
  if (v[0].kind == Value::kNone) throw std::runtime_error("uniform / trainable: the activations are missing");
  const Tensor& x = *v[0].t;
  if (!eager()) return PyBool_FromLong(false);
  for (int i = 0; i < A.n; ++i)
    if (v[i].t && !plain(*v[i].t)) return PyBool_FromLong(false);
  const at::ScalarType dt = x.scalar_type();
  bool ok = x.is_cuda() && (dt == at::kFloat || dt == at::kBFloat16 || dt == at::kHalf) && x.dim() > 1 && x.numel() > 0 && !x.is_neg() &&
            (uintptr_t)x.data_ptr() % 16 == 0;
  for (int i = 1; ok && i < A.n; ++i)
    if (v[i].t) {
      const Tensor& t = *v[i].t;
      ok = t.scalar_type() == dt && t.device() == x.device() && t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0 && !t.is_neg() &&
           (!graph || t.requires_grad());
    }
  return PyBool_FromLong(ok);
}
PyObject* uniform(const Held& A) { return same_storage(A, false); }
PyObject* trainable(const Held& A) { return same_storage(A, true); }

// (autograd function's context) -> int: bit i is set where the running backward pass has use for input i's gradient
// (torch.autograd.grad of a few tensors has none for the others; needs_input_grad only knows what asked in the forward pass)
PyObject* wanted(const Held& A) {
  if (A.n != 1 || !PyObject_TypeCheck(A.a[0], &THPFunctionType)) throw std::runtime_error("wanted: an autograd function's context expected");
  const THPFunction* f = (const THPFunction*)A.a[0];
  const auto node = f->cdata.lock();
  if (!node) throw std::runtime_error("wanted: the context's node is gone");
  long long bits = 0;
  size_t edge = 0;
  for (size_t i = 0; i < f->is_variable_input.size(); ++i)
    if (f->is_variable_input[i] && node->task_should_compute_output(edge++)) bits |= 1ll << i;
  return PyLong_FromLongLong(bits);
}

// (dict, ...) -> bytes: storage address and in-place version of every tensor in the dictionaries' values, in order
PyObject* tensor_versions(const Held& A) {
  std::vector<int64_t> buf;
  for (int i = 0; i < A.n; ++i) {
    if (!PyDict_Check(A.a[i])) throw std::runtime_error("tensor_versions: dictionaries expected");
    PyObject *key, *value;
    Py_ssize_t pos = 0;
    while (PyDict_Next(A.a[i], &pos, &key, &value)) {
      if (value == Py_None) continue;
      if (!THPVariable_Check(value)) throw std::runtime_error("tensor_versions: tensors expected");
      const Tensor& t = THPVariable_Unpack(value);
      buf.push_back((int64_t)(uintptr_t)t.data_ptr());
      buf.push_back((int64_t)t._version());
    }
  }
  return PyBytes_FromStringAndSize((const char*)buf.data(), (Py_ssize_t)(buf.size() * 8));
}

// What the composites' gates ask of modules, (kinds, hooks on every module, bias, module, ...) -> bool: each is of exactly
// one of these types with its class's own call, nobody looking at inputs or outputs; `bias` not None: and holds a weight
// parameter, and a bias parameter or none.  Asked seven times per layer and token: one module 0.52 us, two 0.69, where the
// same questions in Python take 0.70 and 0.97.
PyObject* plain_modules(const Held& A) {
  static PyObject *const forward = PyUnicode_InternFromString("forward"), *const parameters = PyUnicode_InternFromString("_parameters"),
                  *const weight = PyUnicode_InternFromString("weight"), *const bias = PyUnicode_InternFromString("bias"),
                  *const hooks[] = {PyUnicode_InternFromString("_forward_hooks"), PyUnicode_InternFromString("_forward_pre_hooks"),
                                    PyUnicode_InternFromString("_backward_hooks"), PyUnicode_InternFromString("_backward_pre_hooks")};
  if (A.n < 4 || !PyTuple_Check(A.a[0]) || !PyTuple_Check(A.a[1])) throw std::runtime_error("plain_modules: kinds, hooks, bias, modules");
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(A.a[1]); ++i)
    if (PyObject_IsTrue(PyTuple_GET_ITEM(A.a[1], i))) return PyBool_FromLong(false);
  auto absent = [](PyObject* v) { return v == nullptr || v == Py_None; };
  for (Py_ssize_t k = 3; k < A.n; ++k) {
    PyObject* m = A.a[k];
    bool known = false;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(A.a[0]); ++i) known = known || (PyObject*)Py_TYPE(m) == PyTuple_GET_ITEM(A.a[0], i);
    if (!known) return PyBool_FromLong(false);
    PyObject* d = PyObject_GenericGetDict(m, nullptr);
    if (!d) return nullptr;
    bool ok = !PyDict_GetItem(d, forward);
    for (PyObject* h : hooks) {
      PyObject* v = PyDict_GetItem(d, h);
      ok = ok && (!v || !PyObject_IsTrue(v));
    }
    if (ok && A.a[2] != Py_None) {
      PyObject* p = PyDict_GetItem(d, parameters);
      PyObject* b = p && PyDict_Check(p) ? PyDict_GetItem(p, bias) : nullptr;
      ok = p && PyDict_Check(p) && !absent(PyDict_GetItem(p, weight)) && (A.a[2] == Py_True ? !absent(b) : b == Py_None);
    }
    Py_DECREF(d);
    if (!ok) return PyBool_FromLong(false);
  }
  return PyBool_FromLong(true);
}

// ---- entries.  A composite allocates, multiplies and launches without the interpreter lock (and in checked mode waits for
// its stream): other Python threads go on.
constexpr Py_ssize_t kMostArgs = 32;

PyObject* guarded(Result (*f)(const Args&), PyObject* const* a, Py_ssize_t n, const char* who) {
  Value v[kMostArgs];
  if (n > kMostArgs) {
    PyErr_Format(PyExc_RuntimeError, "%s: too many arguments", who);
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!read(a[i], &v[i])) return nullptr;
  Result r;
  std::string error;
  bool failed = false;
  PyThreadState* lock = PyEval_SaveThread();
  try {
    c10::AutoGradMode no_graph(false);
    r = f(Args{v, n, who});
  } catch (const std::exception& e) {
    failed = true;
    error = e.what();
  } catch (...) {
    failed = true;
    error = std::string(who) + ": unknown error";
  }
  PyEval_RestoreThread(lock);
  if (failed) {
    PyErr_SetString(PyExc_RuntimeError, error.c_str());
    return nullptr;
  }
  auto object = [](Tensor& t) { return t.defined() ? THPVariable_Wrap(std::move(t)) : (Py_INCREF(Py_None), Py_None); };
  if (r.one) return object(r.t[0]);
  PyObject* out = PyTuple_New(r.n);
  for (int i = 0; out && i < r.n; ++i) {
    PyObject* o = object(r.t[i]);
    if (!o) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, i, o);
  }
  return out;
}

PyObject* guarded_held(PyObject* (*f)(const Held&), PyObject* const* a, Py_ssize_t n, const char*) {
  try {
    return f(Held{a, n});
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
  } catch (...) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "unknown error");
  }
  return nullptr;
}

#define MEGA_METHOD(f, guard)                                                                                      \
  {#f,                                                                                                             \
   (PyCFunction)(void (*)(void))(PyObject * (*)(PyObject*, PyObject* const*, Py_ssize_t))                          \
       [](PyObject*, PyObject* const* a, Py_ssize_t n) -> PyObject* { return guard(f, a, n, #f); },                \
   METH_FASTCALL, nullptr}
#define MEGA_ENTRY(f) MEGA_METHOD(f, guarded)
#define MEGA_QUESTION(f) MEGA_METHOD(f, guarded_held)
PyMethodDef methods[] = {MEGA_ENTRY(token_gated_attention), MEGA_ENTRY(token_ffn),  MEGA_ENTRY(token_embed),
                         MEGA_ENTRY(token_norm),            MEGA_ENTRY(token_linear), MEGA_ENTRY(norm_ema_step),
                         MEGA_QUESTION(tensor_versions),       MEGA_ENTRY(train_prepare), MEGA_ENTRY(norm_move_forward),
                         MEGA_ENTRY(norm_move_backward),    MEGA_ENTRY(ema_param_backward),
                         MEGA_ENTRY(row_norm_forward),      MEGA_ENTRY(row_norm_backward), MEGA_ENTRY(ffn_forward),
                         MEGA_ENTRY(ffn_backward),          MEGA_ENTRY(swiglu_forward), MEGA_ENTRY(swiglu_backward),
                         MEGA_ENTRY(mix_forward),           MEGA_ENTRY(mix_out_forward), MEGA_ENTRY(mix_out_backward),
                         MEGA_ENTRY(mix_backward),          MEGA_QUESTION(uniform),    MEGA_QUESTION(trainable),
                         MEGA_QUESTION(plain_modules), MEGA_QUESTION(wanted),     MEGA_ENTRY(linear_own),
                         MEGA_ENTRY(attention_product),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "mega_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_mega_host(void) { return PyModule_Create(&module); }
