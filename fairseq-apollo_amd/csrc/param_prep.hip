// The small per-parameter formulas in front of the kernels, one launch each way instead of a chain of
// element-wise launches per formula step:
//   moving-average coefficients from the stored parameters
//     (fairseq/modules/complex_exponential_moving_average.py:79-96, exponential_moving_average.py:71-80) and
//   the TimestepNorm operands (weight + 1, bias, the prior mean and exp(prior log-variance) expanded over the
//     batch; fairseq/modules/norm_layer/timestep_norm.py:118-131),
// each with its backward pass.  Parameters are read in their storage type (fp32, bf16, fp16) and their gradients
// written in it; everything the other kernels consume is fp32.
#include "param_formulas.h"

namespace mega {
namespace {

struct CoeffArgs {
  CoeffSource S;
  // forward results (fp32, the layout every kernel of the library takes)
  float* p;            // [K, N]
  float* q;            // [K, N, 2]
  float* g;            // [K, N, 2]
  float* om;           // [D]
  // backward: gradients of the forward results in, gradients of the parameters out (storage type)
  const float* dp;
  const float* dq;
  const float* dg;
  const float* dom;
  void* dalpha;
  void* ddelta;
  void* dthird;
  void* dgamma;
  void* domega;
};

// one thread per (row, state)
__global__ __launch_bounds__(256) void ema_coeffs_fwd_kernel(const CoeffArgs A) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < A.S.D) A.om[i] = ld(A.S.omega, A.S.dtype, i);
  if (i >= (int64_t)A.S.K * A.S.N) return;
  const int k = (int)(i / A.S.N), n = (int)(i - (int64_t)k * A.S.N);
  const Coeff c = coeff_at(A.S, k, n);
  A.p[i] = c.p;
  A.q[2 * i] = c.qr;
  A.q[2 * i + 1] = c.qi;
  A.g[2 * i] = c.gr;
  A.g[2 * i + 1] = c.gi;
}

// Gradients of one (row, state)'s coefficients to its parameters; returns the state's share of theta's gradient.
// q_grad is (re, im) for the complex layer; the real layer has no imaginary part.
__device__ __forceinline__ float coeff_bwd_at(const CoeffSource& S, int k, int n, float dp, float dqr, float dqi, float dgr,
                                              float dgi, float st0, void* dalpha, void* ddelta, void* dthird, void* dgamma) {
  const int64_t i = (int64_t)k * S.N + n;
  const float a = sigm(ld(S.alpha, S.dtype, i)), d = sigm(ld(S.delta, S.dtype, i));
  float da, dr, share = 0.f;
  if (S.is_complex) {
    const float r = 1.0f - a * d;
    float sn, cs;
    sincosf((float)(n + 1) * (st0 * S.turn), &sn, &cs);
    dr = dqr * cs + dqi * sn;
    share = (float)(n + 1) * (r * (dqi * cs - dqr * sn));
    da = dp;
    st(dgamma, S.dtype, 2 * i, dgr * S.scale);
    st(dgamma, S.dtype, 2 * i + 1, dgi * S.scale);
  } else {
    dr = dqr;
    da = dp * ld(S.third, S.dtype, i);
    st(dthird, S.dtype, i, dp * a);
    st(dgamma, S.dtype, i, dgr * S.scale);
  }
  // r = 1 - a d
  st(dalpha, S.dtype, i, (da - dr * d) * a * (1.0f - a));
  st(ddelta, S.dtype, i, -dr * a * d * (1.0f - d));
  return share;
}

// one lane per (row, state), 64 / N rows per wave (N <= 64): the gradient of theta, a sum over the row's states, is
// collected from the row's lanes.  Rows of more than 64 states: one lane per row walking its states (rpw = 0).
__global__ __launch_bounds__(256) void ema_coeffs_bwd_kernel(const CoeffArgs A, const int rpw) {
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const int gid = (int)blockIdx.x * 256 + (int)threadIdx.x;
  const int N = A.S.N;
  if (gid < A.S.D) st(A.domega, A.S.dtype, gid, A.dom[gid]);
  int k, n0, n1;
  bool live;
  if (rpw > 0) {
    const int r = lane / N;
    k = ((int)blockIdx.x * 4 + wave) * rpw + r;
    n0 = lane - r * N;
    n1 = n0 + 1;
    live = r < rpw && k < A.S.K;
  } else {
    k = gid;
    n0 = 0;
    n1 = N;
    live = k < A.S.K;
  }
  float tsum = 0.f, st0 = 0.f;
  if (live) {
    if (A.S.is_complex) st0 = sigm(ld(A.S.third, A.S.dtype, k));
    for (int n = n0; n < n1; ++n) {
      const int64_t i = (int64_t)k * N + n;
      const bool c = A.S.is_complex;                             // real layer: [K, N] gradients, no pairs
      tsum += coeff_bwd_at(A.S, k, n, A.dp[i], c ? A.dq[2 * i] : A.dq[i], c ? A.dq[2 * i + 1] : 0.f,
                           c ? A.dg[2 * i] : A.dg[i], c ? A.dg[2 * i + 1] : 0.f, st0, A.dalpha, A.ddelta, A.dthird, A.dgamma);
    }
  }
  if (!A.S.is_complex) return;
  if (rpw > 0) {
    // the row's states in order, the same sum every run: lane n0 = 0 of the row adds the others' terms
    const int base = lane - n0;
    float total = 0.f;
    for (int j = 0; j < N; ++j) total += __shfl(tsum, base + j, 64);
    tsum = total;
    live = live && n0 == 0;
  }
  if (live) st(A.dthird, A.S.dtype, k, tsum * A.S.turn * st0 * (1.0f - st0));
}

// From the moving-average backward's sums over time (mega_ema_param_sums: per half, batch row, channel and state
// (sum2, sum1), per row and channel dy . x) straight to the gradients of the stored parameters, and the norm's parameter
// gradients in their storage type beside it: the sums over the batch, the products of ema_parameters.cc:95-96 and the
// coefficients' backward in one launch where there were three (4.7 + 5.8 + 2.4 us at 1024 channels; here 5.5 us).
// A workgroup owns 64 / N coefficient rows; its four waves share the batch rows (fixed order) and meet in LDS.
struct FinishArgs {
  CoeffSource S;
  const float* sums;     // [halves][B][D][N][4]
  const float* dyx;      // [B][D]
  void* dalpha;
  void* ddelta;
  void* dthird;
  void* dgamma;
  void* domega;
  int B, rpw, row_blocks;
  NormParamArgs norm;    // weight gradients; norm.dweight null: no norm
};

__global__ __launch_bounds__(256) void ema_param_finish_kernel(const FinishArgs A) {
  __shared__ float4 s_part[4][64];
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const CoeffSource& S = A.S;
  if ((int)blockIdx.x >= A.row_blocks) {         // the rest of the grid: omega and the norm's parameters
    const int i = ((int)blockIdx.x - A.row_blocks) * 256 + (int)threadIdx.x;
    if (i < S.D) {
      float o = 0.f;
      for (int b = 0; b < A.B; ++b) o += A.dyx[(size_t)b * S.D + i];
      st(A.domega, S.dtype, i, o);
    }
    if (A.norm.dweight) norm_params_bwd_at(A.norm, i);
    return;
  }
  const int r = lane / S.N, n = lane - r * S.N;
  const int k = (int)blockIdx.x * A.rpw + r;
  const bool live = r < A.rpw && k < S.K;
  const int half = live ? k / S.D : 0, d = live ? k - half * S.D : 0;
  float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) {
    const float4* src = (const float4*)A.sums + ((size_t)half * A.B * S.D + d) * S.N + n;
    const size_t step = (size_t)S.D * S.N;
#pragma unroll 4
    for (int b = wave; b < A.B; b += 4) {
      const float4 v = src[b * step];
      t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
    }
  }
  s_part[wave][lane] = t;
  __syncthreads();
  if (wave != 0) return;
  float share = 0.f, st0 = 0.f;
  if (live) {
    float s2r = 0.f, s2i = 0.f, s1r = 0.f, s1i = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float4 v = s_part[w][lane];
      s2r += v.x; s2i += v.y; s1r += v.z; s1i += v.w;
    }
    if (S.is_complex) st0 = sigm(ld(S.third, S.dtype, k));
    const Coeff c = coeff_at(S, k, n);
    // dp = Re(sum2 gamma), dq = conj(sum1 p gamma), dgamma = conj(sum2 p)
    share = coeff_bwd_at(S, k, n, s2r * c.gr - s2i * c.gi, c.p * (s1r * c.gr - s1i * c.gi), -c.p * (s1r * c.gi + s1i * c.gr),
                         c.p * s2r, -c.p * s2i, st0, A.dalpha, A.ddelta, A.dthird, A.dgamma);
  }
  if (!S.is_complex) return;
  const int base = lane - n;
  float total = 0.f;
  for (int j = 0; j < S.N; ++j) total += __shfl(share, base + j, 64);
  if (live && n == 0) st(A.dthird, S.dtype, k, total * S.turn * st0 * (1.0f - st0));
}

__global__ __launch_bounds__(256) void norm_params_fwd_kernel(const NormParamArgs A) {
  norm_params_fwd_at(A, (int)blockIdx.x * 256 + (int)threadIdx.x);
}

__global__ __launch_bounds__(256) void norm_params_bwd_kernel(const NormParamArgs A) {
  norm_params_bwd_at(A, (int)blockIdx.x * 256 + (int)threadIdx.x);
}

bool known(int dtype) { return dtype == MEGA_F32 || dtype == MEGA_BF16 || dtype == MEGA_F16; }

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_ema_coeffs_fwd(const void* alpha, const void* delta, const void* theta_or_beta, const void* gamma,
                                   const void* omega, int dtype, int is_complex, int64_t K, int64_t N, int64_t D,
                                   float* p, float* q, float* gamma_out, float* omega_out, void* stream) {
  MEGA_REQUIRE(known(dtype), MEGA_ERR_ARG, "ema_coeffs_fwd: unknown dtype %d", dtype);
  MEGA_REQUIRE(K > 0 && N > 0 && D > 0 && K * N < (1ll << 30) && (K == D || K == 2 * D), MEGA_ERR_ARG,
               "ema_coeffs_fwd: bad sizes K=%lld N=%lld D=%lld", (long long)K, (long long)N, (long long)D);
  MEGA_REQUIRE(alpha && delta && theta_or_beta && gamma && omega && p && q && gamma_out && omega_out, MEGA_ERR_ARG,
               "ema_coeffs_fwd: null pointer argument");
  CoeffArgs A = {};
  A.S = coeff_source(alpha, delta, theta_or_beta, gamma, omega, dtype, is_complex, K, N, D);
  A.p = p; A.q = q; A.g = gamma_out; A.om = omega_out;
  const int64_t n = K * N > D ? K * N : D;
  hipLaunchKernelGGL(ema_coeffs_fwd_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream, A);
  MEGA_CHECK_LAUNCH("ema_coeffs_fwd");
  return MEGA_OK;
}

extern "C" int mega_ema_coeffs_bwd(const float* p_grad, const float* q_grad, const float* gamma_out_grad,
                                   const float* omega_out_grad, const void* alpha, const void* delta,
                                   const void* theta_or_beta, int dtype, int is_complex, int64_t K, int64_t N,
                                   int64_t D, void* alpha_grad, void* delta_grad, void* theta_or_beta_grad,
                                   void* gamma_grad, void* omega_grad, void* stream) {
  MEGA_REQUIRE(known(dtype), MEGA_ERR_ARG, "ema_coeffs_bwd: unknown dtype %d", dtype);
  MEGA_REQUIRE(K > 0 && N > 0 && D > 0 && K * N < (1ll << 30) && (K == D || K == 2 * D), MEGA_ERR_ARG,
               "ema_coeffs_bwd: bad sizes K=%lld N=%lld D=%lld", (long long)K, (long long)N, (long long)D);
  MEGA_REQUIRE(p_grad && q_grad && gamma_out_grad && omega_out_grad && alpha && delta && theta_or_beta && alpha_grad &&
                   delta_grad && theta_or_beta_grad && gamma_grad && omega_grad,
               MEGA_ERR_ARG, "ema_coeffs_bwd: null pointer argument");
  CoeffArgs A = {};
  A.S = coeff_source(alpha, delta, theta_or_beta, nullptr, nullptr, dtype, is_complex, K, N, D);
  A.dp = p_grad; A.dq = q_grad; A.dg = gamma_out_grad; A.dom = omega_out_grad;
  A.dalpha = alpha_grad; A.ddelta = delta_grad; A.dthird = theta_or_beta_grad; A.dgamma = gamma_grad;
  A.domega = omega_grad;
  const int rpw = N <= 64 ? (int)(64 / N) : 0;                   // rows per wave, one lane per (row, state)
  int64_t blocks = rpw > 0 ? ceil_div(K, 4 * rpw) : ceil_div(K, 256);
  if (blocks * 256 < D) blocks = ceil_div(D, 256);               // the first D threads also copy omega's gradient
  hipLaunchKernelGGL(ema_coeffs_bwd_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, A, rpw);
  MEGA_CHECK_LAUNCH("ema_coeffs_bwd");
  return MEGA_OK;
}

extern "C" int mega_norm_params_fwd(const void* weight, const void* bias, int dtype, const void* prior_mean,
                                    const void* prior_logv, int prior_dtype, int64_t H, int64_t G, int64_t B,
                                    float* gamma, float* beta, float* prev_mean, float* prev_var, void* stream) {
  MEGA_REQUIRE(known(dtype) && known(prior_dtype), MEGA_ERR_ARG, "norm_params_fwd: unknown dtype %d / %d", dtype,
               prior_dtype);
  MEGA_REQUIRE(H > 0 && G > 0 && B > 0 && H < (1ll << 30) && B * G < (1ll << 30), MEGA_ERR_ARG,
               "norm_params_fwd: bad sizes H=%lld G=%lld B=%lld", (long long)H, (long long)G, (long long)B);
  MEGA_REQUIRE(weight && bias && prior_mean && prior_logv && gamma && beta && prev_mean && prev_var, MEGA_ERR_ARG,
               "norm_params_fwd: null pointer argument");
  NormParamArgs A = {};
  A.weight = weight; A.bias = bias; A.prior_mean = prior_mean; A.prior_logv = prior_logv;
  A.wdtype = dtype; A.pdtype = prior_dtype; A.H = (int)H; A.G = (int)G; A.B = (int)B;
  A.gamma = gamma; A.beta = beta; A.prev_mean = prev_mean; A.prev_var = prev_var;
  const int64_t n = H > B * G ? H : B * G;
  hipLaunchKernelGGL(norm_params_fwd_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream, A);
  MEGA_CHECK_LAUNCH("norm_params_fwd");
  return MEGA_OK;
}

extern "C" int mega_norm_params_bwd(const float* gamma_grad, const float* beta_grad, const float* prev_mean_grad,
                                    const float* prev_var_grad, const void* prior_logv, int dtype, int prior_dtype,
                                    int64_t H, int64_t G, int64_t B, void* weight_grad, void* bias_grad,
                                    void* prior_mean_grad, void* prior_logv_grad, void* stream) {
  MEGA_REQUIRE(known(dtype) && known(prior_dtype), MEGA_ERR_ARG, "norm_params_bwd: unknown dtype %d / %d", dtype,
               prior_dtype);
  MEGA_REQUIRE(H > 0 && G > 0 && B > 0 && H < (1ll << 30) && B * G < (1ll << 30), MEGA_ERR_ARG,
               "norm_params_bwd: bad sizes H=%lld G=%lld B=%lld", (long long)H, (long long)G, (long long)B);
  MEGA_REQUIRE(gamma_grad && beta_grad && weight_grad && bias_grad, MEGA_ERR_ARG,
               "norm_params_bwd: null pointer argument");
  MEGA_REQUIRE((prior_mean_grad == nullptr) == (prior_logv_grad == nullptr), MEGA_ERR_ARG,
               "norm_params_bwd: the two prior gradients go together");
  MEGA_REQUIRE(!prior_mean_grad || (prev_mean_grad && prev_var_grad && prior_logv), MEGA_ERR_ARG,
               "norm_params_bwd: the prior's gradients need prev_mean_grad, prev_var_grad and prior_logv");
  NormParamArgs A = {};
  A.prior_logv = prior_logv; A.wdtype = dtype; A.pdtype = prior_dtype; A.H = (int)H; A.G = (int)G; A.B = (int)B;
  A.dgamma = gamma_grad; A.dbeta = beta_grad; A.dprev_mean = prev_mean_grad; A.dprev_var = prev_var_grad;
  A.dweight = weight_grad; A.dbias = bias_grad; A.dprior_mean = prior_mean_grad; A.dprior_logv = prior_logv_grad;
  const int64_t n = H > G ? H : G;
  hipLaunchKernelGGL(norm_params_bwd_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream, A);
  MEGA_CHECK_LAUNCH("norm_params_bwd");
  return MEGA_OK;
}

extern "C" int mega_ema_param_finish(const float* sums, const float* dyx, const MegaEmaParams* e, int64_t B,
                                     const MegaEmaParamGrads* grads, const MegaNormParamGrads* norm, void* stream) {
  MEGA_REQUIRE(sums && dyx && e && grads, MEGA_ERR_ARG, "ema_param_finish: null pointer argument");
  MEGA_REQUIRE(known((int)e->dtype) && e->N > 0 && e->N <= 16 && e->D > 0 && (e->K == e->D || e->K == 2 * e->D) &&
                   e->K * e->N < (1ll << 30) && B > 0,
               MEGA_ERR_ARG, "ema_param_finish: bad sizes");
  MEGA_REQUIRE(e->alpha && e->delta && e->third && e->gamma && grads->alpha && grads->delta && grads->third &&
                   grads->gamma && grads->omega,
               MEGA_ERR_ARG, "ema_param_finish: null pointer argument");
  FinishArgs A = {};
  A.S = coeff_source(e->alpha, e->delta, e->third, e->gamma, nullptr, (int)e->dtype, (int)e->is_complex, e->K, e->N, e->D);
  A.sums = sums; A.dyx = dyx; A.dalpha = grads->alpha; A.ddelta = grads->delta; A.dthird = grads->third;
  A.dgamma = grads->gamma; A.domega = grads->omega; A.B = (int)B;
  A.rpw = (int)(64 / e->N);
  A.row_blocks = (int)ceil_div(e->K, A.rpw);
  int64_t rest = e->D;
  if (norm) {
    MEGA_REQUIRE(known((int)norm->dtype) && known((int)norm->prior_dtype) && norm->gamma_grad && norm->beta_grad &&
                     norm->weight && norm->bias && norm->H > 0 && norm->G > 0 && norm->H < (1ll << 30) &&
                     (norm->prior_mean == nullptr) == (norm->prior_logv_grad == nullptr) &&
                     (!norm->prior_mean || (norm->mean_grad && norm->var_grad && norm->prior_logv)),
                 MEGA_ERR_ARG, "ema_param_finish: bad norm arguments");
    NormParamArgs& P = A.norm;
    P.wdtype = (int)norm->dtype; P.pdtype = (int)norm->prior_dtype; P.H = (int)norm->H; P.G = (int)norm->G; P.B = (int)B;
    P.dgamma = norm->gamma_grad; P.dbeta = norm->beta_grad; P.dprev_mean = norm->mean_grad; P.dprev_var = norm->var_grad;
    P.prior_logv = norm->prior_logv; P.dweight = norm->weight; P.dbias = norm->bias; P.dprior_mean = norm->prior_mean;
    P.dprior_logv = norm->prior_logv_grad;
    rest = rest > norm->H ? rest : norm->H;
    rest = rest > norm->G ? rest : norm->G;
  }
  hipLaunchKernelGGL(ema_param_finish_kernel, dim3((unsigned)(A.row_blocks + ceil_div(rest, 256))), dim3(256), 0,
                     (hipStream_t)stream, A);
  MEGA_CHECK_LAUNCH("ema_param_finish");
  return MEGA_OK;
}
