// The per-parameter formulas shared by the kernels that start from stored parameters: moving-average coefficients
// (fairseq/modules/complex_exponential_moving_average.py:79-96, exponential_moving_average.py:71-80) and the TimestepNorm
// operands (fairseq/modules/norm_layer/timestep_norm.py:118-131).  Parameters are read in their storage type.
#pragma once
#include "common.h"

namespace mega {

__device__ __forceinline__ float ld(const void* p, int dtype, int64_t i) {
  if (dtype == MEGA_F32) return ((const float*)p)[i];
  if (dtype == MEGA_BF16) return to_float(((const bf16_t*)p)[i]);
  return to_float(((const f16_t*)p)[i]);
}
__device__ __forceinline__ void st(void* p, int dtype, int64_t i, float v) {
  if (dtype == MEGA_F32) ((float*)p)[i] = v;
  else if (dtype == MEGA_BF16) ((bf16_t*)p)[i] = from_float<bf16_t>(v);
  else ((f16_t*)p)[i] = from_float<f16_t>(v);
}
__device__ __forceinline__ float sigm(float x) { return 1.0f / (1.0f + expf(-x)); }

struct CoeffSource {
  const void* alpha;   // [K, N]
  const void* delta;   // [K, N]
  const void* third;   // complex: theta [K]; real: beta [K, N]
  const void* gamma;   // complex: [K, N, 2]; real: [K, N]
  const void* omega;   // [D]
  int dtype, is_complex, K, N, D;
  float scale, turn;   // sqrt(1 / N), 2 pi / N
};

inline CoeffSource coeff_source(const void* alpha, const void* delta, const void* third, const void* gamma,
                                const void* omega, int dtype, int is_complex, int64_t K, int64_t N, int64_t D) {
  CoeffSource S;
  S.alpha = alpha; S.delta = delta; S.third = third; S.gamma = gamma; S.omega = omega;
  S.dtype = dtype; S.is_complex = is_complex ? 1 : 0; S.K = (int)K; S.N = (int)N; S.D = (int)D;
  S.scale = (float)sqrt(1.0 / (double)N); S.turn = (float)(2.0 * 3.14159265358979323846 / (double)N);
  return S;
}

struct Coeff {
  float p, qr, qi, gr, gi;
};
__device__ __forceinline__ Coeff coeff_at(const CoeffSource& S, int k, int n) {
  const int64_t i = (int64_t)k * S.N + n;
  const float a = sigm(ld(S.alpha, S.dtype, i)), d = sigm(ld(S.delta, S.dtype, i));
  const float r = 1.0f - a * d;
  Coeff c;
  if (S.is_complex) {
    float sn, cs;
    sincosf((float)(n + 1) * (sigm(ld(S.third, S.dtype, k)) * S.turn), &sn, &cs);
    c.p = a;
    c.qr = r * cs;
    c.qi = r * sn;
    c.gr = ld(S.gamma, S.dtype, 2 * i) * S.scale;
    c.gi = ld(S.gamma, S.dtype, 2 * i + 1) * S.scale;
  } else {
    c.p = a * ld(S.third, S.dtype, i);
    c.qr = r;
    c.qi = 0.f;
    c.gr = ld(S.gamma, S.dtype, i) * S.scale;
    c.gi = 0.f;
  }
  return c;
}

struct NormParamArgs {
  const void* weight;      // [H]
  const void* bias;        // [H]
  const void* prior_mean;  // [G]
  const void* prior_logv;  // [G]
  int wdtype, pdtype, H, G, B;
  float* gamma;            // [H] weight + 1
  float* beta;             // [H]
  float* prev_mean;        // [B, G]
  float* prev_var;         // [B, G]
  const int64_t* prior_count;   // one number, spread over prev_count [B]; or null
  int64_t* prev_count;
  const float* dgamma;     // backward: gradients of the four results
  const float* dbeta;
  const float* dprev_mean;
  const float* dprev_var;
  void* dweight;
  void* dbias;
  void* dprior_mean;       // null: the prior is a buffer
  void* dprior_logv;
};

// element i of the larger of [H] and [B, G]
__device__ __forceinline__ void norm_params_fwd_at(const NormParamArgs& A, int i) {
  if (i < A.H) {
    A.gamma[i] = ld(A.weight, A.wdtype, i) + 1.0f;
    A.beta[i] = ld(A.bias, A.wdtype, i);
  }
  if (i < A.B * A.G) {
    const int g = i % A.G;
    A.prev_mean[i] = ld(A.prior_mean, A.pdtype, g);
    A.prev_var[i] = expf(ld(A.prior_logv, A.pdtype, g));
  }
  if (A.prior_count && i < A.B) A.prev_count[i] = *A.prior_count;
}

__device__ __forceinline__ void norm_params_bwd_at(const NormParamArgs& A, int i) {
  if (i < A.H) {
    st(A.dweight, A.wdtype, i, A.dgamma[i]);
    st(A.dbias, A.wdtype, i, A.dbeta[i]);
  }
  if (i < A.G && A.dprior_mean) {
    float sm = 0.f, sv = 0.f;
    for (int b = 0; b < A.B; ++b) {            // batch rows in order: the same sum every run
      sm += A.dprev_mean[b * A.G + i];
      sv += A.dprev_var[b * A.G + i];
    }
    st(A.dprior_mean, A.pdtype, i, sm);
    st(A.dprior_logv, A.pdtype, i, sv * expf(ld(A.prior_logv, A.pdtype, i)));
  }
}

}  // namespace mega
