// What the 16-bit product kernels share: operands, the matrix instruction, what happens to a finished value.
#pragma once

#include "common.h"

namespace mega {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) short s16x4;

struct Gemm16P {
  const void *A, *B;   // element (m, k): m * lda + k, or (K-major) k * lda + m; (n, k) alike
  void* C;             // m * ldc + n
  const void* bias;    // [N] or null
  const void* R;       // added: m * ldr + n, or null
  void* pre;           // the value before the activation, or null
  int64_t lda, ldb, ldc, ldr;
  int M, N, K, silu;
  int mt, nt;
  int kstep;           // reduction indices of a split
  float* part;         // [splits][M][N], or null
  int full, splits;    // (wide tiles) tiles that are formed whole; parts of the others, part: [splits][tiles - full][tile]
};

// gemm16_wide.hip: tiles of 256 rows and tn columns
constexpr int kWideM = 256;
struct WidePlan {
  double us;           // estimated
  int tn, splits, full, kstep;
  size_t bytes;        // of partial sums
};
WidePlan gemm16_wide_plan(int64_t M, int64_t N, int64_t K);
void gemm16_wide_launch(Gemm16P G, const WidePlan& p, bool bf16, int ka, int kb, void* parts, hipStream_t s);

template <typename T>
__device__ __forceinline__ f32x4 mma16(uint4 a, uint4 b, f32x4 c) {
  if constexpr (__is_same(T, bf16_t))
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// v / (1 + e^-v): the reciprocal's quotient (scaled, so that it stays a normal number to the end of the exponential's range) and
// one Newton step from its remainder; an infinite denominator has none.  Of all bf16 values none differs from the division's
// result (the bare reciprocal's: 4, and nothing below -87.3), of fp16 one tie; on wide tiles 2 us of 8192 x 2048 x 1024 (40.5),
// the division 5.
__device__ __forceinline__ float silu_h(float v) {
  const float n = v * 0x1p-8f, d = fmaf(__expf(-v), 0x1p-8f, 0x1p-8f), y = __builtin_amdgcn_rcpf(d), q = n * y;
  return fmaf(fminf(fmaf(-d, q, n), 0x1p127f), y, q);
}

// E consecutive values of row m from column n on: bias and residual, one rounding, silu of the rounded value
template <typename T, int E>
__device__ __forceinline__ void finish16(const Gemm16P& G, int m, int n, float (&v)[E]) {
  T* const C = (T*)G.C;
  if (G.bias) {
    const Vec<T, E> b = *(const Vec<T, E>*)((const T*)G.bias + n);
#pragma unroll
    for (int u = 0; u < E; ++u) v[u] += to_float(b.v[u]);
  }
  if (G.R) {
    const Vec<T, E> r = *(const Vec<T, E>*)((const T*)G.R + (int64_t)m * G.ldr + n);
#pragma unroll
    for (int u = 0; u < E; ++u) v[u] += to_float(r.v[u]);
  }
  Vec<T, E> o;
#pragma unroll
  for (int u = 0; u < E; ++u) o.v[u] = from_float<T>(v[u]);
  if (G.pre) *(Vec<T, E>*)((T*)G.pre + (int64_t)m * G.ldc + n) = o;
  if (G.silu) {
#pragma unroll
    for (int u = 0; u < E; ++u) o.v[u] = from_float<T>(silu_h(to_float(o.v[u])));
  }
  *(Vec<T, E>*)(C + (int64_t)m * G.ldc + n) = o;
}

}  // namespace mega
