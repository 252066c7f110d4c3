// Per-token normalisations of the layers with their backward passes, and column sums that ride along with an
// element-wise backward pass:
//   row_norm_fwd   y = (x - mean) / sqrt(var + eps) * (w + 1) + b      (LayerNorm: norm_layer/layer_norm.py:85-111)
//                  y = x / sqrt(mean(x^2) + eps) * (w + 1)             (RMSNorm: norm_layer/layer_norm.py:41-59)
//   row_norm_bwd   dx (+ a gradient that joins it), dw, db
//   silu_bwd_sum   dx = dy silu'(x) and the sum of dx over the tokens (the bias gradient of the projection in front)
// All of them are bound by memory: one wave holds a token's row in registers (16-byte loads, all in flight together),
// so every operand crosses memory once.  Statistics are formed again in the backward pass: the row is in registers
// anyway, and nothing has to be kept between the passes.  At 8192 tokens of 1024 channels in bf16: LayerNorm 9.1 us
// forwards (3.7 TB/s) and 22.6 us backwards with a joined gradient and the parameter sums (67 MB: 3.0 TB/s; 29.5 us
// before the next token's rows were fetched ahead), RMSNorm 8.9 and 16.0; as torch operations under autograd the two
// cost a training step of a two-layer model about 700 us more than here.  dx = dy silu'(x) with its sums, 8192 x 2816:
// 22.3 us (100 MB, 4.5 TB/s), where a pass for dx and one for its sums took 20.4 and 31.
#include "common.h"

namespace mega {
namespace {

constexpr int kThreads = 256;            // 4 waves
constexpr int kWaves = kThreads / 64;
constexpr int kMaxRows = 512;            // workgroups (rows of partial sums) of a backward launch

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// A row of D values as NV vectors per lane: vector u of a lane starts at column (u * 64 + lane) * VEC.
template <typename T, int VEC, int NV>
__device__ __forceinline__ void load_row(const T* row, int D, int lane, float (&f)[NV][VEC]) {
  Vec<T, VEC> v[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = (u * 64 + lane) * VEC;
    if (j < D) v[u] = *(const Vec<T, VEC>*)(row + j);
  }
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = (u * 64 + lane) * VEC;
#pragma unroll
    for (int e = 0; e < VEC; ++e) f[u][e] = j < D ? to_float(v[u].v[e]) : 0.f;
  }
}

// mean (0 for RMS) and 1 / sqrt of a row in registers; columns past D hold zeros
template <int VEC, int NV, bool LN>
__device__ __forceinline__ void row_stats(const float (&f)[NV][VEC], int D, int lane, float eps, float& mu, float& rs) {
  float s = 0.f, q = 0.f;
  if (LN) {
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int e = 0; e < VEC; ++e) s += f[u][e];
    mu = wave_sum(s) / (float)D;
  } else {
    mu = 0.f;
  }
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const bool in = (u * 64 + lane) * VEC < D;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float d = in ? f[u][e] - mu : 0.f;
      q = fmaf(d, d, q);
    }
  }
  rs = rsqrtf(wave_sum(q) / (float)D + eps);
}

template <typename T, int VEC, int NV, bool LN>
__global__ __launch_bounds__(kThreads) void row_norm_fwd_kernel(const T* __restrict__ x, int64_t xs,
                                                                const T* __restrict__ w, const T* __restrict__ b,
                                                                T* __restrict__ y, int64_t T_, int D, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (t >= T_) return;
  float f[NV][VEC];
  load_row<T, VEC, NV>(x + t * xs, D, lane, f);
  float mu, rs;
  row_stats<VEC, NV, LN>(f, D, lane, eps, mu, rs);
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = (u * 64 + lane) * VEC;
    if (j < D) {
      Vec<T, VEC> o, wv, bv;
      if (w) wv = *(const Vec<T, VEC>*)(w + j);
      if (LN && b) bv = *(const Vec<T, VEC>*)(b + j);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float r = (f[u][e] - mu) * rs;
        if (w) r *= to_float(wv.v[e]) + 1.0f;
        if (LN && b) r += to_float(bv.v[e]);
        o.v[e] = from_float<T>(r);
      }
      *(Vec<T, VEC>*)(y + t * (int64_t)D + j) = o;
    }
  }
}

// A wave walks tokens t, t + waves, ...: its columns' shares of dw and db stay in registers until the end; the waves of
// a workgroup add up in LDS in wave order, one row of 2 D sums per workgroup goes to `part`, and column_finish adds
// the rows in a fixed order: the same bits on every run.
template <typename T, int VEC, int NV, bool LN>
__global__ __launch_bounds__(kThreads) void row_norm_bwd_kernel(const T* __restrict__ dy, const T* __restrict__ x,
                                                                int64_t xs, const T* __restrict__ w,
                                                                const T* __restrict__ add, T* __restrict__ dx,
                                                                float* __restrict__ part, int64_t T_, int D, float eps) {
  extern __shared__ float s_acc[];                     // [2][D]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float aw[NV][VEC], ab[LN ? NV : 1][VEC];
#pragma unroll
  for (int u = 0; u < NV; ++u)
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      aw[u][e] = 0.f;
      if (LN) ab[LN ? u : 0][e] = 0.f;
    }
  const float inv = 1.0f / (float)D;
  const int64_t stride = (int64_t)gridDim.x * kWaves;
  int64_t t = (int64_t)blockIdx.x * kWaves + wave;
  Vec<T, VEC> nx[NV], ny[NV], na[NV];                  // the next token's rows, on their way while this one is worked on
  auto fetch = [&](int64_t tt) {
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int j = (u * 64 + lane) * VEC;
      if (tt < T_ && j < D) {
        nx[u] = *(const Vec<T, VEC>*)(x + tt * xs + j);
        ny[u] = *(const Vec<T, VEC>*)(dy + tt * (int64_t)D + j);
        if (add) na[u] = *(const Vec<T, VEC>*)(add + tt * (int64_t)D + j);
      }
    }
  };
  fetch(t);
  for (; t < T_; t += stride) {
    float f[NV][VEC], g[NV][VEC];
    Vec<T, VEC> av[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const bool in = (u * 64 + lane) * VEC < D;
      av[u] = na[u];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        f[u][e] = in ? to_float(nx[u].v[e]) : 0.f;
        g[u][e] = in ? to_float(ny[u].v[e]) : 0.f;
      }
    }
    fetch(t + stride);
    float mu, rs;
    row_stats<VEC, NV, LN>(f, D, lane, eps, mu, rs);
    float c1 = 0.f, c2 = 0.f;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int j = (u * 64 + lane) * VEC;
      if (j < D) {
        Vec<T, VEC> wv;
        if (w) wv = *(const Vec<T, VEC>*)(w + j);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const float xh = (f[u][e] - mu) * rs;
          f[u][e] = xh;
          aw[u][e] = fmaf(g[u][e], xh, aw[u][e]);
          if (LN) ab[LN ? u : 0][e] += g[u][e];
          if (w) g[u][e] *= to_float(wv.v[e]) + 1.0f;
          c2 = fmaf(g[u][e], xh, c2);
          if (LN) c1 += g[u][e];
        }
      }
    }
    c2 = wave_sum(c2) * inv;
    if (LN) c1 = wave_sum(c1) * inv;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int j = (u * 64 + lane) * VEC;
      if (j < D) {
        Vec<T, VEC> o;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          float r = rs * (g[u][e] - c1 - f[u][e] * c2);
          if (add) r += to_float(av[u].v[e]);
          o.v[e] = from_float<T>(r);
        }
        *(Vec<T, VEC>*)(dx + t * (int64_t)D + j) = o;
      }
    }
  }
  for (int k = 0; k < kWaves; ++k) {
    __syncthreads();
    if (wave == k) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int j = (u * 64 + lane) * VEC;
        if (j < D)
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            s_acc[j + e] = (k ? s_acc[j + e] : 0.f) + aw[u][e];
            if (LN) s_acc[D + j + e] = (k ? s_acc[D + j + e] : 0.f) + ab[LN ? u : 0][e];
          }
      }
    }
  }
  __syncthreads();
  const int W = LN ? 2 * D : D;
  for (int i = threadIdx.x; i < W; i += kThreads) part[(size_t)blockIdx.x * W + i] = s_acc[i];
}

// out[c] = sum over rows of part[row][c] (fixed order: 16 waves each every 16th row, then the waves in order).
// The columns below `split` go to out0, the rest to out1 (null: dropped).
constexpr int kSlices = 16;
template <typename T>
__global__ __launch_bounds__(64 * kSlices) void column_finish_kernel(const float* __restrict__ part, int rows, int W, int split,
                                                                     T* __restrict__ out0, T* __restrict__ out1) {
  __shared__ float s_sum[kSlices][64];
  const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
  if (c < W) {
    int r = slice;
    for (; r + 3 * kSlices < rows; r += 4 * kSlices) {
      a0 += part[(size_t)r * W + c];
      a1 += part[(size_t)(r + kSlices) * W + c];
      a2 += part[(size_t)(r + 2 * kSlices) * W + c];
      a3 += part[(size_t)(r + 3 * kSlices) * W + c];
    }
    for (; r < rows; r += kSlices) a0 += part[(size_t)r * W + c];
  }
  s_sum[slice][lane] = (a0 + a1) + (a2 + a3);
  __syncthreads();
  if (slice == 0 && c < W) {
    float a = 0.f;
#pragma unroll
    for (int w = 0; w < kSlices; ++w) a += s_sum[w][lane];
    if (c < split) {
      if (out0) out0[c] = from_float<T>(a);
    } else if (out1) {
      out1[c - split] = from_float<T>(a);
    }
  }
}

// dx = dy silu'(x) (SILU) or nothing but the sums (x = null), and one row of column sums per slab of rows.  A workgroup
// owns 64 VEC columns and `slab` rows; its four waves take every fourth row, four rows in flight each.
template <typename T, int VEC, bool SILU>
__global__ __launch_bounds__(kThreads) void sum_rows_kernel(const T* __restrict__ dy, int64_t rs, const T* __restrict__ x,
                                                            T* __restrict__ dx, float* __restrict__ part, int64_t T_, int W,
                                                            int slab) {
  using V = Vec<T, VEC>;
  __shared__ float s_acc[kWaves - 1][64 * VEC];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c0 = ((int)blockIdx.x * 64 + lane) * VEC;
  const int64_t r0 = (int64_t)blockIdx.y * slab, r1 = r0 + slab < T_ ? r0 + slab : T_;
  float acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
  if (c0 < W) {
    for (int64_t r = r0 + wave; r < r1; r += 16) {
      V v[4], a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t rr = r + 4 * u;
        if (rr < r1) {
          v[u] = *(const V*)(dy + rr * rs + c0);
          if (SILU) a[u] = *(const V*)(x + rr * W + c0);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t rr = r + 4 * u;
        if (rr < r1) {
          if (SILU) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
              const float xv = to_float(a[u].v[e]);
              const float sg = __builtin_amdgcn_rcpf(1.0f + __expf(-xv));
              v[u].v[e] = from_float<T>(to_float(v[u].v[e]) * sg * fmaf(xv, 1.0f - sg, 1.0f));
            }
            *(V*)(dx + rr * W + c0) = v[u];
          }
#pragma unroll
          for (int e = 0; e < VEC; ++e) acc[e] += to_float(v[u].v[e]);
        }
      }
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) s_acc[wave - 1][lane * VEC + e] = acc[e];
  }
  __syncthreads();
  if (wave == 0 && c0 < W) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      float t = acc[e];
      for (int w = 0; w < kWaves - 1; ++w) t += s_acc[w][lane * VEC + e];
      part[(int64_t)blockIdx.y * W + c0 + e] = t;
    }
  }
}

// Rows per slab: enough workgroups to fill the chip several times (a slab of 256 rows left 64 of them at 8192 x 1024:
// 20.7 us), at least 32 rows so that the partial sums stay small beside the matrix, at most 256.
int slab_rows(int64_t T_, int64_t W, int vec) {
  const int64_t xb = ceil_div(W, 64 * vec);
  int64_t slab = 256;
  while (slab > 32 && xb * ceil_div(T_, slab) < 2048) slab /= 2;
  return (int)slab;
}

template <typename T>
int finish(const float* part, int rows, int W, int split, void* o0, void* o1, hipStream_t s) {
  hipLaunchKernelGGL(column_finish_kernel<T>, dim3((unsigned)ceil_div(W, 64)), dim3(64 * kSlices), 0, s, part, rows, W, split,
                     (T*)o0, (T*)o1);
  MEGA_CHECK_LAUNCH("column sums");
  return MEGA_OK;
}

template <typename T, bool LN>
int launch_fwd(const void* x, int64_t xs, const void* w, const void* b, void* y, int64_t T_, int64_t D, float eps,
               hipStream_t s) {
  constexpr int VEC = 16 / (int)sizeof(T);
  const dim3 grid((unsigned)ceil_div(T_, kWaves));
  const int64_t nv = ceil_div(D, 64 * VEC);
#define MEGA_RN(NV)                                                                                                        \
  hipLaunchKernelGGL((row_norm_fwd_kernel<T, VEC, NV, LN>), grid, dim3(kThreads), 0, s, (const T*)x, xs, (const T*)w,      \
                     (const T*)b, (T*)y, T_, (int)D, eps)
  constexpr int kMost = 2048 / (64 * VEC);    // a row has at most 2048 columns
  if (nv <= 1) MEGA_RN(1); else if (nv <= 2) MEGA_RN(2); else if (nv <= 4) MEGA_RN(4); else MEGA_RN(kMost);
#undef MEGA_RN
  MEGA_CHECK_LAUNCH("row_norm_fwd");
  return MEGA_OK;
}

int bwd_rows(int64_t T_) {
  const int64_t w = ceil_div(T_, kWaves);
  return (int)(w < kMaxRows ? w : kMaxRows);
}

template <typename T, bool LN>
int launch_bwd(const void* dy, const void* x, int64_t xs, const void* w, const void* add, void* dx, void* dw, void* db,
               int64_t T_, int64_t D, float eps, float* part, hipStream_t s) {
  constexpr int VEC = 16 / (int)sizeof(T);
  const int rows = bwd_rows(T_);
  const int64_t nv = ceil_div(D, 64 * VEC);
  const size_t smem = (size_t)2 * D * 4;
#define MEGA_RN(NV)                                                                                                        \
  hipLaunchKernelGGL((row_norm_bwd_kernel<T, VEC, NV, LN>), dim3(rows), dim3(kThreads), smem, s, (const T*)dy, (const T*)x, \
                     xs, (const T*)w, (const T*)add, (T*)dx, part, T_, (int)D, eps)
  constexpr int kMost = 2048 / (64 * VEC);    // a row has at most 2048 columns
  if (nv <= 1) MEGA_RN(1); else if (nv <= 2) MEGA_RN(2); else if (nv <= 4) MEGA_RN(4); else MEGA_RN(kMost);
#undef MEGA_RN
  MEGA_CHECK_LAUNCH("row_norm_bwd");
  if (!dw && !db) return MEGA_OK;
  return finish<T>(part, rows, (int)(LN ? 2 * D : D), (int)D, dw, db, s);
}

bool row_shape(int dtype, int64_t D) {
  const int vec = dtype == MEGA_F32 ? 4 : 8;
  return D > 0 && D % vec == 0 && D <= (int64_t)64 * 32;
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_row_norm_covers(int dtype, int64_t D) {
  return (dtype == MEGA_F32 || dtype == MEGA_BF16 || dtype == MEGA_F16) && row_shape(dtype, D) ? 1 : 0;
}

extern "C" int mega_row_norm_fwd(const void* x, int64_t x_stride, const void* weight, const void* bias, void* y, int dtype,
                                 int kind, int64_t T_, int64_t D, double eps, void* stream) {
  MEGA_REQUIRE(mega_row_norm_covers(dtype, D) && T_ >= 0 && (kind == MEGA_TOKEN_RMSNORM || kind == MEGA_TOKEN_LAYERNORM),
               MEGA_ERR_UNSUPPORTED, "row_norm_fwd: D=%ld, dtype %d", (long)D, dtype);
  if (T_ == 0) return MEGA_OK;
  const int es = dtype == MEGA_F32 ? 4 : 2;
  MEGA_REQUIRE(x && y && x_stride * es % 16 == 0 && (((uintptr_t)x | (uintptr_t)y | (uintptr_t)weight | (uintptr_t)bias) % 16) == 0 &&
                   ceil_div(T_, kWaves) < (int64_t)1 << 31,
               MEGA_ERR_ARG, "row_norm_fwd: null or unaligned rows");
  hipStream_t s = (hipStream_t)stream;
  const bool ln = kind == MEGA_TOKEN_LAYERNORM;
#define MEGA_D(T) return ln ? launch_fwd<T, true>(x, x_stride, weight, bias, y, T_, D, (float)eps, s) \
                            : launch_fwd<T, false>(x, x_stride, weight, nullptr, y, T_, D, (float)eps, s)
  if (dtype == MEGA_F32) MEGA_D(float);
  if (dtype == MEGA_BF16) MEGA_D(bf16_t);
  MEGA_D(f16_t);
#undef MEGA_D
}

extern "C" size_t mega_row_norm_bwd_workspace_bytes(int64_t T_, int64_t D) {
  if (T_ <= 0 || D <= 0) return 256;
  return align_up((size_t)bwd_rows(T_) * 2 * D * 4, 256);
}

extern "C" int mega_row_norm_bwd(const void* dy, const void* x, int64_t x_stride, const void* weight, const void* add, void* dx,
                                 void* dw, void* db, int dtype, int kind, int64_t T_, int64_t D, double eps, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  MEGA_REQUIRE(mega_row_norm_covers(dtype, D) && T_ > 0 && (kind == MEGA_TOKEN_RMSNORM || kind == MEGA_TOKEN_LAYERNORM),
               MEGA_ERR_UNSUPPORTED, "row_norm_bwd: D=%ld, dtype %d", (long)D, dtype);
  const int es = dtype == MEGA_F32 ? 4 : 2;
  MEGA_REQUIRE(dy && x && dx && x_stride * es % 16 == 0 &&
                   (((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dx | (uintptr_t)weight | (uintptr_t)add) % 16) == 0,
               MEGA_ERR_ARG, "row_norm_bwd: null or unaligned rows");
  const size_t need = mega_row_norm_bwd_workspace_bytes(T_, D);
  MEGA_REQUIRE(workspace && workspace_bytes >= need, MEGA_ERR_WORKSPACE, "row_norm_bwd: workspace of %zu bytes needed", need);
  if (audit_on()) {
    audit_use(workspace, need, "row_norm_bwd: partial sums");
    audit_use(dy, (size_t)T_ * D * es, "row_norm_bwd: dy");
    audit_use(x, (size_t)((T_ - 1) * x_stride + D) * es, "row_norm_bwd: x");
    audit_use(dx, (size_t)T_ * D * es, "row_norm_bwd: dx");
    return MEGA_OK;
  }
  hipStream_t s = (hipStream_t)stream;
  const bool ln = kind == MEGA_TOKEN_LAYERNORM;
  float* part = (float*)workspace;
#define MEGA_D(T)                                                                                              \
  return ln ? launch_bwd<T, true>(dy, x, x_stride, weight, add, dx, dw, db, T_, D, (float)eps, part, s)        \
            : launch_bwd<T, false>(dy, x, x_stride, weight, add, dx, dw, nullptr, T_, D, (float)eps, part, s)
  if (dtype == MEGA_F32) MEGA_D(float);
  if (dtype == MEGA_BF16) MEGA_D(bf16_t);
  MEGA_D(f16_t);
#undef MEGA_D
}

extern "C" size_t mega_sum_rows_workspace_bytes(int dtype, int64_t T_, int64_t W) {
  if (T_ <= 0 || W <= 0) return 256;
  return align_up((size_t)ceil_div(T_, slab_rows(T_, W, dtype == MEGA_F32 ? 4 : 8)) * W * 4, 256);
}

// sums over the tokens of dy (x = NULL), or of dx = dy silu'(x), which is written as well
extern "C" int mega_sum_rows(const void* dy, int64_t row_stride, const void* x, void* dx, int dtype, int64_t T_, int64_t W,
                             void* out, void* workspace, size_t workspace_bytes, void* stream) {
  MEGA_REQUIRE(dtype == MEGA_F32 || dtype == MEGA_BF16 || dtype == MEGA_F16, MEGA_ERR_ARG, "sum_rows: unknown dtype %d", dtype);
  const int es = dtype == MEGA_F32 ? 4 : 2, vec = 16 / es;
  MEGA_REQUIRE(T_ > 0 && W > 0 && W % vec == 0 && row_stride % vec == 0 && W < (int64_t)1 << 30, MEGA_ERR_UNSUPPORTED,
               "sum_rows: rows must be whole 16-byte pieces (W=%ld)", (long)W);
  MEGA_REQUIRE(dy && out && (x == nullptr) == (dx == nullptr) && (((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dx) % 16) == 0,
               MEGA_ERR_ARG, "sum_rows: null or unaligned pointer");
  const size_t need = mega_sum_rows_workspace_bytes(dtype, T_, W);
  MEGA_REQUIRE(workspace && workspace_bytes >= need, MEGA_ERR_WORKSPACE, "sum_rows: workspace of %zu bytes needed", need);
  const int slab = slab_rows(T_, W, vec);
  const dim3 grid((unsigned)ceil_div(W, 64 * vec), (unsigned)ceil_div(T_, slab));
  MEGA_REQUIRE(ceil_div(T_, slab) <= 65535, MEGA_ERR_UNSUPPORTED, "sum_rows: too many rows");
  hipStream_t s = (hipStream_t)stream;
  float* part = (float*)workspace;
#define MEGA_D(T, V)                                                                                                       \
  {                                                                                                                        \
    if (x)                                                                                                                 \
      hipLaunchKernelGGL((sum_rows_kernel<T, V, true>), grid, dim3(kThreads), 0, s, (const T*)dy, row_stride, (const T*)x,  \
                         (T*)dx, part, T_, (int)W, slab);                                                                  \
    else                                                                                                                   \
      hipLaunchKernelGGL((sum_rows_kernel<T, V, false>), grid, dim3(kThreads), 0, s, (const T*)dy, row_stride,             \
                         (const T*)nullptr, (T*)nullptr, part, T_, (int)W, slab);                                          \
    MEGA_CHECK_LAUNCH("sum_rows");                                                                                         \
    return finish<T>(part, (int)grid.y, (int)W, (int)W, out, nullptr, s);                                                  \
  }
  if (dtype == MEGA_F32) MEGA_D(float, 4)
  if (dtype == MEGA_BF16) MEGA_D(bf16_t, 8)
  MEGA_D(f16_t, 8)
#undef MEGA_D
}
