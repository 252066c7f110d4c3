// One token of every stream through a layer with carried state (incremental_state with one new position:
// fairseq/modules/moving_average_gated_attention.py:263-417, normalized_feedforward_network.py:77-93,
// models/mega_lm.py:313-386), 16-bit activations.
//
// A step of few streams reads every weight once and does almost no arithmetic: what bounds it is the stream of
// weights and cached keys / values from memory (the 27 MB of a layer of 1024 channels: 6 us at this card's copy
// rate) and, in practice, the number of launches in a row.  So the chain is cut at the points where a value needs all
// channels of the one before, and everything in between rides along:
//   norm_ema_token   TimestepNorm of one token, moving-average state update       (decode.hip, with the padding mask)
//   token_linear     up to two projections per launch (v and mx): normalisation of the input row while it is staged,
//                    bias, silu, residual or the output gate while the result leaves
//   token_attention  q, k of the new token, scores against the cached keys of one block of positions, its share of
//                    the weighted sum of values; the same pass writes the grown key / value cache
//   token_combine    adds the blocks up, applies the r gate
// 7 launches per layer where the same step as separate operators took about 45: two layers of 1024 channels, one stream
// behind 700 cached positions: 19 launches, 111 us of device time and 183 us per token with the host's work, where the
// operators one by one took 97 launches, 338 us and 1230 us.  40 streams behind 900 positions: 345 us of device time, half
// of it the copy of the key / value cache (330 MB at 3.5 TB/s).
#include "common.h"

namespace mega {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

template <typename T>
__device__ __forceinline__ f32x4 mfma16(uint4 a, uint4 b, f32x4 c);
template <>
__device__ __forceinline__ f32x4 mfma16<bf16_t>(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16<f16_t>(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ float silu_f(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }
__device__ __forceinline__ float sigmoid_f(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// ---------------------------------------------------------------------------------------------
// out[b, n] = epilogue(sum_k W[n, k] prologue(x[b])[k] + bias[n]) for B <= 64 tokens.  A workgroup of 8 waves owns 16
// rows of W; the waves share the reduction (a wave takes every eighth 64-element piece, so the two loads of a lane
// finish a row's 128-byte line), W goes straight from memory into the matrix instruction's A operand (every byte is
// used once: LDS would only add a trip), the tokens are its columns, 16 per tile and MT tiles.  The eight partial
// tiles meet in LDS.  16 rows per workgroup: 64 to 400 workgroups at the layer's widths; 32 rows left half the CUs
// without work on the narrow projections.
constexpr int kLinWaves = 8, kLinThreads = 64 * kLinWaves;

// one wave: dst = prologue(src), a row of K values
template <typename T>
__device__ __forceinline__ void normalise_row(const MegaTokenLinear& P, const T* src, T* dst, int K, int lane) {
  float s = 0.f, ss = 0.f;
  for (int c = lane * 8; c < K; c += 512) {
    const Vec<T, 8> v = *(const Vec<T, 8>*)(src + c);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = to_float(v.v[e]);
      s += f;
      ss = fmaf(f, f, ss);
    }
  }
  float mu = 0.f, rs = 1.f;
  if (P.prologue == MEGA_TOKEN_RMSNORM) {
    rs = rsqrtf(wave_sum(ss) / (float)K + P.eps);
  } else if (P.prologue == MEGA_TOKEN_LAYERNORM) {
    mu = wave_sum(s) / (float)K;
    float q = 0.f;                                // centred: the row is in the cache, a second read costs nothing
    for (int c = lane * 8; c < K; c += 512) {
      const Vec<T, 8> v = *(const Vec<T, 8>*)(src + c);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = to_float(v.v[e]) - mu;
        q = fmaf(d, d, q);
      }
    }
    rs = rsqrtf(wave_sum(q) / (float)K + P.eps);
  }
  const T* nw = (const T*)P.norm_weight;
  const T* nb = (const T*)P.norm_bias;
  for (int c = lane * 8; c < K; c += 512) {
    const Vec<T, 8> v = *(const Vec<T, 8>*)(src + c);
    Vec<T, 8> o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = to_float(v.v[e]);
      float r;
      if (P.prologue == MEGA_TOKEN_SILU) {
        r = silu_f(f);
      } else {
        r = (f - mu) * rs;
        if (nw) r *= to_float(nw[c + e]) + 1.0f;              // weights are stored as offsets from one
        if (nb) r += to_float(nb[c + e]);
      }
      o.v[e] = from_float<T>(r);
    }
    *(Vec<T, 8>*)(dst + c) = o;
  }
}

// the same into memory, one wave per row (rows of K values, contiguous)
template <typename T>
__global__ __launch_bounds__(64) void token_rows_kernel(const MegaTokenLinear P) {
  const int b = blockIdx.x, K = (int)P.K;
  normalise_row<T>(P, (const T*)P.x + (size_t)b * P.x_stride, (T*)P.scratch + (size_t)b * K, K, threadIdx.x);
}

template <typename T, int MT>
__global__ __launch_bounds__(kLinThreads) void token_linear_kernel(const MegaTokenLinear P0, const MegaTokenLinear P1,
                                                                   int blocks0, int B) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const bool second = (int)blockIdx.x >= blocks0;
  const MegaTokenLinear& P = second ? P1 : P0;
  const int n0 = ((int)blockIdx.x - (second ? blocks0 : 0)) * 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int K = (int)P.K, N = (int)P.N;
  const int n = lane & 15, g = lane >> 4;
  const T* W = (const T*)P.weight + (size_t)min(n0 + n, N - 1) * K + 8 * g;
  const int xp = K * 2 + 16;                      // LDS pitch of a staged token row: the 16 tokens of a fragment read
                                                  // start on different banks
  const int npc = (K + 63) / 64;                  // 64-element pieces of the reduction
  // a wave's pieces in batches of PB: a whole batch of loads is in flight while the one before is multiplied, the
  // first one while the input row is normalised (K <= 2048 is one batch: one trip to memory per launch)
  constexpr int PB = 4;
  uint4 w[2 * PB];
  auto load_w = [&](int pc0) {
#pragma unroll
    for (int u = 0; u < PB; ++u) {
      const int pc = pc0 + u * kLinWaves;
      w[2 * u] = w[2 * u + 1] = make_uint4(0, 0, 0, 0);
      if (pc < npc) {
        w[2 * u] = *(const uint4*)(W + pc * 64);
        if (pc * 64 + 32 < K) w[2 * u + 1] = *(const uint4*)(W + pc * 64 + 32);
      }
    }
  };
  load_w(wave);
  if (P.prologue) {
    for (int b = wave; b < B; b += kLinWaves)
      normalise_row<T>(P, (const T*)P.x + (size_t)b * P.x_stride, (T*)(lds + (size_t)b * xp), K, lane);
    __syncthreads();
  }
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // token rows of this lane's columns (rows past the last stream repeat it; their results are dropped)
  const char* xrow[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int b = min(16 * t + n, B - 1);
    xrow[t] = P.prologue ? lds + (size_t)b * xp + 16 * g
                         : (const char*)((const T*)P.x + (size_t)b * P.x_stride + 8 * g);
  }
  for (int pc0 = wave; pc0 < npc; pc0 += PB * kLinWaves) {
    uint4 a[2 * PB];
#pragma unroll
    for (int u = 0; u < 2 * PB; ++u) a[u] = w[u];
    if (pc0 + PB * kLinWaves < npc) load_w(pc0 + PB * kLinWaves);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      uint4 x[2 * PB];
#pragma unroll
      for (int u = 0; u < PB; ++u) {
        const int pc = pc0 + u * kLinWaves;
        x[2 * u] = x[2 * u + 1] = make_uint4(0, 0, 0, 0);
        if (pc < npc) {
          x[2 * u] = *(const uint4*)(xrow[t] + pc * 128);
          if (pc * 64 + 32 < K) x[2 * u + 1] = *(const uint4*)(xrow[t] + pc * 128 + 64);
        }
      }
#pragma unroll
      for (int u = 0; u < 2 * PB; ++u) acc[t] = mfma16<T>(a[u], x[u], acc[t]);
    }
  }
  // partial tiles: [wave][MT][16 tokens][16 rows] fp32 in LDS (the staged rows are no longer read)
  __syncthreads();
  float* red = (float*)lds;
#pragma unroll
  for (int t = 0; t < MT; ++t)                    // D: column (token) lane & 15, rows 4 g + {0..3}
    *(f32x4*)(red + ((wave * MT + t) * 16 + n) * 20 + 4 * g) = acc[t];
  __syncthreads();
  for (int i = tid; i < MT * 256; i += kLinThreads) {
    const int t = i >> 8, b = 16 * t + ((i >> 4) & 15), r = i & 15;
    const int row = n0 + r;
    if (b >= B || row >= N) continue;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kLinWaves; ++w) v += red[((w * MT + t) * 16 + ((i >> 4) & 15)) * 20 + r];
    if (P.bias) v += to_float(((const T*)P.bias)[row]);
    if (P.epilogue == MEGA_TOKEN_SILU) {
      v = silu_f(v);
    } else if (P.epilogue == MEGA_TOKEN_RESIDUAL) {
      if (P.scale) v *= to_float(((const T*)P.scale)[row]);
      v += to_float(((const T*)P.residual)[(size_t)b * P.residual_stride + row]);
    } else if (P.epilogue == MEGA_TOKEN_GATE) {
      const float res = to_float(((const T*)P.residual)[(size_t)b * P.residual_stride + row]);
      const float u = to_float(((const T*)P.gate_u)[(size_t)b * P.gate_stride + row]);
      const float hx = to_float(((const T*)P.gate_hx)[(size_t)b * P.gate_stride + row]);
      v = res + sigmoid_f(u) * (silu_f(hx + v) - res);
    }
    ((T*)P.out)[(size_t)b * P.out_stride + row] = from_float<T>(v);
  }
}

// ---------------------------------------------------------------------------------------------
// Attention of one new token per stream.  A workgroup owns (stream, head, block of SL positions, slab of value
// columns): it forms q (rotated to its position) and the new key from z, takes the scores of its positions, their
// exponentials against the block's own maximum, and the weighted sum of its value slab; the same pass copies the keys
// and values it has just read into the grown cache.  Blocks of positions and slabs exist to fill the chip for a single
// stream; the score work repeated per slab is small (z / heads against hidden / heads columns).
constexpr int kAttnThreads = 256;
constexpr int kMaxHd = 512;            // z features per head
constexpr int kSlab = 512;             // value columns per workgroup

struct TokAttn {
  const void* base;      // [B, W] projection rows; z at column zoff
  int64_t base_stride;
  int64_t zoff;
  const void* v_new;     // [B, hidden]
  const void* k_old;     // [B, n, S] or null
  const void* v_old;     // [B, n, hidden]
  void* k_out;           // [B, n + 1, S] or null: the cache is not kept
  void* v_out;
  const void* gamma;     // [2, S] offsets from one, [2, S]
  const void* beta;
  const float* cis;      // [>= n + 1, S / heads / 2, 2]: cos, sin of position x frequency
  float* part_o;         // [B, Nh, splits, hd]
  float* part_ml;        // [B, Nh, splits, 2]
  int64_t k_row, k_batch;
  int B, n, S, Nh, hidden, SL, splits, slabs;
};

template <typename T>
__global__ __launch_bounds__(kAttnThreads) void token_attention_kernel(const TokAttn A) {
  __shared__ float s_q[kMaxHd], s_k[kMaxHd], s_p[256], s_red[8];
  __shared__ float s_o[4][kSlab];
  int id = blockIdx.x;
  const int slab = id % A.slabs;
  id /= A.slabs;
  const int sp = id % A.splits;
  id /= A.splits;
  const int h = id % A.Nh, b = id / A.Nh;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int Hd = A.S / A.Nh, hd = A.hidden / A.Nh, half = Hd / 2;
  const int j0 = sp * A.SL, j1 = min(j0 + A.SL, A.n + 1);       // positions of this block; n is the new token
  // ---- the block's first keys and value rows are on their way before anything else
  // scores: a group of LG lanes (a power of two) per position, 8 features per lane (at most 512 per head)
  const int vecs = Hd / 8;
  int lgs = 0;
  while ((1 << lgs) < vecs) ++lgs;
  const int LG = 1 << lgs, per = 64 >> lgs;                    // positions per wave and step
  const int sub = lane & (LG - 1), grp = lane >> lgs;
  constexpr int UK = 4;                                        // steps in flight
  Vec<T, 8> kr[UK];
  auto load_k = [&](int jb) {
#pragma unroll
    for (int u = 0; u < UK; ++u) {
      const int j = jb + (u * 4 + wave) * per + grp;
      if (j < min(j1, A.n) && sub < vecs)
        kr[u] = *(const Vec<T, 8>*)((const T*)A.k_old + b * A.k_batch + j * A.k_row + h * Hd + 8 * sub);
    }
  };
  // values: 64 lanes x 8 columns cover a slab of 512; narrower heads put several positions side by side
  const int c0 = slab * kSlab, cols = min(kSlab, hd - c0), cv = cols / 8;
  int cls = 0;
  while ((1 << cls) < cv) ++cls;
  const int CL = 1 << cls, kper = 64 >> cls;
  const int cl = lane & (CL - 1), kg = lane >> cls;
  const T* vo = (const T*)A.v_old + (size_t)b * A.n * A.hidden + h * hd + c0 + 8 * cl;
  const T* vn = (const T*)A.v_new + (size_t)b * A.hidden + h * hd + c0 + 8 * cl;
  constexpr int UV = 8;                                        // rows in flight
  Vec<T, 8> vr[UV];
  auto load_v = [&](int jb) {
#pragma unroll
    for (int u = 0; u < UV; ++u) {
      const int j = jb + u * 4 * kper;
      if (j < j1 && cl < cv) vr[u] = *(const Vec<T, 8>*)(j < A.n ? vo + (size_t)j * A.hidden : vn);
    }
  };
  load_k(j0);
  load_v(j0 + wave * kper + kg);
  // ---- q and the new key of this head
  const T* z = (const T*)A.base + (size_t)b * A.base_stride + A.zoff;
  float ss = 0.f;
  for (int c = tid; c < A.S; c += kAttnThreads) {
    const float f = to_float(z[c]);
    ss = fmaf(f, f, ss);
  }
  ss = wave_sum(ss);
  if (lane == 0) s_red[wave] = ss;
  __syncthreads();
  const float inv = 1.0f / fmaxf(sqrtf(s_red[0] + s_red[1] + s_red[2] + s_red[3]), 1e-5f);
  const T* ga = (const T*)A.gamma;
  const T* be = (const T*)A.beta;
  for (int i = tid; i < half; i += kAttnThreads) {
    const int f = h * Hd + 2 * i;
    const float z0 = to_float(z[f]) * inv, z1 = to_float(z[f + 1]) * inv;
    const float q0 = fmaf(z0, to_float(ga[f]) + 1.f, to_float(be[f]));
    const float q1 = fmaf(z1, to_float(ga[f + 1]) + 1.f, to_float(be[f + 1]));
    const float k0 = fmaf(z0, to_float(ga[A.S + f]) + 1.f, to_float(be[A.S + f]));
    const float k1 = fmaf(z1, to_float(ga[A.S + f + 1]) + 1.f, to_float(be[A.S + f + 1]));
    const float2 cs = *(const float2*)(A.cis + ((size_t)A.n * half + i) * 2);
    s_q[2 * i] = q0 * cs.x - q1 * cs.y;
    s_q[2 * i + 1] = q0 * cs.y + q1 * cs.x;
    s_k[2 * i] = to_float(from_float<T>(k0));                  // the cache holds keys in the activation type, unrotated
    s_k[2 * i + 1] = to_float(from_float<T>(k1));
  }
  __syncthreads();
  // ---- scores
  for (int jb = j0; jb < j1; jb += 4 * per * UK) {
    if (jb > j0) load_k(jb);
#pragma unroll
    for (int u = 0; u < UK; ++u) {
      if (jb + u * 4 * per >= j1) break;                       // uniform
      const int j = jb + (u * 4 + wave) * per + grp;
      float acc = 0.f;
      if (j < j1 && sub < vecs) {
        Vec<T, 8> kv = kr[u];
        if (j == A.n)
#pragma unroll
          for (int e = 0; e < 8; ++e) kv.v[e] = from_float<T>(s_k[8 * sub + e]);
        if (A.k_out && slab == 0)
          *(Vec<T, 8>*)((T*)A.k_out + ((size_t)b * (A.n + 1) + j) * A.S + h * Hd + 8 * sub) = kv;
        const float4* cs = (const float4*)(A.cis + ((size_t)j * half + 4 * sub) * 2);
        const float4 r0 = cs[0], r1 = cs[1];
        const float cc[4] = {r0.x, r0.z, r1.x, r1.z}, sn[4] = {r0.y, r0.w, r1.y, r1.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float k0 = to_float(kv.v[2 * e]), k1 = to_float(kv.v[2 * e + 1]);
          const float q0 = s_q[8 * sub + 2 * e], q1 = s_q[8 * sub + 2 * e + 1];
          acc = fmaf(cc[e], fmaf(k0, q0, k1 * q1), acc);       // (R k) . q with the rotation folded into the two products
          acc = fmaf(sn[e], fmaf(k0, q1, -k1 * q0), acc);
        }
      }
      for (int o = LG >> 1; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
      if (sub == 0 && j < j1) s_p[j - j0] = acc;
    }
  }
  __syncthreads();
  // ---- the block's maximum and exponentials (every wave for itself: at most 256 positions)
  float m = -INFINITY;
  for (int j = lane; j < j1 - j0; j += 64) m = fmaxf(m, s_p[j]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  float l = 0.f;
  for (int j = lane; j < j1 - j0; j += 64) l += __expf(s_p[j] - m);
  l = wave_sum(l);
  const size_t pr = ((size_t)b * A.Nh + h) * A.splits + sp;
  if (slab == 0 && tid == 0) {
    A.part_ml[pr * 2] = m;
    A.part_ml[pr * 2 + 1] = l;
  }
  // ---- values
  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
  T* vd = (T*)A.v_out + (size_t)b * (A.n + 1) * A.hidden + h * hd + c0 + 8 * cl;
  for (int j00 = j0; j00 < j1; j00 += 4 * kper * UV) {
    const int jb = j00 + wave * kper + kg;
    if (j00 > j0) load_v(jb);
#pragma unroll
    for (int u = 0; u < UV; ++u) {
      const int j = jb + u * 4 * kper;
      if (j < j1 && cl < cv) {
        if (A.v_out) *(Vec<T, 8>*)(vd + (size_t)j * A.hidden) = vr[u];
        const float p = __expf(s_p[j - j0] - m);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = fmaf(p, to_float(vr[u].v[e]), o[e]);
      }
    }
  }
  for (int s = CL; s < 64; s <<= 1)
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] += __shfl_xor(o[e], s);
  if (kg == 0 && cl < cv)
#pragma unroll
    for (int e = 0; e < 8; ++e) s_o[wave][8 * cl + e] = o[e];
  __syncthreads();
  float* po = A.part_o + pr * hd + c0;
  for (int c = tid; c < cols; c += kAttnThreads) po[c] = (s_o[0][c] + s_o[1][c]) + (s_o[2][c] + s_o[3][c]);
}

// a[b, c] = (sum over blocks e^(m_s - M) O_s[c]) / (sum e^(m_s - M) l_s) * silu(r[b, c]).  A workgroup owns 64 columns
// of a stream (inside one head: a multiple of 8 columns), its four waves share the blocks; the weights are formed once.
template <typename T>
__global__ __launch_bounds__(256) void token_combine_kernel(const float* __restrict__ part_o,
                                                            const float* __restrict__ part_ml, const T* __restrict__ r,
                                                            int64_t r_stride, T* __restrict__ out, int Nh, int splits,
                                                            int hidden, int cblocks) {
  extern __shared__ float s_w[];                  // [splits] weights, then 4 x 64 partial sums
  const int hd = hidden / Nh;
  const int cb = blockIdx.x % cblocks, bh = blockIdx.x / cblocks, h = bh % Nh, b = bh / Nh;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const size_t pr = (size_t)bh * splits;
  float M = -INFINITY, den = 0.f;
  for (int s = lane; s < splits; s += 64) M = fmaxf(M, part_ml[(pr + s) * 2]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
  for (int s = lane; s < splits; s += 64) {
    const float w = __expf(part_ml[(pr + s) * 2] - M);
    den = fmaf(w, part_ml[(pr + s) * 2 + 1], den);
    if (wave == 0) s_w[s] = w;
  }
  den = wave_sum(den);
  __syncthreads();
  const int c = cb * 64 + lane;
  float num = 0.f;
  if (c < hd)
#pragma unroll 4
    for (int s = wave; s < splits; s += 4) num = fmaf(s_w[s], part_o[(pr + s) * hd + c], num);
  float* s_n = s_w + splits;
  s_n[tid] = num;
  __syncthreads();
  if (wave == 0 && c < hd) {
    num = (s_n[lane] + s_n[64 + lane]) + (s_n[128 + lane] + s_n[192 + lane]);
    const size_t col = (size_t)h * hd + c;
    out[(size_t)b * hidden + col] = from_float<T>(num / den * silu_f(to_float(r[(size_t)b * r_stride + col])));
  }
}

int check_linear(const MegaTokenLinear& p, int64_t B, const char* who) {
  MEGA_REQUIRE(p.N > 0 && p.K > 0 && p.K % 32 == 0 && p.N < (int64_t)1 << 26 && p.K <= 65536, MEGA_ERR_UNSUPPORTED,
               "%s: N=%ld, K=%ld (K must be a multiple of 32)", who, (long)p.N, (long)p.K);
  MEGA_REQUIRE(p.weight && p.x && p.out, MEGA_ERR_ARG, "%s: null pointer argument", who);
  MEGA_REQUIRE(p.x_stride % 8 == 0 && ((uintptr_t)p.x % 16) == 0 && ((uintptr_t)p.weight % 16) == 0, MEGA_ERR_UNSUPPORTED,
               "%s: rows must be whole 16-byte pieces", who);
  MEGA_REQUIRE(!p.prologue || B * (p.K * 2 + 16) <= 144 * 1024, MEGA_ERR_UNSUPPORTED,
               "%s: %ld rows of %ld do not fit in LDS with a prologue", who, (long)B, (long)p.K);
  MEGA_REQUIRE(p.epilogue != MEGA_TOKEN_RESIDUAL || p.residual, MEGA_ERR_ARG, "%s: residual missing", who);
  MEGA_REQUIRE(p.epilogue != MEGA_TOKEN_GATE || (p.residual && p.gate_u && p.gate_hx), MEGA_ERR_ARG,
               "%s: gate operands missing", who);
  return MEGA_OK;
}

template <typename T>
int launch_linear(const MegaTokenLinear& p0, const MegaTokenLinear* p1, int64_t B, hipStream_t s) {
  const int blocks0 = (int)ceil_div(p0.N, 16);
  const int blocks = blocks0 + (p1 ? (int)ceil_div(p1->N, 16) : 0);
  const int mt = B <= 16 ? 1 : B <= 32 ? 2 : 4;
  size_t smem = (size_t)kLinWaves * mt * 16 * 20 * 4;
  if (p0.prologue) smem = smem > (size_t)B * (p0.K * 2 + 16) ? smem : (size_t)B * (p0.K * 2 + 16);
  if (p1 && p1->prologue) smem = smem > (size_t)B * (p1->K * 2 + 16) ? smem : (size_t)B * (p1->K * 2 + 16);
  const MegaTokenLinear& q = p1 ? *p1 : p0;
#define MEGA_TL(MT_)                                                                                            \
  {                                                                                                             \
    static uint64_t seen = 0;                                                                                   \
    raise_lds_limit(&seen, 144 * 1024, token_linear_kernel<T, MT_>);                                            \
    hipLaunchKernelGGL((token_linear_kernel<T, MT_>), dim3(blocks), dim3(kLinThreads), smem, s, p0, q, blocks0, (int)B); \
  }
  if (mt == 1) MEGA_TL(1) else if (mt == 2) MEGA_TL(2) else MEGA_TL(4)
#undef MEGA_TL
  MEGA_CHECK_LAUNCH("token_linear");
  return MEGA_OK;
}

// Every workgroup of a projection repeats the normalisation of its input rows.  For one stream that is 1 us under the
// first weights' way from memory and saves a launch; the repetition grows with the rows (40 rows of 1024: 22 us per
// projection on average over a layer's, 11 us without the repetition plus 6 us for the extra launch), so more than
// kFusedRows rows are normalised once, by a launch of their own.
constexpr int64_t kFusedRows = 4;

int linear_dispatch(MegaTokenLinear p0, const MegaTokenLinear* p1, int dtype, int64_t B, hipStream_t s) {
  if (p0.prologue && p0.scratch && B > kFusedRows) {
    MEGA_REQUIRE(p0.x && p0.K > 0 && p0.K % 8 == 0 && p0.x_stride % 8 == 0 && ((uintptr_t)p0.x % 16) == 0 &&
                     ((uintptr_t)p0.scratch % 16) == 0,
                 MEGA_ERR_UNSUPPORTED, "token_linear: rows must be whole 16-byte pieces");
    if (dtype == MEGA_BF16) hipLaunchKernelGGL(token_rows_kernel<bf16_t>, dim3((unsigned)B), dim3(64), 0, s, p0);
    else hipLaunchKernelGGL(token_rows_kernel<f16_t>, dim3((unsigned)B), dim3(64), 0, s, p0);
    p0.prologue = MEGA_TOKEN_NONE;
    p0.x = p0.scratch;
    p0.x_stride = p0.K;
  }
  int rc = check_linear(p0, B, "token_linear");
  if (rc == MEGA_OK && p1) rc = check_linear(*p1, B, "token_linear");
  if (rc != MEGA_OK) return rc;
  return dtype == MEGA_BF16 ? launch_linear<bf16_t>(p0, p1, B, s) : launch_linear<f16_t>(p0, p1, B, s);
}

struct TokenPlan {
  int SL, splits, slabs;
  size_t xn, y, yn, v, base, a, po, ml, total;
};

// Positions per workgroup: 32 while that still leaves CUs idle (a single stream of 700 positions and 2048 columns is
// then 88 workgroups), up to 256 once the streams alone fill the chip twice over.
TokenPlan token_plan(int64_t B, int64_t n, int64_t D, int64_t S, int64_t hidden, int64_t Nh) {
  TokenPlan t;
  const int64_t hd = hidden / Nh;
  t.slabs = (int)ceil_div(hd, kSlab);
  t.SL = 32;
  while (t.SL < 256 && B * Nh * t.slabs * ceil_div(n + 1, t.SL) > 4096) t.SL *= 2;
  t.splits = (int)ceil_div(n + 1, t.SL);
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += align_up(bytes, 256);
    return at;
  };
  t.xn = take((size_t)B * D * 2);
  t.y = take((size_t)B * D * 2);
  t.yn = take((size_t)B * D * 2);
  t.v = take((size_t)B * hidden * 2);
  t.base = take((size_t)B * (2 * D + S + hidden) * 2);
  t.a = take((size_t)B * hidden * 2);
  t.po = take((size_t)B * Nh * t.splits * hd * 4);
  t.ml = take((size_t)B * Nh * t.splits * 8);
  t.total = o;
  return t;
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_token_linear(const MegaTokenLinear* p, int dtype, int64_t B, void* stream) {
  MEGA_REQUIRE(dtype == MEGA_BF16 || dtype == MEGA_F16, MEGA_ERR_UNSUPPORTED, "token_linear: 16-bit activations only");
  MEGA_REQUIRE(p && B >= 0 && B <= 64, MEGA_ERR_ARG, "token_linear: at most 64 rows (B=%ld)", (long)B);
  if (B == 0) return MEGA_OK;
  return linear_dispatch(*p, nullptr, dtype, B, (hipStream_t)stream);
}

extern "C" size_t mega_token_attention_workspace_bytes(int64_t B, int64_t n, int64_t D, int64_t S, int64_t hidden,
                                                       int64_t heads) {
  if (B <= 0 || n < 0 || D <= 0 || S <= 0 || hidden <= 0 || heads <= 0) return 0;
  return token_plan(B, n, D, S, hidden, heads).total;
}

extern "C" int mega_token_gated_attention(const MegaTokenAttention* a, void* stream) {
  MEGA_REQUIRE(a, MEGA_ERR_ARG, "token_gated_attention: null argument");
  const int dtype = (int)a->dtype;
  MEGA_REQUIRE(dtype == MEGA_BF16 || dtype == MEGA_F16, MEGA_ERR_UNSUPPORTED,
               "token_gated_attention: 16-bit activations only");
  const int64_t B = a->B, D = a->D, S = a->S, hidden = a->hidden, Nh = a->heads, n = a->context;
  MEGA_REQUIRE(B > 0 && B <= 64 && D > 0 && S > 0 && hidden > 0 && Nh > 0 && n >= 0 && n <= (int64_t)1 << 20, MEGA_ERR_ARG,
               "token_gated_attention: bad shape");
  MEGA_REQUIRE(D % 32 == 0 && hidden % 32 == 0 && S % Nh == 0 && hidden % Nh == 0 && (S / Nh) % 8 == 0 &&
                   (hidden / Nh) % 8 == 0 && S / Nh <= kMaxHd,
               MEGA_ERR_UNSUPPORTED, "token_gated_attention: widths D=%ld S=%ld hidden=%ld heads=%ld", (long)D, (long)S,
               (long)hidden, (long)Nh);
  MEGA_REQUIRE(a->x && a->out && a->cis && a->gamma && a->beta && (n == 0 || (a->k_old && a->v_old)) &&
                   (!a->k_out == !a->v_out),
               MEGA_ERR_ARG, "token_gated_attention: null pointer argument");
  const TokenPlan t = token_plan(B, n, D, S, hidden, Nh);
  MEGA_REQUIRE(a->workspace && a->workspace_bytes >= (int64_t)t.total, MEGA_ERR_WORKSPACE,
               "token_gated_attention: workspace of %ld bytes needed", (long)t.total);
  const uintptr_t al = (uintptr_t)a->x | (uintptr_t)a->k_old | (uintptr_t)a->v_old | (uintptr_t)a->k_out |
                       (uintptr_t)a->v_out | (uintptr_t)a->workspace | (uintptr_t)a->cis;
  MEGA_REQUIRE(al % 16 == 0, MEGA_ERR_UNSUPPORTED, "token_gated_attention: operands must be 16-byte aligned");
  MEGA_REQUIRE(a->k_row % 8 == 0 && a->k_batch % 8 == 0, MEGA_ERR_UNSUPPORTED,
               "token_gated_attention: cached key rows must be whole 16-byte pieces");
  MEGA_REQUIRE(B * Nh * t.splits * t.slabs < (int64_t)1 << 31, MEGA_ERR_UNSUPPORTED, "token_gated_attention: too large");
  char* ws = (char*)a->workspace;
  hipStream_t s = (hipStream_t)stream;
  // TimestepNorm of the token and the moving average's state update
  int rc = norm_ema_token(a->x, ws + t.xn, ws + t.y, dtype, a->mask, a->prev_count, a->prev_mean, a->prev_var, a->count,
                          a->mean, a->var, a->norm_gamma, a->norm_beta, a->norm_eps, a->p, a->q, a->ema_gamma, a->omega,
                          a->h_in, a->h_out, B, D, a->groups, a->states, s);
  if (rc != MEGA_OK) return rc;
  // v = silu(Wv xn + bv) and the four-way projection of the activated moving average, one launch
  const int64_t W = 2 * D + S + hidden;
  MegaTokenLinear pv = {}, pm = {}, ph = {};
  pv.weight = a->v_weight; pv.bias = a->v_bias; pv.x = ws + t.xn; pv.x_stride = D; pv.out = ws + t.v;
  pv.out_stride = hidden; pv.N = hidden; pv.K = D; pv.epilogue = MEGA_TOKEN_SILU;
  pm.weight = a->mx_weight; pm.bias = a->mx_bias; pm.x = ws + t.y; pm.x_stride = D; pm.out = ws + t.base;
  pm.out_stride = W; pm.N = W; pm.K = D; pm.prologue = (int)a->move_act; pm.norm_weight = a->move_norm_weight;
  pm.eps = (float)a->move_norm_eps; pm.scratch = ws + t.yn;
  rc = linear_dispatch(pm, &pv, dtype, B, s);
  if (rc != MEGA_OK) return rc;
  TokAttn A;
  A.base = ws + t.base; A.base_stride = W; A.zoff = D; A.v_new = ws + t.v; A.k_old = a->k_old; A.v_old = a->v_old;
  A.k_out = a->k_out; A.v_out = a->v_out; A.gamma = a->gamma; A.beta = a->beta; A.cis = a->cis;
  A.part_o = (float*)(ws + t.po); A.part_ml = (float*)(ws + t.ml); A.B = (int)B; A.n = (int)n; A.S = (int)S;
  A.k_row = a->k_row; A.k_batch = a->k_batch;
  A.Nh = (int)Nh; A.hidden = (int)hidden; A.SL = t.SL; A.splits = t.splits; A.slabs = t.slabs;
  const int cblocks = (int)ceil_div(hidden / Nh, 64);
  const size_t csmem = (size_t)(t.splits + 256) * 4;
  const dim3 grid((unsigned)(B * Nh * t.splits * t.slabs)), cgrid((unsigned)(B * Nh * cblocks));
  const size_t roff = (size_t)(D + S) * 2;
  if (dtype == MEGA_BF16) {
    hipLaunchKernelGGL(token_attention_kernel<bf16_t>, grid, dim3(kAttnThreads), 0, s, A);
    hipLaunchKernelGGL(token_combine_kernel<bf16_t>, cgrid, dim3(256), csmem, s, A.part_o, A.part_ml,
                       (const bf16_t*)(ws + t.base + roff), W, (bf16_t*)(ws + t.a), (int)Nh, t.splits, (int)hidden, cblocks);
  } else {
    hipLaunchKernelGGL(token_attention_kernel<f16_t>, grid, dim3(kAttnThreads), 0, s, A);
    hipLaunchKernelGGL(token_combine_kernel<f16_t>, cgrid, dim3(256), csmem, s, A.part_o, A.part_ml,
                       (const f16_t*)(ws + t.base + roff), W, (f16_t*)(ws + t.a), (int)Nh, t.splits, (int)hidden, cblocks);
  }
  MEGA_CHECK_LAUNCH("token_gated_attention");
  // output projection, output activation and the residual mix
  ph.weight = a->h_weight; ph.x = ws + t.a; ph.x_stride = hidden; ph.out = a->out; ph.out_stride = D; ph.N = D;
  ph.K = hidden; ph.epilogue = MEGA_TOKEN_GATE; ph.residual = a->x; ph.residual_stride = D; ph.gate_u = ws + t.base;
  ph.gate_hx = ws + t.base + (size_t)(D + S + hidden) * 2; ph.gate_stride = W;
  return linear_dispatch(ph, nullptr, dtype, B, s);
}
