// 16-bit attention with its weights in memory: the weights (below), and the long products y = P v, dv = w^T dy, and dS, whose
// epilogue is the softmax's backward (fairseq/csrc/ops/attention_kernel.cu:40-131, 155-203).  The products: tall tiles of gemm16_wide.h (256 x 128, memory straight to
// LDS, two groups of waves in turn), one product per (row, head).
//
// What bounds them: the number of tiles and the turns they are taken in.  16 waves on 256 x 256 with register staging had 80 tiles
// at the diagonal and below for 256 compute units (8 entries of 1024 x 1024), and their reads, products and LDS writes ran in step.
// Half as wide tiles are 160; only those that hold a pair are launched, the longest reductions first across all entries of an
// XCD.  us before and now, entries x positions x width:    dS          y = P v      dv = w^T dy
//                                    8 x 1024 x 2048    67.9, 36.7    45.1, 30.7    43.7, 28.7
//                                   16 x 2048 x 1024     154,  116         -        98.8, 87.2
#include "attention_wide.h"
#include "gemm16_wide.h"

namespace mega {
namespace {

// A wave's part of dS.  EDGE: rows or columns beyond the matrix.
template <typename T, bool EDGE, int FM, int FN>
__device__ __forceinline__ void store_score_grad(const AttnWideP& P, const T* E, T* C, const float* rowdot, int m0, int n0, int lane,
                                                 const f32x4 (&acc)[FM][FN]) {
  const int g = lane >> 4, own = n0 + g * 4, mine = n0 + (g & 1) * 16 + (g >> 1) * 8;
  const int seen = P.causal ? 0 : P.N;                 // columns up to m + seen take part
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + i * 16 + (lane & 15), mr = EDGE ? min(m, P.M - 1) : m;
    const T* e = E + (int64_t)mr * P.lde;
    const float dot = rowdot[mr];
#pragma unroll
    for (int j = 0; j < FN; j += 2) {
      uint32_t q[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = own + (j + h) * 16;
        const Vec<T, 4> w = *(const Vec<T, 4>*)(e + (EDGE ? min(n, P.N - 4) : n));
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float d = P.alpha * to_float(w.v[u]) * (acc[i][j + h][u] - dot);
          v[u] = n + u <= m + seen ? d : 0.f;
        }
        q[2 * h] = pack16<T>(v[0], v[1]);
        q[2 * h + 1] = pack16<T>(v[2], v[3]);
      }
      const uint4 x = eight(q);
      if (!EDGE || (m < P.M && mine + j * 16 < P.N)) *(uint4*)(C + (int64_t)m * P.ldc + mine + j * 16) = x;   // (N % 8 == 0)
    }
  }
}

// A workgroup's tile: batch entry, rows, columns
template <AttnWide KIND, int TN>
__device__ __forceinline__ void attn_place(const AttnWideP& P, int& z, int& m0, int& n0) {
  const int x = P.xcd ? (int)blockIdx.x & 7 : 0, id = P.xcd ? (int)blockIdx.x >> 3 : (int)blockIdx.x;
  if constexpr (KIND == kScoreGrad) {
    // (equal reductions: entry by entry)
    const int e = id / P.tiles;
    int t = id - e * P.tiles, i = 0;
    z = P.xcd ? e * 8 + x : e;
    if (P.causal) {
      constexpr int wide = kWideM / TN;                // tiles that a row of tiles has more than the one above
      while (t >= (i + 1) * wide) t -= ++i * wide;
    } else {
      i = t / P.nt;
      t -= i * P.nt;
    }
    m0 = i * kWideM;
    n0 = t * TN;
  } else {
    const int here = P.xcd ? P.batches >> 3 : P.batches, row = here * P.nt;
    const int i = id / row, r = id - i * row, e = r / P.nt;
    z = P.xcd ? e * 8 + x : e;
    m0 = (KIND == kValueGrad ? i : P.mt - 1 - i) * kWideM;
    n0 = (r - e * P.nt) * TN;
  }
}

template <typename T, AttnWide KIND, bool RAG>
__global__ __launch_bounds__(512, 2) void attn_wide_kernel(const AttnWideP P) {
  constexpr bool KA = KIND == kValueGrad, KB = KIND != kScoreGrad;
  using K = Tall<T, KA, KB, RAG>;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int z, m0, n0;
  attn_place<KIND, K::TN>(P, z, m0, n0);
  const int zo = z / P.nin, zi = z - zo * P.nin;
  const T* A = (const T*)P.A + zo * P.sa + zi * P.sai;
  const T* B = (const T*)P.B + zo * P.sb + zi * P.sbi;
  T* C = (T*)P.C + zo * P.sc + zi * P.sci;
  const int kb = KIND == kValueGrad && P.causal ? m0 : 0, ke = KIND == kValues && P.causal ? min(P.K, m0 + kWideM) : P.K;
  const int wm = (wave / K::WN) * K::FM, wn = (wave % K::WN) * K::FN;
  const char* ta = (const char*)(A + (KA ? (int64_t)kb * P.lda + m0 : (int64_t)m0 * P.lda + kb));
  const char* tb = (const char*)(B + (KB ? (int64_t)kb * P.ldb + n0 : (int64_t)n0 * P.ldb + kb));
  f32x4 acc[K::FM][K::FN];
  K::sums(lds, ta, tb, P.lda, P.ldb, P.M - m0, P.N - n0, ke - kb, tid, wm, wn, acc);
  const bool whole = m0 + kWideM <= P.M && n0 + K::TN <= P.N;
  if constexpr (KIND == kScoreGrad) {
    const T* E = (const T*)P.E + zo * P.se + zi * P.sei;
    const float* dot = P.rowdot + (int64_t)z * P.M;
    if (whole) store_score_grad<T, false>(P, E, C, dot, m0 + wm * 16, n0 + wn * 16, lane, acc);
    else store_score_grad<T, true>(P, E, C, dot, m0 + wm * 16, n0 + wn * 16, lane, acc);
  } else {
    Gemm16P G = {};
    G.C = C;
    G.ldc = P.ldc;
    G.M = P.M;
    G.N = P.N;
    Place at = {};
    at.m0 = m0;
    at.n0 = n0;
    if (whole) store_wave<T, false, 0, false>(G, at, wm, wn, lane, acc);
    else store_wave<T, false, 0, true>(G, at, wm, wn, lane, acc);
  }
}

template <typename T, AttnWide KIND, bool RAG>
void launch(const AttnWideP& P, hipStream_t s) {
  using K = Tall<T, KIND == kValueGrad, KIND != kScoreGrad, RAG>;
  static uint64_t seen = 0;
  const auto kern = attn_wide_kernel<T, KIND, RAG>;
  raise_lds_limit(&seen, K::kLds, kern);
  hipLaunchKernelGGL(kern, dim3((unsigned)(P.tiles * P.batches)), dim3(K::kWT), K::kLds, s, P);
}
template <typename T>
void launch_kind(const AttnWideP& P, AttnWide kind, hipStream_t s) {
  const bool rag = P.K % kKS != 0;
  if (kind == kScoreGrad) rag ? launch<T, kScoreGrad, true>(P, s) : launch<T, kScoreGrad, false>(P, s);
  else if (kind == kValues) rag ? launch<T, kValues, true>(P, s) : launch<T, kValues, false>(P, s);
  else rag ? launch<T, kValueGrad, true>(P, s) : launch<T, kValueGrad, false>(P, s);
}

// tiles of a batch entry
int64_t entry_tiles(const AttnWideP& P, AttnWide kind) {
  const int64_t mt = ceil_div(P.M, kWideM), nt = ceil_div(P.N, 128);
  if (kind != kScoreGrad || !P.causal) return mt * nt;
  // (square; the last row of tiles is one short where its second tile lies beyond the matrix)
  return mt * (mt + 1) - (nt < 2 * mt ? 1 : 0);
}

// ---- the weights, without the fp32 scores in memory.
//
// A workgroup owns 64 queries of a batch entry, in registers as the matrix instruction's columns; its waves take tiles of 64 keys
// in turn, fragments straight from memory (k fits an L2).  Scores are formed twice: for the rows' maxima and
// sums, which the waves exchange once through LDS, and for the weights.  Both are 32-bit throughout, as they were between the
// three passes over the scores.  What bounds it is a wave's turn (fragments on their way, products, exponentials one after the
// other) and the writing: 16 x 2048 x 2048 in bf16, 134 MB, 49 us (85 as product and softmax).
constexpr int kQBlocks = 4;
template <typename T, int KS>
__global__ __launch_bounds__(256, 2) void attn_weights_kernel(const AttnWeightsP A) {
  constexpr int FQ = kQBlocks, KB = 4, NW = 4, BQ = 16 * FQ, BK = 16 * KB;   // blocks of queries, of keys; waves
  __shared__ float2 stat[NW][BQ];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // longest rows first, the shortest of them last beside them: two workgroups of a compute unit have about the same keys
  const int x = A.xcd ? (int)blockIdx.x & 7 : 0, id = A.xcd ? (int)blockIdx.x >> 3 : (int)blockIdx.x;
  const int here = A.xcd ? A.batches >> 3 : A.batches, total = here * A.qt, half = (total + 1) >> 1;
  const int o = id < half ? id : total - 1 - (id - half);
  const int z = (o % here) * (A.xcd ? 8 : 1) + x, q0 = (A.qt - 1 - o / here) * BQ;
  const int b = z / A.Nh, h = z - b * A.Nh;
  const int64_t rs = (int64_t)A.Nh * A.H1, base = (int64_t)b * A.L * rs + (int64_t)h * A.H1;
  const T* const Q = (const T*)A.q + base;
  const T* const Kp = (const T*)A.k + base;
  T* const P = (T*)A.P + (int64_t)z * A.L * A.L;
  uint4 fq[FQ][KS];
#pragma unroll
  for (int j = 0; j < FQ; ++j)
#pragma unroll
    for (int s = 0; s < KS; ++s) fq[j][s] = *(const uint4*)(Q + min(q0 + 16 * j + n, A.L - 1) * rs + s * 32 + g * 8);
  const int seen = A.causal ? min(A.L, q0 + BQ) : A.L;             // keys that any of the rows sees
  const int tiles = (seen + BK - 1) / BK;
  // scores of the tile of keys from k0 on: key k0 + 16 kb + 4 g + u of query q0 + 16 j + n; invisible: -inf
  auto scores = [&](const int k0, f32x4 (&S)[KB][FQ]) {
    uint4 fk[KB][KS];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int s = 0; s < KS; ++s) fk[kb][s] = *(const uint4*)(Kp + min(k0 + 16 * kb + n, A.L - 1) * rs + s * 32 + g * 8);
    __builtin_amdgcn_sched_barrier(0);                             // (all in flight together)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        S[kb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) S[kb][j] = mma16<T>(fk[kb][s], fq[j][s], S[kb][j]);
      }
    const bool edge = k0 + BK > A.L || (A.causal && k0 + BK - 1 > q0);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < FQ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) S[kb][j][u] *= A.scale;
    if (edge) {
#pragma unroll
      for (int j = 0; j < FQ; ++j) {
        const int last = A.causal ? min(q0 + 16 * j + n, A.L - 1) : A.L - 1;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int u = 0; u < 4; ++u) S[kb][j][u] = k0 + 16 * kb + 4 * g + u <= last ? S[kb][j][u] : -INFINITY;
      }
    }
  };
  float mx[FQ], sum[FQ];
#pragma unroll
  for (int j = 0; j < FQ; ++j) {
    mx[j] = -INFINITY;
    sum[j] = 0.f;
  }
  // e^(s - m), s <= m: the difference is scaled for exp2, not the scores, which may be anything in 32 bits
  auto expd = [](float s, float m) { return __builtin_amdgcn_exp2f((s - m) * 1.4426950408889634f); };
  // two parts of a row: (m, l) takes (m2, l2) in
  auto join = [&](float& m, float& l, float m2, float l2) {
    const float both = fmaxf(m, m2), from = both == -INFINITY ? 0.f : both;
    l = l * expd(m, from) + l2 * expd(m2, from);
    m = both;
  };
  f32x4 S[KB][FQ];
  int t = wave;
  for (; t < tiles; t += NW) {
    scores(t * BK, S);
#pragma unroll
    for (int j = 0; j < FQ; ++j) {
      float m = mx[j];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int u = 0; u < 4; ++u) m = fmaxf(m, S[kb][j][u]);
      const float from = m == -INFINITY ? 0.f : m;
      float l = 0.f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int u = 0; u < 4; ++u) l += expd(S[kb][j][u], from);
      sum[j] = sum[j] * expd(mx[j], from) + l;
      mx[j] = m;
    }
  }
#pragma unroll
  for (int j = 0; j < FQ; ++j) {
#pragma unroll
    for (int d = 16; d <= 32; d <<= 1) {
      const float m2 = __shfl_xor(mx[j], d), l2 = __shfl_xor(sum[j], d);
      join(mx[j], sum[j], m2, l2);
    }
    if (g == 0) stat[wave][16 * j + n] = make_float2(mx[j], sum[j]);
  }
  __syncthreads();
  float from[FQ], inv[FQ];
  bool odd = false;                                     // a row of zeros or of NaN
#pragma unroll
  for (int j = 0; j < FQ; ++j) {
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float2 v = stat[w][16 * j + n];
      join(m, l, v.x, v.y);
    }
    // nothing visible, or beyond 32 bits: zeros (a NaN among visible scores makes the row NaN)
    const bool dead = m == -INFINITY || m == INFINITY || l == 0.f;
    from[j] = dead ? INFINITY : m;
    inv[j] = dead ? 0.f : 1.0f / l;
    odd = odd || dead || !(l == l);
  }
  odd = __any(odd);
  const int width = A.causal && !A.zero_all ? min(A.L, (q0 + BQ + 255) / 256 * 256) : A.L, all = (width + BK - 1) / BK;
  const int eighth = (g & 1) * 16 + (g >> 1) * 8;
  T* const row0 = P + (int64_t)(q0 + n) * A.L + eighth;
  for (int f = t; f < all; f += NW) {
#pragma unroll
    for (int j = 0; j < FQ; ++j)
#pragma unroll
      for (int kb = 0; kb < KB; kb += 2) {
        const int c = f * BK + 16 * kb;
        if (q0 + 16 * j + n < A.L && c + eighth < width) *(uint4*)(row0 + 16 * j * (int64_t)A.L + c) = make_uint4(0, 0, 0, 0);
      }
  }
  // the last tile's scores are still there
  for (t -= NW; t >= 0;) {
#pragma unroll
    for (int j = 0; j < FQ; ++j) {
      const int r = q0 + 16 * j + n;
#pragma unroll
      for (int kb = 0; kb < KB; kb += 2) {
        const int c = t * BK + 16 * kb;
        uint32_t p[4];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          float v[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) v[u] = expd(S[kb + e][j][u], from[j]) * inv[j];
          if (odd) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (from[j] == INFINITY || (A.causal && c + 16 * e + 4 * g + u > r)) v[u] = 0.f;
          }
          p[2 * e] = pack16<T>(v[0], v[1]);
          p[2 * e + 1] = pack16<T>(v[2], v[3]);
        }
        const uint4 w = eight(p);
        if (r < A.L && c + eighth < width) *(uint4*)(row0 + 16 * j * (int64_t)A.L + c) = w;
      }
    }
    t -= NW;
    if (t >= 0) scores(t * BK, S);
  }
}

template <typename T, int KS>
void launch_weights(AttnWeightsP A, hipStream_t s) {
  A.qt = (int)ceil_div(A.L, 16 * kQBlocks);
  hipLaunchKernelGGL((attn_weights_kernel<T, KS>), dim3((unsigned)((int64_t)A.batches * A.qt)), dim3(256), 0, s, A);
}
template <typename T>
void launch_weights_type(const AttnWeightsP& A, hipStream_t s) {
  if (A.H1 == 64) launch_weights<T, 2>(A, s);
  else launch_weights<T, 4>(A, s);
}

}  // namespace

bool attention_wide_takes(const AttnWideP& P, AttnWide kind) {
  const int64_t far = (int64_t)1 << 22;                // 256 rows within 2 GB
  return P.lda < far && P.ldb < far && entry_tiles(P, kind) * P.batches < (int64_t)1 << 31;
}

void attention_wide_launch(AttnWideP P, AttnWide kind, bool bf16, hipStream_t s) {
  P.mt = (int)ceil_div(P.M, kWideM);
  P.nt = (int)ceil_div(P.N, 128);
  P.tiles = (int)entry_tiles(P, kind);
  P.xcd = P.batches % 8 == 0;
  if (bf16) launch_kind<bf16_t>(P, kind, s);
  else launch_kind<f16_t>(P, kind, s);
}

// Rows of at most 256 keys, which a workgroup's waves take in one turn, and products that give every compute unit a workgroup:
// fewer workgroups with longer rows are a chain of turns (2.7 us each with one wave on a SIMD), where the scores' own
// product has more tiles.  us, product and softmax beside this kernel, entries x positions x width (causal, full):
//      1 x  256 x 128     9.1, 9.2     9.0, 9.1       16 x 1024 x  64    33.8, 21.1    40.9, 21.6
//      8 x  256 x  64     9.4, 7.7     9.6, 7.5       16 x 2048 x 128    85.4, 49.1     159, 72.1
//      1 x  512 x 128     9.6, 14.2 (not)              4 x 2048 x 128    30.5, 39.5    39.8, 40.4 (not)
//      8 x 1024 x 128    24.4, 25.2 (not)              2 x 4096 x 128    99.7, 68.9     156, 71.5 (missed)
// Width 256: fragments from memory for half as many queries; 8 x 1024 x 256 24.5, 31.3 (not).
bool attention_weights_takes(const AttnWeightsP& A) {
  return (A.H1 == 64 || A.H1 == 128) && A.L % 8 == 0 && ((uintptr_t)A.P % 16) == 0 && (int64_t)A.batches * A.L < (int64_t)1 << 31 &&
         (A.L <= 256 || A.batches * ceil_div(A.L, 64) >= device_cu_count());
}

void attention_weights_launch(AttnWeightsP A, bool bf16, hipStream_t s) {
  A.xcd = A.batches % 8 == 0;
  if (bf16) launch_weights_type<bf16_t>(A, s);
  else launch_weights_type<f16_t>(A, s);
}

}  // namespace mega
