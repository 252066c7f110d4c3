// 16-bit attention with its weights in memory: the long products y = P v, dv = w^T dy, and dS, whose
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

}  // namespace mega
