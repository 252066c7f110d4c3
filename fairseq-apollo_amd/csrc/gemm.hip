// Matrix products of single-precision activations on the matrix cores: C = alpha op(A) op(B) (+ bias) (+ residual), and
// silu of it.  fp32 models' linear layers and their three training products come here at the sizes of gemm_wins, the
// attention's products at those of gemm_batched_wins.
//
// The matrix cores' fp32 form runs at 157 TFLOP/s, their bf16 form at 2.5 PFLOP/s.  An fp32 value is the sum of three
// bf16 values (3 x 8 significant bits, each term rounded to nearest; exactly from 2^-110 on, below that the last term
// runs out of bf16's range and an absolute 2^-134 is lost), so a product of two matrices is the sum
// of nine bf16 products; the three smallest (below 2^-26 of the largest each, of either sign) are left out, six are
// formed, accumulation is fp32 throughout.  Measured against 64 bits the result is closer than the library's fp32
// products (which round after every four reduction indices; here after 32): see the figures at gemm_plan.
// Infinities, NaN and values that round beyond bf16's largest leave the split as NaN: an output element that is not
// finite is formed again with plain fp32 multiply-adds.
//
// A workgroup owns a 128 x 128 (eight waves) or 64 x 64 (four) tile of C, 32 reduction indices a step: fp32 pieces go
// from memory to registers two steps ahead, are split there and wait in LDS as three 16-bit planes per operand, two
// steps of them.  An operand whose
// rows run along the reduction (k-contiguous) lies in LDS as rows of 32 indices; one stored the other way round
// ([K][M]: weight gradients, dX = dY W) lies there as it is in memory and its fragments come out of transposing LDS
// reads.  Both are XOR-swizzled so that fragment reads fall on different banks.
#include <type_traits>

#include "common.h"

namespace mega {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) short s16x4;

constexpr int kGK = 32;           // reduction indices a step
constexpr int kTerms = 3;         // bf16 terms of an fp32 value
constexpr int kAhead = 2;         // steps whose values are on their way from memory

struct GemmP {
  const float* A;      // element (m, k): m * lda + k, or (K-major) k * lda + m
  const float* B;      // element (n, k): n * ldb + k, or (K-major) k * ldb + n
  float* C;            // element (m, n): m * ldc + n
  const float* bias;   // [N] or null
  const float* R;      // added: m * ldr + n, or null
  float* pre;          // the value before the activation, m * ldc + n, or null
  int64_t lda, ldb, ldc, ldr;
  int64_t sa, sai, sb, sbi, sc, sci;     // batch entry z = o * nin + i: base + o * s? + i * s?i
  int nin;
  int M, N, K;
  float alpha;
  int silu;
  int causal;          // 1: elements with n > m are not needed; 2: B's k > m is zero in A; 3: A's k < m is zero
  int mt, nt;          // tiles
  int kstep;           // reduction indices of a split (a multiple of kGK)
  float* part;         // [splits][M][N] partial sums, or null
  int vc;              // 16-byte stores fit
};

__device__ __forceinline__ f32x4 mma(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// a pair of fp32 values as three packed pairs of bf16 terms
__device__ __forceinline__ void split3(float x, float y, uint32_t (&t)[kTerms]) {
#pragma unroll
  for (int i = 0; i < kTerms; ++i) {
    const bf16x2 h = {(__bf16)x, (__bf16)y};
    t[i] = __builtin_bit_cast(uint32_t, h);
    if (i + 1 < kTerms) {
      x -= __uint_as_float(t[i] << 16);
      y -= __uint_as_float(t[i] & 0xffff0000u);
    }
  }
}

__device__ __forceinline__ float silu_f(float v) { return v / (1.f + __expf(-v)); }

// One operand's side of the tile: W rows (of A) or columns (of B), KM: stored K-major, kGT threads.
template <int W, bool KM, int kGT>
struct Side {
  static constexpr int Row = KM ? W * 2 : kGK * 2;                // bytes of a row of a plane
  static constexpr int Plane = W * kGK * 2;
  static constexpr int NP = W * kGK / 4 / kGT;                    // 16-byte pieces of memory per thread

  // piece h of a thread: (row along W or k, first index along the other)
  static __device__ __forceinline__ void piece(int tid, int h, int& w, int& k) {
    if constexpr (KM) {
      const int p = tid + h * kGT;
      w = (p % (W / 4)) * 4;
      k = p / (W / 4);
    } else {                                                       // pieces 2 j and 2 j + 1 are eight indices of a row
      const int p = tid + (h >> 1) * kGT;
      w = p / 4;
      k = (p % 4) * 8 + (h & 1) * 4;
    }
  }
  // swizzle of the 32-byte spans of a K-major row / the 16-byte pieces of a k-contiguous one
  static __device__ __forceinline__ int turn(int row) {
    if constexpr (KM) return W == 128 ? (row & 3) + 4 * ((row >> 3) & 1) : ((row >> 1) & 1) + 2 * ((row >> 3) & 1);
    else return (0x78 >> (row >> 1 & 6)) & 3;        // 0, 2, 3, 1
  }

  // byte offset of piece h from the tile's first element in a step of `left` reduction indices; rows and indices beyond
  // the matrix replaced by the last piece inside it (the rows are never stored, the indices are cleared below)
  static __device__ __forceinline__ uint32_t offset(int64_t ld, int tid, int h, int room, int left) {
    int w, k;
    piece(tid, h, w, k);
    // (sizes that are no multiple of four come with padded rows: the last piece is whole in memory)
    w = min(w, KM ? ((room + 3) & ~3) - 4 : room - 1);
    k = min(k, KM ? left - 1 : ((left + 3) & ~3) - 4);
    return (uint32_t)((KM ? (int64_t)k * ld + w : (int64_t)w * ld + k) * 4);
  }
  static __device__ __forceinline__ void load(const float* tile, const uint32_t (&off)[NP], float4 (&v)[NP]) {
#pragma unroll
    for (int h = 0; h < NP; ++h) v[h] = *(const float4*)((const char*)tile + off[h]);
  }
  static __device__ __forceinline__ void clear_beyond(int tid, int left, float4 (&v)[NP]) {
#pragma unroll
    for (int h = 0; h < NP; ++h) {
      int w, k;
      piece(tid, h, w, k);
      if constexpr (KM) {
        if (k >= left) v[h] = make_float4(0.f, 0.f, 0.f, 0.f);
      } else {
        v[h].x = k < left ? v[h].x : 0.f;
        v[h].y = k + 1 < left ? v[h].y : 0.f;
        v[h].z = k + 2 < left ? v[h].z : 0.f;
        v[h].w = k + 3 < left ? v[h].w : 0.f;
      }
    }
  }
  // the same for operands off 16 bytes or of odd sizes, element by element
  static __device__ __forceinline__ void load_edge(const float* src, int64_t ld, int w0, int k0, int wmax, int kmax, int tid,
                                                   float4 (&v)[NP]) {
#pragma unroll
    for (int h = 0; h < NP; ++h) {
      int w, k;
      piece(tid, h, w, k);
      w += w0;
      k += k0;
      float r[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int wu = KM ? w + u : w, ku = KM ? k : k + u;
        const bool in = wu < wmax && ku < kmax;
        r[u] = in ? src[KM ? (int64_t)ku * ld + wu : (int64_t)wu * ld + ku] : 0.f;
      }
      v[h] = make_float4(r[0], r[1], r[2], r[3]);
    }
  }
  // the terms of the pieces, packed as they go to LDS
  static __device__ __forceinline__ void pack(const float4 (&v)[NP], uint2 (&q)[kTerms][NP]) {
#pragma unroll
    for (int h = 0; h < NP; ++h) {
      uint32_t a[kTerms], b[kTerms];
      split3(v[h].x, v[h].y, a);
      split3(v[h].z, v[h].w, b);
#pragma unroll
      for (int t = 0; t < kTerms; ++t) q[t][h] = make_uint2(a[t], b[t]);
    }
  }
  static __device__ __forceinline__ void store(char* lds, int tid, const uint2 (&q)[kTerms][NP]) {
#pragma unroll
    for (int h = 0; h < NP; h += KM ? 1 : 2) {
      int w, k;
      piece(tid, h, w, k);
      if constexpr (KM) {
        char* at = lds + k * Row + (((w >> 4) ^ turn(k)) << 5) + (w & 15) * 2;
#pragma unroll
        for (int t = 0; t < kTerms; ++t) *(uint2*)(at + t * Plane) = q[t][h];
      } else {
        char* at = lds + w * Row + (((k >> 3) ^ turn(w)) << 4);
#pragma unroll
        for (int t = 0; t < kTerms; ++t)
          *(uint4*)(at + t * Plane) = make_uint4(q[t][h].x, q[t][h].y, q[t][h + 1].x, q[t][h + 1].y);
      }
    }
  }
  // fragment: lane (n = lane & 15, g = lane >> 4) gets reduction indices 8 g .. 8 g + 7 of row / column w16 * 16 + n
  static __device__ __forceinline__ uint4 frag(const char* plane, int w16, int lane) {
    const int n = lane & 15, g = lane >> 4;
    if constexpr (KM) {
      const int row = 8 * g + (n >> 2);
      const char* q = plane + row * Row + ((w16 ^ turn(row)) << 5) + (n & 3) * 8;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(q));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(q + 4 * Row));
      const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
      return make_uint4(l2.x, l2.y, h2.x, h2.y);
    } else {
      const int row = w16 * 16 + n;
      return *(const uint4*)(plane + row * Row + ((g ^ turn(row)) << 4));
    }
  }
};

// TM x TN: the tile; two waves along its rows, WN along its columns.  FORM 0: whole steps of 32 reduction indices and
// 16-byte accesses; 1: a partial last step; 2: operands that 16-byte accesses do not fit
template <int TM, int TN, int WN, bool KA, bool KB, int FORM>
__global__ __launch_bounds__(128 * WN, 2) void gemm_f32_kernel(const GemmP G) {
  using SA = Side<TM, KA, 128 * WN>;
  using SB = Side<TN, KB, 128 * WN>;
  constexpr int FM = TM / 32, FN = TN / (16 * WN);                 // 16 x 16 blocks of a wave each way
  constexpr int kStage = kTerms * (SA::Plane + SB::Plane);
  extern __shared__ __attribute__((aligned(16))) char lds[];       // two stages of the operands' planes
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tiles = G.mt * G.nt;
  // consecutive workgroup ids go to the 8 XCDs in turn: every XCD gets neighbouring tiles
  const int total = (int)gridDim.x;
  const int id = total % 8 == 0 ? ((int)blockIdx.x & 7) * (total >> 3) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
  const int z = id / tiles, tl = id - z * tiles;                   // z: batch entry, or split
  const int mi = tl / G.nt, m0 = mi * TM, n0 = (tl - mi * G.nt) * TN;
  if (G.causal == 1 && n0 > m0 + TM - 1) return;                    // nothing of the tile is needed
  const float *A = G.A, *B = G.B;
  float* C = G.C;
  int kb = 0, ke = G.K;
  if (G.part) {
    kb = z * G.kstep;
    ke = min(G.K, kb + G.kstep);
    C = G.part + (int64_t)z * G.M * G.N;
  } else {
    const int o = z / G.nin, i = z - o * G.nin;
    A += o * G.sa + i * G.sai;
    B += o * G.sb + i * G.sbi;
    C += o * G.sc + i * G.sci;
    if (G.causal == 2) ke = min(ke, m0 + TM);
    if (G.causal == 3) kb = m0 / kGK * kGK;
  }
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = (wave / WN) * FM, wn = (wave % WN) * FN;            // the wave's first 16-row / 16-column block
  float4 ra[kAhead][SA::NP], rb[kAhead][SB::NP];                   // values of the coming steps
  uint32_t oa[SA::NP], ob[SB::NP];
  auto offsets = [&](const int left) {
#pragma unroll
    for (int h = 0; h < SA::NP; ++h) oa[h] = SA::offset(G.lda, tid, h, G.M - m0, left);
#pragma unroll
    for (int h = 0; h < SB::NP; ++h) ob[h] = SB::offset(G.ldb, tid, h, G.N - n0, left);
  };
  if (FORM != 2) offsets(kGK);
  const float* const ta = A + (KA ? (int64_t)kb * G.lda + m0 : (int64_t)m0 * G.lda + kb);
  const float* const tb = B + (KB ? (int64_t)kb * G.ldb + n0 : (int64_t)n0 * G.ldb + kb);
  const int64_t da = KA ? kGK * G.lda : kGK, db = KB ? kGK * G.ldb : kGK;
  const int steps = (ke - kb + kGK - 1) / kGK;
  // the values of step s (of the last one again behind it: the loop below has no branches, so that the splitting is
  // scheduled between the matrix products)
  auto load = [&](int s, float4 (&va)[SA::NP], float4 (&vb)[SB::NP]) {
    s = min(s, steps - 1);
    if constexpr (FORM == 2) {
      SA::load_edge(A, G.lda, m0, kb + s * kGK, G.M, ke, tid, va);
      SB::load_edge(B, G.ldb, n0, kb + s * kGK, G.N, ke, tid, vb);
    } else {
      if (FORM == 1) offsets(min(kGK, ke - kb - s * kGK));
      SA::load(ta + s * da, oa, va);
      SB::load(tb + s * db, ob, vb);
    }
  };
  auto store = [&](int s, char* stage, float4 (&va)[SA::NP], float4 (&vb)[SB::NP]) {
    if (FORM == 1) {
      SA::clear_beyond(tid, ke - kb - s * kGK, va);
      SB::clear_beyond(tid, ke - kb - s * kGK, vb);
    }
    uint2 qa[kTerms][SA::NP], qb[kTerms][SB::NP];
    SA::pack(va, qa);
    SB::pack(vb, qb);
    SA::store(stage, tid, qa);
    SB::store(stage + kTerms * SA::Plane, tid, qb);
  };
  // Step s: its terms lie in stage s mod 2 of the LDS.  The values of step s + 1, asked for kAhead steps ago, are split
  // and stored to the other stage beside this step's products, and their registers take the values of step
  // s + 1 + kAhead: a wait for memory is spread over kAhead steps.
  auto step = [&](auto P, const int s) {
    constexpr int p = decltype(P)::value, q = (p + 1) % kAhead;
    const char* la = lds + (p & 1) * kStage;
    const char* lb = la + kTerms * SA::Plane;
    uint4 fa[kTerms][FM];
#pragma unroll
    for (int t = 0; t < kTerms; ++t)
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[t][i] = SA::frag(la + t * SA::Plane, wm + i, lane);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      uint4 fb[kTerms];
#pragma unroll
      for (int t = 0; t < kTerms; ++t) fb[t] = SB::frag(lb + t * SB::Plane, wn + j, lane);
      // the operands swapped: a lane ends up with four consecutive columns of a row; the smallest products first
#pragma unroll
      for (int o = kTerms - 1; o >= 0; --o)
#pragma unroll
        for (int t = 0; t <= o; ++t)
#pragma unroll
          for (int i = 0; i < FM; ++i) acc[i][j] = mma(fb[o - t], fa[t][i], acc[i][j]);
    }
    store(s + 1, lds + (1 - (p & 1)) * kStage, ra[q], rb[q]);
    // (not above the splitting: the loop would end with copies of registers that wait for every load in flight)
    __builtin_amdgcn_sched_barrier(0);
    load(s + 1 + kAhead, ra[q], rb[q]);
    __syncthreads();
  };
  if (steps > 0) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s) load(s, ra[s], rb[s]);
    store(0, lds, ra[0], rb[0]);
    load(kAhead, ra[0], rb[0]);
    __syncthreads();
  }
  for (int s = 0; s < steps; s += kAhead) {
    step(std::integral_constant<int, 0>{}, s);
    if (s + 1 >= steps) break;
    step(std::integral_constant<int, 1>{}, s + 1);
  }
  const int64_t ldc = G.part ? G.N : G.ldc;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + (wm + i) * 16 + (lane & 15);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + (wn + j) * 16 + (lane >> 4) * 4;
      if (m >= G.M || n >= G.N) continue;
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      const float chk = (v[0] - v[0]) + (v[1] - v[1]) + (v[2] - v[2]) + (v[3] - v[3]);
      if (chk != 0.f) {
        // Something is not finite: in plain fp32, lane by lane, eight indices on their way at a time.  Weight gradient 1024 x
        // 1024 x 8000 (180 us) with one row that is not finite 3.9 ms, without a finite element 7.3 (15 and 30 one index at a
        // time; 0.9 and 1.6 by the matrix cores' fp32 form, whose code here had the compiler schedule the loop above worse:
        // every product of finite values 3 - 8 % slower).
#pragma unroll 1
        for (int u = 0; u < 4; ++u) {
          if (n + u >= G.N) break;
          const float* pa = A + (KA ? (int64_t)m : (int64_t)m * G.lda);
          const float* pb = B + (KB ? (int64_t)(n + u) : (int64_t)(n + u) * G.ldb);
          float s = 0.f;
#pragma unroll 8
          for (int k = kb; k < ke; ++k) s = fmaf(pa[KA ? (int64_t)k * G.lda : k], pb[KB ? (int64_t)k * G.ldb : k], s);
          if (u == 0) v[0] = s;
          if (u == 1) v[1] = s;
          if (u == 2) v[2] = s;
          if (u == 3) v[3] = s;
        }
      }
      float* c = C + (int64_t)m * ldc + n;
      if (G.part) {
        if (G.N % 4 == 0) {
          *(float4*)c = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (n + u < G.N) c[u] = v[u];
        }
        continue;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        v[u] *= G.alpha;
        if (n + u < G.N) {
          if (G.bias) v[u] += G.bias[n + u];
          if (G.R) v[u] += G.R[(int64_t)m * G.ldr + n + u];
        }
      }
      if (G.vc && n + 4 <= G.N) {
        if (G.pre) *(float4*)(G.pre + (int64_t)m * ldc + n) = make_float4(v[0], v[1], v[2], v[3]);
        if (G.silu) *(float4*)c = make_float4(silu_f(v[0]), silu_f(v[1]), silu_f(v[2]), silu_f(v[3]));
        else *(float4*)c = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (n + u < G.N) {
            if (G.pre) G.pre[(int64_t)m * ldc + n + u] = v[u];
            c[u] = G.silu ? silu_f(v[u]) : v[u];
          }
      }
    }
  }
}

// C = alpha sum of the splits' partial sums (+ bias) (+ residual), silu: four columns a thread when they fit
__global__ __launch_bounds__(256) void gemm_sum_kernel(const GemmP G, int splits, int vec) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * vec, total = (int64_t)G.M * G.N;
  if (i >= total) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (vec == 4) {
    for (int s = 0; s < splits; ++s) {
      const float4 p = *(const float4*)(G.part + s * total + i);
      v[0] += p.x; v[1] += p.y; v[2] += p.z; v[3] += p.w;
    }
  } else {
    for (int s = 0; s < splits; ++s) v[0] += G.part[s * total + i];
  }
  const int m = (int)(i / G.N), n = (int)(i - (int64_t)m * G.N);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    if (u >= vec) break;
    v[u] *= G.alpha;
    if (G.bias) v[u] += G.bias[n + u];
    if (G.R) v[u] += G.R[(int64_t)m * G.ldr + n + u];
    const int64_t o = (int64_t)m * G.ldc + n + u;
    if (G.pre) G.pre[o] = v[u];
    G.C[o] = G.silu ? silu_f(v[u]) : v[u];
  }
}

struct Plan {
  int tile, splits, kstep;
};

// Tiles of 128 (half the LDS traffic of a product) where there are several of them for every compute unit, of 64
// otherwise.  A product of fewer tiles than compute units is split along the reduction, 256 indices and more each, into
// partial sums that a second kernel adds up in order.
// What bounds a step of a tile is LDS: three planes are written and read for every fp32 operand (72 KB a step of a
// 64 x 64 tile, 576 cycles at 128 bytes a cycle beside 384 of matrix products on each SIMD), and the waves of a
// workgroup read, multiply and write in step; the 128 tile's waves do so for twice the products.
// Errors against 64 bits in 1e-7 of the result, the library's fp32 products behind the comma: x W^T 8000 x 512 x 256 2.3,
// 2.9; 2048 x 512 x 1024 3.4, 5.7; 4096 x 4096 x 4096 10, 11.5; dY^T X 512 x 256 x 8000 3.6, 16; 1088 x 256 x 8000 5.0, 16.
Plan gemm_plan(int64_t M, int64_t N, int64_t K, int64_t batch) {
  const int cus = device_cu_count();
  Plan p = {64, 1, 0};
  if (ceil_div(M, 128) * ceil_div(N, 128) * batch >= 4 * cus) p.tile = 128;
  const int64_t tiles = ceil_div(M, p.tile) * ceil_div(N, p.tile) * batch;
  if (batch == 1 && tiles < cus) {
    int64_t s = ceil_div(2 * cus, tiles);
    const int64_t most = K / 256;
    if (s > most) s = most;
    if (s > 64) s = 64;
    if (s > 1) {
      p.kstep = (int)(ceil_div(ceil_div(K, s), kGK) * kGK);
      p.splits = (int)ceil_div(K, p.kstep);
    }
  }
  return p;
}

// Sizes that come here, us of device time, one kernel after the other, beside the GEMM library's.  A library call takes
// 24 - 26 us of host time, one here 6; what loses more than 9 us and a tenth of device time against that is left to it.
//   two and more workgroups a compute unit, two only for short reductions (one alone waits at every barrier: 0.70 us a
//   step of 32, two 0.51 a piece, three 0.46, the library's rate is 0.45):
//     8000 x 512 x 256     24, library 23       2048 x 2176 x 512    42, 63       2048 x 1024 x 1024    35, 35
//     8000 x 1024 x 2816  311, 318              4096 x 1024 x 2816  164, 157
//   tiles of 128:  16384 x 2048 x 1024  397, 479      4096 x 4096 x 2048   365, 479
//   up to 3 GFLOP, counted in whole tiles (small ones are a launch's latency, 10 us here and 5 there):
//     2048 x 512 x 1024    24, 21       512 x 1024 x 2816    33, 27       300 x 2048 x 1024    26, 18
//     512 x 512 x 1024     15, 10       64 x 4096 x 2048     19, 16       1 x 4096 x 2048      18, 9
//   weight gradients (both K-major) onto at most 300,000 elements, whose long reductions the library hardly splits:
//     512 x 256 x 8000     29, 46       1088 x 256 x 8000    53, 63       128 x 128 x 1000     17, 62
//   and not (the library's):
//     512 x 2048 x 4096    89, 63       1000 x 1024 x 4352   97, 68       2048 x 1024 x 2816   88, 80
//     1024 x 1024 x 8000 177, 112       2048 x 1024 x 8000  255, 229       512 x 1024 x 8000   72, 65 (both K-major)
// Operands that 16-byte accesses do not fit go to the library (element-wise loads: 1000 x 1022 x 1026 57, 24).
bool gemm_wins(int64_t M, int64_t N, int64_t K, int a_kmajor, int b_kmajor) {
  const Plan p = gemm_plan(M, N, K, 1);
  if (p.tile == 128) return true;
  const int64_t tiles = ceil_div(M, 64) * ceil_div(N, 64), two = 2 * device_cu_count();
  if (2.0 * 64 * 64 * (double)tiles * (double)K <= 3e9) return true;
  return tiles * p.splits > two || (tiles * p.splits == two && K / p.splits <= 1024) || (a_kmajor && b_kmajor && M * N <= 300000);
}

// The same for a batch of products over positions (attention's; `heads` of them interleaved in every row of the operands,
// which the library's call copies apart first), from replayed graphs:
//   fewer workgroups than twice the compute units are a chain of steps (batches are not split): only short ones
//     q k^T   8 x 512 x 512 x 128       own 12, library 13       w v   8 x 1000 x 64 x 1000   own 31, library 15 (not)
//             1 x 512 x 512 x 1024          25, 9 (not)                2 x 4096 x 64 x 4096      101, 37 (not)
//     just as many: up to 1024 indices, or half of them (causal w v 2 x 1024 x 1024 x 1024 37, 34; full 8 x 2048 x 128 x 2048
//     74, 63 (not))
//   several heads: own (4 x 1000 x 4 heads x 64: q k^T 16, 36)
//   tiles of 128: own from 256 reduction indices on (4 x 2048 x 2048 x 1024 208, 245); little reduction onto 2^25 scores
//     and more, or 64 rows, waste it (8 x 2048 x 2048 x 32 57, 41; 64 x 64 x 2048 x 64 36, 20)
//   tiles of 64: own (8 x 1000 x 1000 x 512 69, 72), unless the second operand's rows overflow an XCD's 4 MB of L2
//     (2 x 2048 x 2048 x 512 78, 66) and no causal limit saves half of it
bool gemm_batched_wins(int64_t M, int64_t N, int64_t K, int64_t batch, int64_t heads, int causal, int a_kmajor) {
  const Plan p = gemm_plan(M, N, K, batch);
  const int64_t tiles = ceil_div(M, 64) * ceil_div(N, 64) * batch, splits = causal ? 1 : p.splits, two = 2 * device_cu_count();
  if (tiles * splits < two) return K / splits <= 512;
  if (tiles * splits == two) return causal >= 2 || K <= 1024;
  if (heads > 1) return true;
  if (p.tile == 128) return M > 64 && (K > 128 || tiles < 8192);
  if (N * K >= 1 << 20 && !a_kmajor) return causal == 2 || (causal == 1 && batch > 1);
  return true;
}

template <int TM, int TN, int WN, bool KA, bool KB, int FORM>
void gemm_launch_form(const GemmP& G, unsigned blocks, hipStream_t s) {
  static uint64_t attr_seen = 0;
  const auto kern = gemm_f32_kernel<TM, TN, WN, KA, KB, FORM>;
  constexpr int smem = 2 * kTerms * (TM + TN) * kGK * 2;
  if (smem > 64 * 1024) raise_lds_limit(&attr_seen, smem, kern);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(128 * WN), smem, s, G);
}

template <int TM, int TN, int WN, int FORM>
void gemm_launch(const GemmP& G, int ka, int kb, unsigned blocks, hipStream_t s) {
  if (ka && kb) gemm_launch_form<TM, TN, WN, true, true, FORM>(G, blocks, s);
  else if (ka) gemm_launch_form<TM, TN, WN, true, false, FORM>(G, blocks, s);
  else if (kb) gemm_launch_form<TM, TN, WN, false, true, FORM>(G, blocks, s);
  else gemm_launch_form<TM, TN, WN, false, false, FORM>(G, blocks, s);
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_gemm_f32_pays(int64_t M, int64_t N, int64_t K, int a_kmajor, int b_kmajor) {
  return M > 0 && N > 0 && K > 0 && gemm_wins(M, N, K, a_kmajor, b_kmajor) ? 1 : 0;
}

extern "C" int mega_gemm_f32_batched_pays(int64_t M, int64_t N, int64_t K, int64_t batch, int64_t heads, int causal, int a_kmajor) {
  return M > 0 && N > 0 && K > 0 && batch > 0 && gemm_batched_wins(M, N, K, batch, heads, causal, a_kmajor) ? 1 : 0;
}

extern "C" size_t mega_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t batch) {
  if (M <= 0 || N <= 0 || K <= 0 || batch != 1) return 0;
  const Plan p = gemm_plan(M, N, K, batch);
  return p.splits > 1 ? (size_t)p.splits * M * N * 4 : 0;
}

extern "C" int mega_gemm_f32(const MegaGemm* g, void* workspace, size_t workspace_bytes, void* stream) {
  MEGA_REQUIRE(g, MEGA_ERR_ARG, "gemm_f32: null argument");
  MEGA_REQUIRE(g->M >= 0 && g->N >= 0 && g->K >= 0 && g->batch >= 0 && g->inner >= 1, MEGA_ERR_ARG, "gemm_f32: bad shape");
  if (g->M == 0 || g->N == 0 || g->batch == 0) return MEGA_OK;
  MEGA_REQUIRE(g->c && (g->K == 0 || (g->a && g->b)), MEGA_ERR_ARG, "gemm_f32: null pointer argument");
  MEGA_REQUIRE(g->M < (int64_t)1 << 30 && g->N < (int64_t)1 << 30 && g->K < (int64_t)1 << 30, MEGA_ERR_UNSUPPORTED,
               "gemm_f32: sizes below 2^30");
  MEGA_REQUIRE(g->lda >= (g->a_kmajor ? g->M : g->K) && g->ldb >= (g->b_kmajor ? g->N : g->K) && g->ldc >= g->N &&
                   (!g->residual || g->ldr >= g->N),
               MEGA_ERR_ARG, "gemm_f32: a leading dimension is shorter than its row");
  MEGA_REQUIRE(g->batch == 1 || (!g->bias && !g->residual && !g->pre && !g->silu), MEGA_ERR_UNSUPPORTED,
               "gemm_f32: batched products take no bias, residual or activation");
  MEGA_REQUIRE(g->causal >= 0 && g->causal <= 3 && (!g->causal || g->M == (g->causal == 1 ? g->N : g->K)), MEGA_ERR_ARG,
               "gemm_f32: a causal product is square in its positions");
  GemmP G = {};
  G.A = (const float*)g->a; G.B = (const float*)g->b; G.C = (float*)g->c;
  G.bias = (const float*)g->bias; G.R = (const float*)g->residual; G.pre = (float*)g->pre;
  G.lda = g->lda; G.ldb = g->ldb; G.ldc = g->ldc; G.ldr = g->ldr;
  G.sa = g->sa; G.sai = g->sai; G.sb = g->sb; G.sbi = g->sbi; G.sc = g->sc; G.sci = g->sci;
  G.nin = (int)g->inner; G.M = (int)g->M; G.N = (int)g->N; G.K = (int)g->K;
  G.alpha = g->alpha; G.silu = g->silu; G.causal = g->causal;
  auto on16 = [](const void* p, int64_t ld, int64_t s, int64_t si) {
    return (uintptr_t)p % 16 == 0 && ld % 4 == 0 && s % 4 == 0 && si % 4 == 0;
  };
  // (whole pieces along the contiguous axis, a tile's rows within 4 GB of its first element)
  const int64_t far = ((int64_t)1 << 32) / 4 / 128;
  const bool edge = !(on16(g->a, g->lda, g->sa, g->sai) && (g->a_padded || (g->a_kmajor ? g->M : g->K) % 4 == 0) && g->lda < far &&
                      on16(g->b, g->ldb, g->sb, g->sbi) && (g->b_kmajor ? g->N : g->K) % 4 == 0 && g->ldb < far);
  G.vc = on16(g->c, g->ldc, g->sc, g->sci) && (uintptr_t)g->pre % 16 == 0;
  Plan p = gemm_plan(g->M, g->N, g->K, g->batch);
  if (edge) p.tile = 64;
  G.mt = (int)ceil_div(g->M, p.tile);
  G.nt = (int)ceil_div(g->N, p.tile);
  const bool split = p.splits > 1 && g->causal == 0;
  if (split) {
    const size_t need = (size_t)p.splits * g->M * g->N * 4;
    MEGA_REQUIRE(workspace && workspace_bytes >= need && (uintptr_t)workspace % 16 == 0, MEGA_ERR_WORKSPACE,
                 "gemm_f32: workspace of %zu bytes needed", need);
    G.part = (float*)workspace;
    G.kstep = p.kstep;
  }
  const int64_t blocks = (int64_t)G.mt * G.nt * (split ? p.splits : g->batch);
  MEGA_REQUIRE(blocks < (int64_t)1 << 31, MEGA_ERR_UNSUPPORTED, "gemm_f32: too many tiles");
  hipStream_t s = (hipStream_t)stream;
  const int ka = g->a_kmajor, kb = g->b_kmajor;
  const unsigned nb = (unsigned)blocks;
  const bool ragged = g->K % kGK != 0;
  if (edge) gemm_launch<64, 64, 2, 2>(G, ka, kb, nb, s);
  else if (p.tile == 128) ragged ? gemm_launch<128, 128, 4, 1>(G, ka, kb, nb, s) : gemm_launch<128, 128, 4, 0>(G, ka, kb, nb, s);
  else ragged ? gemm_launch<64, 64, 2, 1>(G, ka, kb, nb, s) : gemm_launch<64, 64, 2, 0>(G, ka, kb, nb, s);
  MEGA_CHECK_LAUNCH("gemm_f32");
  if (split) {
    const int vec = g->N % 4 == 0 ? 4 : 1;
    const int64_t items = g->M * g->N / vec;
    hipLaunchKernelGGL(gemm_sum_kernel, dim3((unsigned)ceil_div(items, 256)), dim3(256), 0, s, G, p.splits, vec);
    MEGA_CHECK_LAUNCH("gemm_f32 (sum of the splits)");
  }
  return MEGA_OK;
}
