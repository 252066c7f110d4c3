// Matrix products of bf16 / fp16 activations: C = op(A) op(B) (+ bias) (+ residual), and silu of the rounded value.  A library
// call costs 26 us of host time, more than most products of a few thousand tokens take, and its weight gradients (both
// operands stored along the other axis, a reduction over thousands of tokens onto a small matrix) run at a third to a half
// of its forward products' rate.  Here are the kernel for few tokens and the entry; wide tiles: gemm16_wide.h.
//
// A workgroup of four waves owns a 64 x 64 tile, 64 reduction indices a step: 16-byte pieces go from memory
// to registers two steps ahead and from there to one of two LDS stages, k-contiguous operands as rows of a step's indices,
// the others as they lie in memory, their fragments read by transposing LDS loads.  Sums are fp32 throughout, also
// between the parts of a product that is split along the reduction.
#include <type_traits>

#include "gemm16.h"

namespace mega {
namespace {

constexpr int kHT = 256;          // threads
constexpr int kTile = 64;         // rows, columns and reduction indices of a step

// One operand's side of the tile: 64 rows (of A) or columns (of B), KM: stored K-major.
template <bool KM>
struct Side16 {
  static constexpr int Row = kTile * 2;                           // bytes of a row
  static constexpr int Bytes = kTile * kTile * 2;
  static constexpr int NP = kTile * kTile / 8 / kHT;              // 16-byte pieces per thread

  static __device__ __forceinline__ void piece(int tid, int h, int& w, int& k) {
    const int p = tid + h * kHT;
    if constexpr (KM) {
      w = (p % (kTile / 8)) * 8;
      k = p / (kTile / 8);
    } else {
      w = p / (kTile / 8);
      k = (p % (kTile / 8)) * 8;
    }
  }
  static __device__ __forceinline__ int turn(int row) {
    if constexpr (KM) return ((row >> 1) & 1) + 2 * ((row >> 3) & 1);
    else return (row >> 1) & 7;
  }
  // byte offset of piece h from the tile's first element in a step of `left` indices; what lies beyond the matrix is
  // replaced by the last piece inside it (rows are never stored, indices are cleared below)
  static __device__ __forceinline__ uint32_t offset(int64_t ld, int tid, int h, int room, int left) {
    int w, k;
    piece(tid, h, w, k);
    w = min(w, KM ? room - 8 : room - 1);
    k = min(k, KM ? left - 1 : left - 8);
    return (uint32_t)((KM ? (int64_t)k * ld + w : (int64_t)w * ld + k) * 2);
  }
  static __device__ __forceinline__ void load(const char* tile, const uint32_t (&off)[NP], uint4 (&v)[NP]) {
#pragma unroll
    for (int h = 0; h < NP; ++h) v[h] = *(const uint4*)(tile + off[h]);
  }
  static __device__ __forceinline__ void store(char* lds, int tid, int left, const uint4 (&v)[NP]) {
#pragma unroll
    for (int h = 0; h < NP; ++h) {
      int w, k;
      piece(tid, h, w, k);
      const bool in = k < left;                                    // (left = 64 at compile time in whole steps)
      const uint4 x = make_uint4(in ? v[h].x : 0u, in ? v[h].y : 0u, in ? v[h].z : 0u, in ? v[h].w : 0u);
      char* at = KM ? lds + k * Row + (((w >> 4) ^ turn(k)) << 5) + (w & 15) * 2 : lds + w * Row + (((k >> 3) ^ turn(w)) << 4);
      *(uint4*)at = x;
    }
  }
  // fragment of 32 indices (kk-th of the step): lane (n, g) gets indices 8 g .. 8 g + 7 of row / column w16 * 16 + n
  static __device__ __forceinline__ uint4 frag(const char* lds, int w16, int kk, int lane) {
    const int n = lane & 15, g = lane >> 4;
    if constexpr (KM) {
      const int row = 8 * g + (n >> 2);
      const char* q = lds + (kk * 32 + row) * Row + ((w16 ^ turn(row)) << 5) + (n & 3) * 8;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(q));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(q + 4 * Row));
      const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
      return make_uint4(l2.x, l2.y, h2.x, h2.y);
    } else {
      const int row = w16 * 16 + n;
      return *(const uint4*)(lds + row * Row + (((kk * 4 + g) ^ turn(row)) << 4));
    }
  }
};

// RAG: a partial last step
template <typename T, bool KA, bool KB, bool RAG>
__global__ __launch_bounds__(kHT, 2) void gemm16_kernel(const Gemm16P G) {
  using SA = Side16<KA>;
  using SB = Side16<KB>;
  constexpr int F = kTile / 32;                                  // 16 x 16 blocks of a wave each way
  constexpr int kStage = SA::Bytes + SB::Bytes;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tiles = G.mt * G.nt, total = (int)gridDim.x;
  const int id = total % 8 == 0 ? ((int)blockIdx.x & 7) * (total >> 3) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
  const int z = id / tiles, tl = id - z * tiles;
  const int mi = tl / G.nt, m0 = mi * kTile, n0 = (tl - mi * G.nt) * kTile;
  const int kb = G.part ? z * G.kstep : 0, ke = G.part ? min(G.K, kb + G.kstep) : G.K;
  f32x4 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = (wave >> 1) * F, wn = (wave & 1) * F;
  uint4 ra[2][SA::NP], rb[2][SB::NP];
  uint32_t oa[SA::NP], ob[SB::NP];
  auto offsets = [&](const int left) {
#pragma unroll
    for (int h = 0; h < SA::NP; ++h) oa[h] = SA::offset(G.lda, tid, h, G.M - m0, left);
#pragma unroll
    for (int h = 0; h < SB::NP; ++h) ob[h] = SB::offset(G.ldb, tid, h, G.N - n0, left);
  };
  offsets(kTile);
  const char* const ta = (const char*)G.A + (KA ? (int64_t)kb * G.lda + m0 : (int64_t)m0 * G.lda + kb) * 2;
  const char* const tb = (const char*)G.B + (KB ? (int64_t)kb * G.ldb + n0 : (int64_t)n0 * G.ldb + kb) * 2;
  const int64_t da = (KA ? kTile * G.lda : kTile) * 2, db = (KB ? kTile * G.ldb : kTile) * 2;
  const int steps = (ke - kb + kTile - 1) / kTile;
  auto load = [&](int s, uint4 (&va)[SA::NP], uint4 (&vb)[SB::NP]) {
    s = min(s, steps - 1);
    if (RAG) offsets(min(kTile, ke - kb - s * kTile));
    SA::load(ta + s * da, oa, va);
    SB::load(tb + s * db, ob, vb);
  };
  auto store = [&](int s, char* stage, uint4 (&va)[SA::NP], uint4 (&vb)[SB::NP]) {
    const int left = RAG ? ke - kb - s * kTile : kTile;
    SA::store(stage, tid, left, va);
    SB::store(stage + SA::Bytes, tid, left, vb);
  };
  auto step = [&](auto P, const int s) {
    constexpr int p = decltype(P)::value;
    const char* la = lds + p * kStage;
    const char* lb = la + SA::Bytes;
#pragma unroll
    for (int kk = 0; kk < kTile / 32; ++kk) {
      uint4 fa[F], fb[F];
#pragma unroll
      for (int i = 0; i < F; ++i) fa[i] = SA::frag(la, wm + i, kk, lane);
#pragma unroll
      for (int j = 0; j < F; ++j) fb[j] = SB::frag(lb, wn + j, kk, lane);
      // the operands swapped: a lane ends up with four consecutive columns of a row
#pragma unroll
      for (int j = 0; j < F; ++j)
#pragma unroll
        for (int i = 0; i < F; ++i) acc[i][j] = mma16<T>(fb[j], fa[i], acc[i][j]);
    }
    store(s + 1, lds + (1 - p) * kStage, ra[1 - p], rb[1 - p]);
    __builtin_amdgcn_sched_barrier(0);
    load(s + 3, ra[1 - p], rb[1 - p]);
    __syncthreads();
  };
  if (steps > 0) {
    load(0, ra[0], rb[0]);
    load(1, ra[1], rb[1]);
    store(0, lds, ra[0], rb[0]);
    load(2, ra[0], rb[0]);
    __syncthreads();
  }
  for (int s = 0; s < steps; s += 2) {
    step(std::integral_constant<int, 0>{}, s);
    if (s + 1 >= steps) break;
    step(std::integral_constant<int, 1>{}, s + 1);
  }
  float* part = G.part ? G.part + (int64_t)z * G.M * G.N : nullptr;
#pragma unroll
  for (int i = 0; i < F; ++i) {
    const int m = m0 + (wm + i) * 16 + (lane & 15);
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int n = n0 + (wn + j) * 16 + (lane >> 4) * 4;
      if (m >= G.M || n >= G.N) continue;                          // (N is a multiple of eight)
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      if (part) *(float4*)(part + (int64_t)m * G.N + n) = make_float4(v[0], v[1], v[2], v[3]);
      else finish16<T, 4>(G, m, n, v);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void gemm16_sum_kernel(const Gemm16P G, int splits) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, total = (int64_t)G.M * G.N;
  if (i >= total) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < splits; ++s) {
    const float4 p = *(const float4*)(G.part + s * total + i);
    v[0] += p.x; v[1] += p.y; v[2] += p.z; v[3] += p.w;
  }
  const int m = (int)(i / G.N);
  finish16<T, 4>(G, m, (int)(i - (int64_t)m * G.N), v);
}

struct Plan16 {
  int splits, kstep;
};

// A product of few tiles is split along the reduction.
Plan16 gemm16_plan(int64_t M, int64_t N, int64_t K) {
  const int cus = device_cu_count();
  Plan16 p = {1, 0};
  const int64_t tiles = ceil_div(M, kTile) * ceil_div(N, kTile);
  if (tiles <= cus / 2) {
    int64_t s = ceil_div(2 * cus, tiles);
    const int64_t most = K / 512;
    if (s > most) s = most;
    if (s > 32) s = 32;
    if (s > 1) {
      p.kstep = (int)(ceil_div(ceil_div(K, s), kTile) * kTile);
      p.splits = (int)ceil_div(K, p.kstep);
    }
  }
  return p;
}

// What a product costs here, us of device time: 0.36 a step of a compute unit's only workgroup, half a microsecond of the two it
// holds, the second kernel's 5 and its traffic at 4 TB/s.  (600 x 1024 x 2816 19.3, 1000 x 1024 x 2816 19.8, 768 x 768 x 2048
// 15.3, 300 x 2048 x 4096 26.5, 1000 x 2048 x 4096 33.5.)
double gemm16_small_us(int64_t M, int64_t N, int64_t K) {
  const Plan16 p = gemm16_plan(M, N, K);
  const double tiles = (double)ceil_div(M, kTile) * ceil_div(N, kTile) * p.splits, two = 2.0 * device_cu_count();
  return 4 + (2 * tiles > two ? 0.5 : 0.36) * ceil_div(ceil_div(K, p.splits), kTile) * (tiles > two ? tiles / two : 1) +
         (p.splits > 1 ? 5 + (double)M * N * (4 * p.splits + 2) / 4e6 : 0);
}

// Wide tiles (gemm16_wide.h) where their estimate is the smaller one; us, tiles of 64 and wide ones:
//     300 x 4352 x 1024   10, 15       600 x 4352 x 1024   16.5, 15     1000 x 4352 x 1024   25, 16
//    2048 x 2048 x 1024   19, 16      2048 x 4352 x 1024   43, 26       5000 x 1536 x 768    27, 16
//     600 x 1024 x 2816   19, 24      1000 x 1024 x 2816   20, 23      1000 x 2048 x 4096   34, 29
//   both K-major   264 x 1024 x 8192   22, 24     1024 x 2048 x 2000   21, 27     1536 x 768 x 4503   39, 26
//                  768 x 768 x 2048    15, 22
bool gemm16_wide(int64_t M, int64_t N, int64_t K, WidePlan* p) {
  *p = gemm16_wide_plan(M, N, K);
  return p->us < gemm16_small_us(M, N, K);
}

// Products that come here.  us of device time beside the library's, between a pass that writes the operand and one that reads
// the result (x W^T in whole tiles), otherwise operands and results from memory (more than 600 MB of them in turn; *: the same
// ones each time):
//   x W^T, whole rounds of tiles or less than two
//                5000 x 2048 x 1024   28.0, 24.2     8192 x 1024 x 2048   34.2, 35.6     8192 x 2816 x 1024   57.7, 53.3
//                5000 x 2048 x 4096   88.1, 70.2     8192 x 2048 x 5632    130, 123     32768 x 5632 x 2048    571, 528
//     more than two, the last one partial    12000 x 2816 x 1024   76.7, 84.6     12000 x 4352 x 1024    115, 147
//                8192 x 5632 x 2048    156, 163      8192 x 8704 x 2048    246, 260     12000 x 4096 x 4096    284, 443
//                8192 x 4352 x 1024   82.4, 73.1    10000 x 5632 x 2048    198, 180     16384 x 8704 x 2048    464, 435
//     N not in whole tiles   8192 x 1032 x 1024   29.6, 29.9     8192 x 3264 x 768   56.3, 67.4    65536 x 776 x 1024    123, 156
//               20000 x 2056 x 512    61.7, 116      8192 x 8200 x 2048    233, 275     65536 x 2056 x 2048   499, 451
//     with silu (the library's takes another pass)    2048 x 4096 x 2048   36.5, 43.0    8192 x 4096 x 2048    126, 129
//               16384 x 1536 x 768    58.7, 63.7    32768 x 8192 x 4096   1551, 1601    16384 x 8192 x 8192   1493, 1464
//   dY W         8192 x 1024 x 2048   36.2, 39.6     5000 x 2048 x 4096   92.7, 80.9     8192 x 2048 x 8704    223, 232
//               16384 x 5632 x 2048    321, 362     16384 x 16384 x 16384*  6221, 6574
//   dY^T X       1024 x 2048 x 8192   44.5, 76.3     4352 x 1024 x 12000   117, 172      8704 x 2048 x 8192    248, 320
//                2816 x 1024 x 2048   29.3, 26.2    16384 x 16384 x 16384*  6315, 7585
// x W^T in whole tiles: the library is 6 % ahead on average (127 sizes), but where its tiles leave a partial round behind more than
// two whole ones, 6 % behind (33 sizes, 0.89 to 1.56).  Its call costs the host 26 us, so that calls made of products below
// 20 GFLOP (20 us and less) are bound by the host with it, and those of up to 4096 tokens, with less beside the products, below
// 40 GFLOP; beyond, the device is the bound: 5000 tokens of 2048 channels 1032 with all of them here, 947 in the library.  us of
// whole calls, those of 20 to 40 GFLOP in the library and here:
//   model, width 1024   3 x 1000   540, 507     8 x 461   577, 520     4 x 1024   585, 580     1 x 5000   673, 678 (not)     2 x 2991   751, 755 (not)
//   layer   4096 x 1024   307, 297     1024 x 2048   319, 301     1536 x 2048   355, 377     2560 x 2048   497, 498     5120 x 1024   350, 351 (not)
// (below: a layer of 2048 tokens of 1024 channels 299 with the library, 217.  Missed: 2048 x 2048, 473, all of them here 448.)  N not
// in whole tiles: 10 - 25 % ahead to 200 GFLOP, even to 400.  silu: ahead by the pass, whose share is 1 / K.  dY W is even to
// 130 GFLOP, 2 - 5 % ahead beyond, dY^T X 20 - 70 % ahead.  Nothing is measured beyond 1e13.
bool gemm16_wins(int64_t M, int64_t N, int64_t K, int a_kmajor, int b_kmajor, bool silu) {
  const double flops = 2.0 * (double)M * (double)N * (double)K;
  if (a_kmajor || b_kmajor) return flops <= 1e13;
  if (silu && K <= 4096) return flops <= 2.5e12;
  const int64_t tiles = ceil_div(M, kWideM) * ceil_div(N, 256), round = device_cu_count();
  return flops <= (N % 256 || (tiles > 2 * round && tiles % round) ? 5e11 : M <= 4096 ? 4e10 : 2e10);
}

// Sizes that the kernels hold in 32 bits, tiles that a launch takes (2^32 threads)
bool gemm16_launchable(int64_t M, int64_t N, int64_t K) {
  const int64_t most = (int64_t)1 << 30;
  return M < most && N < most && K < most && ceil_div(M, kTile) * ceil_div(N, kTile) < ((int64_t)1 << 32) / kHT;
}

template <typename T, bool KA, bool KB>
void launch16(const Gemm16P& G, unsigned blocks, hipStream_t s) {
  constexpr int smem = 2 * 2 * kTile * kTile * 2;
  static_assert(smem <= 64 * 1024, "within the LDS that every launch may ask for");
  const auto kern = G.K % kTile ? gemm16_kernel<T, KA, KB, true> : gemm16_kernel<T, KA, KB, false>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kHT), smem, s, G);
}
template <typename T>
void launch16_type(const Gemm16P& G, const Plan16& p, int ka, int kb, unsigned blocks, hipStream_t s) {
  if (ka && kb) launch16<T, true, true>(G, blocks, s);
  else if (ka) launch16<T, true, false>(G, blocks, s);
  else if (kb) launch16<T, false, true>(G, blocks, s);
  else launch16<T, false, false>(G, blocks, s);
  if (p.splits > 1)
    hipLaunchKernelGGL((gemm16_sum_kernel<T>), dim3((unsigned)ceil_div((int64_t)G.M * G.N, 1024)), dim3(256), 0, s, G, p.splits);
}

}  // namespace
}  // namespace mega

using namespace mega;

extern "C" int mega_gemm16_pays(int64_t M, int64_t N, int64_t K, int a_kmajor, int b_kmajor) {
  return gemm16_launchable(M, N, K) && gemm16_wins(M, N, K, a_kmajor, b_kmajor, false) ? 1 : 0;
}

extern "C" int mega_gemm16_silu_pays(int64_t M, int64_t N, int64_t K, int a_kmajor, int b_kmajor) {
  return gemm16_launchable(M, N, K) && gemm16_wins(M, N, K, a_kmajor, b_kmajor, true) ? 1 : 0;
}

extern "C" size_t mega_gemm16_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const Plan16 p = gemm16_plan(M, N, K);
  const size_t small = p.splits > 1 ? (size_t)p.splits * M * N * 4 : 0;
  WidePlan w;
  return gemm16_wide(M, N, K, &w) && w.bytes > small ? w.bytes : small;
}

extern "C" int mega_gemm16(const MegaGemm* g, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  MEGA_REQUIRE(g && (dtype == MEGA_BF16 || dtype == MEGA_F16), MEGA_ERR_ARG, "gemm16: bf16 or fp16 operands");
  MEGA_REQUIRE(g->M > 0 && g->N > 0 && g->K > 0 && g->batch == 1 && !g->causal && g->alpha == 1.f, MEGA_ERR_UNSUPPORTED,
               "gemm16: single products without a factor");
  MEGA_REQUIRE(g->a && g->b && g->c, MEGA_ERR_ARG, "gemm16: null pointer argument");
  MEGA_REQUIRE(gemm16_launchable(g->M, g->N, g->K), MEGA_ERR_UNSUPPORTED, "gemm16: sizes below 2^30, fewer than 2^24 tiles of 64 x 64");
  MEGA_REQUIRE(g->lda >= (g->a_kmajor ? g->M : g->K) && g->ldb >= (g->b_kmajor ? g->N : g->K) && g->ldc >= g->N &&
                   (!g->residual || g->ldr >= g->N),
               MEGA_ERR_ARG, "gemm16: a leading dimension is shorter than its row");
  const int64_t far = ((int64_t)1 << 32) / 2 / 128;
  auto on16 = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  MEGA_REQUIRE(on16(g->a) && on16(g->b) && on16(g->c) && on16(g->bias) && on16(g->residual) && on16(g->pre) && g->lda % 8 == 0 &&
                   g->ldb % 8 == 0 && g->ldc % 8 == 0 && (!g->residual || g->ldr % 8 == 0) && g->N % 8 == 0 &&
                   (g->a_kmajor ? g->M : g->K) % 8 == 0 && (g->b_kmajor ? g->N : g->K) % 8 == 0 && g->lda < far && g->ldb < far,
               MEGA_ERR_UNSUPPORTED, "gemm16: rows of whole 16-byte pieces");
  Gemm16P G = {};
  G.A = g->a; G.B = g->b; G.C = g->c; G.bias = g->bias; G.R = g->residual; G.pre = g->pre;
  G.lda = g->lda; G.ldb = g->ldb; G.ldc = g->ldc; G.ldr = g->ldr;
  G.M = (int)g->M; G.N = (int)g->N; G.K = (int)g->K; G.silu = g->silu;
  WidePlan w;
  // (rows of a wide tile within 4 GB of its first element)
  if (gemm16_wide(g->M, g->N, g->K, &w) && g->lda < far / 2 && g->ldb < far / 2) {
    MEGA_REQUIRE(!w.bytes || (workspace && workspace_bytes >= w.bytes && on16(workspace)), MEGA_ERR_WORKSPACE,
                 "gemm16: workspace of %zu bytes needed", w.bytes);
    gemm16_wide_launch(G, w, dtype == MEGA_BF16, g->a_kmajor, g->b_kmajor, workspace, (hipStream_t)stream);
    MEGA_CHECK_LAUNCH("gemm16 (wide tiles)");
    return MEGA_OK;
  }
  const Plan16 p = gemm16_plan(g->M, g->N, g->K);
  G.mt = (int)ceil_div(g->M, kTile);
  G.nt = (int)ceil_div(g->N, kTile);
  if (p.splits > 1) {
    const size_t need = (size_t)p.splits * g->M * g->N * 4;
    MEGA_REQUIRE(workspace && workspace_bytes >= need && on16(workspace), MEGA_ERR_WORKSPACE, "gemm16: workspace of %zu bytes needed",
                 need);
    G.part = (float*)workspace;
    G.kstep = p.kstep;
  }
  const int64_t blocks = (int64_t)G.mt * G.nt * p.splits;          // (split only where they are few)
  if (dtype == MEGA_BF16) launch16_type<bf16_t>(G, p, g->a_kmajor, g->b_kmajor, (unsigned)blocks, (hipStream_t)stream);
  else launch16_type<f16_t>(G, p, g->a_kmajor, g->b_kmajor, (unsigned)blocks, (hipStream_t)stream);
  MEGA_CHECK_LAUNCH("gemm16");
  return MEGA_OK;
}
