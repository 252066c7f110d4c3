// 16-bit matrix products of many tiles, C = op(A) op(B) (+ bias) (+ residual), and silu of the rounded value.
//
// Two kernels.  Four waves on a 256 x 256 tile, one wave on each SIMD with 128 x 128 of it: 256 accumulator registers, read
// 1.5 times less LDS than eight waves would, 64 matrix instructions a half step beside 16 fragment reads and 16 loads spread
// between them.  Eight waves on a 256 x 128 tile, for shapes of too few tiles: two groups of four, one wave of each on every
// SIMD, one reads its fragments while the other multiplies.  Memory goes straight to LDS (16 bytes a lane, no registers), 64
// reduction indices a step, so that every request is a whole 128-byte line: with steps of 32 (half lines, twice the requests
// and more power, and power is what bounds a large product: 1.55 - 1.75 GHz) the first kernel ran at 1380 TFLOP/s on
// 8192 x 8192 x 8192, as it is at 1529; the library's 1582.  32 x 32 x 16 instructions: 1305 (1.55 GHz instead of 1.77).
#pragma once

#include <type_traits>
#include <utility>

#include "gemm16.h"

namespace mega {
namespace {

constexpr int kKS = 64;           // reduction indices a step
// 16 bytes a lane from memory to LDS: lane l's go to byte lds + 16 l.  (The compiler does not honour a clobber of M0.  That it
// keeps nothing of its own there is part of the build's check: putting it back each time costs 2 % of a product.)
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t off, const char* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

// One operand's side of the tile: W rows (of A) or columns (of B), KM: stored K-major, kWT threads.
template <int W, bool KM, int kWT>
struct Wide {
  static constexpr int Row = KM ? W * 2 : kKS * 2;
  static constexpr int Bytes = W * kKS * 2;
  static constexpr int NP = Bytes / 16 / kWT;                     // 16-byte pieces per thread

  static __device__ __forceinline__ int turn(int row) {
    if constexpr (KM) return (row & 3) + 4 * ((row >> 3) & 1);
    else return (row >> 1) & 7;
  }
  // byte offset in memory (from the tile's first element) of the piece that goes to LDS place h * kWT + tid of a step of
  // `left` indices; beyond the matrix the last piece inside it
  static __device__ __forceinline__ uint32_t offset(int64_t ld, int tid, int h, int room, int left) {
    const int p = tid + h * kWT;
    int w, k;
    if constexpr (KM) {
      k = p / (W / 8);
      const int s = p % (W / 8);
      w = (((s >> 1) ^ turn(k)) << 4) + (s & 1) * 8;
    } else {
      w = p / (kKS / 8);
      k = ((p % (kKS / 8)) ^ turn(w)) * 8;
    }
    w = min(w, KM ? room - 8 : room - 1);
    k = min(k, KM ? left - 1 : left - 8);
    return (uint32_t)((KM ? (int64_t)k * ld + w : (int64_t)w * ld + k) * 2);
  }
  // LDS byte address parts of the fragments of 16-row blocks w16 .. w16 + F - 1
  static constexpr int NB = KM ? 1 : kKS / 32;
  template <int F>
  struct Frags {
    uint32_t at[KM ? F : NB];
    __device__ __forceinline__ void init(int w16, int lane) {
      const int n = lane & 15, g = lane >> 4;
      if constexpr (KM) {
        const int row = 8 * g + (n >> 2);
#pragma unroll
        for (int i = 0; i < F; ++i) at[i] = row * Row + (((w16 + i) ^ turn(row)) << 5) + (n & 3) * 8;
      } else {
#pragma unroll
        for (int kk = 0; kk < NB; ++kk) at[kk] = (w16 * 16 + n) * Row + (((kk * 4 + g) ^ turn(n)) << 4);
      }
    }
    __device__ __forceinline__ uint4 get(const char* lds, int i, int kk) const {
      if constexpr (KM) {
        const char* q = lds + at[i] + kk * 32 * Row;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(q));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(q + 4 * Row));
        const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
        return make_uint4(l2.x, l2.y, h2.x, h2.y);
      } else {
        return *(const uint4*)(lds + at[kk] + i * 16 * Row);
      }
    }
  };
};

__device__ __forceinline__ uint32_t keep2(uint32_t v, int k, int left) {
  return k + 1 < left ? v : k < left ? v & 0xffffu : 0u;
}
// indices k0 .. k0 + 7 of a fragment, those from `left` on cleared
__device__ __forceinline__ uint4 keep(uint4 f, int k0, int left) {
  return make_uint4(keep2(f.x, k0, left), keep2(f.y, k0 + 2, left), keep2(f.z, k0 + 4, left), keep2(f.w, k0 + 6, left));
}

// c += a b with the accumulator in the accumulator registers (left to itself the compiler keeps it in the others and moves it
// to and fro).  The compiler pads its own matrix instructions with the wait states that a vector instruction before them, or
// behind them on their result, calls for; these it does not see.  None is needed where it puts no register copy between them,
// which the build checks in the compiled kernels (check_assembly of build.py) instead of paying for it here: two wait
// states with each cost 3 - 5 % of a product (8192 x 8192 x 8192 705, 730 us), with every fourth as much.
template <typename T>
__device__ __forceinline__ void mma_acc(f32x4& c, uint4 a, uint4 b) {
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  const u32x4 x = {a.x, a.y, a.z, a.w}, y = {b.x, b.y, b.z, b.w};
  if constexpr (__is_same(T, bf16_t)) asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
  else asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
}

// rows and columns of tile t
template <int TN>
__device__ __forceinline__ void tile_at(const Gemm16P& G, int t, int& m0, int& n0) {
  const int deep = 4 * G.nt, grp = t / deep, in = t - grp * deep, rows = min(4, G.mt - grp * 4);
  m0 = (grp * 4 + in % rows) * kWideM;
  n0 = in / rows * TN;
}

// Which tile, and which part of the reduction, a workgroup has: G.full tiles whole, the others in G.splits parts
struct Place {
  int m0, n0, kb, ke;
  float* part;                       // where the tile's partial sums go, or null
};
template <int TN>
__device__ __forceinline__ Place place(const Gemm16P& G) {
  // consecutive workgroup ids go to the 8 XCDs in turn: each gets a run of tiles, four rows of them deep
  const int first = (int)blockIdx.x < G.full ? 0 : G.full, total = first ? (int)gridDim.x - G.full : G.full ? G.full : (int)gridDim.x;
  const int b = (int)blockIdx.x - first, x = b & 7;
  int id = x * (total >> 3) + min(x, total & 7) + (b >> 3);
  Place p;
  p.kb = 0;
  p.ke = G.K;
  p.part = nullptr;
  const int rest = G.mt * G.nt - G.full;
  if (G.part && (int)blockIdx.x >= G.full) {
    const int z = id / rest;
    p.part = G.part + (int64_t)id * (kWideM * TN);
    id -= z * rest;
    p.kb = z * G.kstep;
    p.ke = min(G.K, p.kb + G.kstep);
  }
  tile_at<TN>(G, first + id, p.m0, p.n0);
  return p;
}

template <typename T>
__device__ __forceinline__ uint32_t pack16(float x, float y) {
  const T a = from_float<T>(x), b = from_float<T>(y);
  return (uint32_t)__builtin_bit_cast(uint16_t, a) | (uint32_t)__builtin_bit_cast(uint16_t, b) << 16;
}
template <typename T>
__device__ __forceinline__ float low16(uint32_t v) { return to_float(__builtin_bit_cast(T, (uint16_t)v)); }

// a block's values out of the accumulator registers, here and not before (ACC); or as they are
template <bool ACC>
__device__ __forceinline__ f32x4 values(f32x4 x) {
  if constexpr (ACC) asm volatile("" : "+v"(x));
  return x;
}

// Two neighbouring 16 x 16 blocks of values packed in pairs: a lane holds columns 4 g .. 4 g + 3 of its row (lane & 15) in
// each (g = lane >> 4).  Exchanged between neighbouring lane groups, it has eight columns of one: a 16-byte store.
__device__ __forceinline__ uint4 eight(const uint32_t (&p)[4]) {
  const auto x = __builtin_amdgcn_permlane16_swap(p[0], p[2], false, false), y = __builtin_amdgcn_permlane16_swap(p[1], p[3], false, false);
  return make_uint4(x[0], y[0], x[1], y[1]);
}

// A wave's blocks to memory, EDGE: some beyond the matrix.  Nothing runs beside it in the square kernel (one wave on each
// SIMD), so instructions count: bias in registers, rows' pointers once, rounded pairs exchanged instead of single values
// (8192 x 2048 x 1024 with 256-column tiles: 32.0 us, 34.3 through finish16 on eight exchanged floats).
//
// Branches between the blocks keep one block's loads and exponentials from running beside the next one's, so the frequent
// kinds are whole: 0 the sums alone, 1 with a bias, 2 with a residual, 3 silu of 1, 4 anything (8192 x 2048 x 1024: 31, 31, 38,
// 36 us; residual and silu with branches 41 and 39, silu by the bare reciprocal 34).
template <typename T, bool ACC, int KIND, bool EDGE, int FM, int FN>
__device__ __forceinline__ void store_wave(const Gemm16P& G, const Place& p, int wm, int wn, int lane, const f32x4 (&acc)[FM][FN]) {
  const int g = lane >> 4, row = wm * 16 + (lane & 15), col = wn * 16;
  const int m0 = p.m0 + row, n0 = p.n0 + col, own = n0 + g * 4, mine = n0 + (g & 1) * 16 + (g >> 1) * 8;
  float bias[FN][4];
  if (KIND && KIND != 2 && G.bias) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = EDGE ? min(own + j * 16, G.N - 4) : own + j * 16;
      const Vec<T, 4> b = *(const Vec<T, 4>*)((const T*)G.bias + n);
#pragma unroll
      for (int u = 0; u < 4; ++u) bias[j][u] = to_float(b.v[u]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) bias[j][u] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + i * 16, mr = EDGE ? min(m, G.M - 1) : m;
    const int64_t at = (int64_t)mr * G.ldc + mine;
    const T* r = KIND == 2 || (KIND == 4 && G.R) ? (const T*)G.R + (int64_t)mr * G.ldr : nullptr;
#pragma unroll
    for (int j = 0; j < FN; j += 2) {
      const bool in = !EDGE || (m < G.M && mine + j * 16 < G.N);   // (N is a multiple of eight)
      uint32_t q[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[4];
        const f32x4 sum = values<ACC>(acc[i][j + h]);
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = KIND && KIND != 2 ? sum[u] + bias[j + h][u] : sum[u];
        if (KIND == 2 || (KIND == 4 && r)) {
          const int n = own + (j + h) * 16;
          const Vec<T, 4> t = *(const Vec<T, 4>*)(r + (EDGE ? min(n, G.N - 4) : n));
#pragma unroll
          for (int u = 0; u < 4; ++u) v[u] += to_float(t.v[u]);
        }
        q[2 * h] = pack16<T>(v[0], v[1]);
        q[2 * h + 1] = pack16<T>(v[2], v[3]);
      }
      if (KIND == 4 && G.pre) {
        const uint4 x = eight(q);
        if (in) *(uint4*)((T*)G.pre + at + j * 16) = x;
      }
      if (KIND == 3 || (KIND == 4 && G.silu)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = pack16<T>(silu_h(low16<T>(q[u])), silu_h(low16<T>(q[u] >> 16)));
      }
      const uint4 x = eight(q);
      if (in) *(uint4*)((T*)G.C + at + j * 16) = x;
    }
  }
}

template <typename T, bool ACC, int TN, int FM, int FN>
__device__ __forceinline__ void finish_wave(const Gemm16P& G, const Place& p, int wm, int wn, int lane, const f32x4 (&acc)[FM][FN]) {
  if (p.part) {
    float* c = p.part + (wm * 16 + (lane & 15)) * TN + wn * 16 + (lane >> 4) * 4;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) *(f32x4*)(c + i * 16 * TN + j * 16) = values<ACC>(acc[i][j]);
  } else if (p.m0 + kWideM <= G.M && p.n0 + TN <= G.N) {
    if (G.pre || (G.R && (G.bias || G.silu))) store_wave<T, ACC, 4, false>(G, p, wm, wn, lane, acc);
    else if (G.R) store_wave<T, ACC, 2, false>(G, p, wm, wn, lane, acc);
    else if (G.silu) store_wave<T, ACC, 3, false>(G, p, wm, wn, lane, acc);
    else if (G.bias) store_wave<T, ACC, 1, false>(G, p, wm, wn, lane, acc);
    else store_wave<T, ACC, 0, false>(G, p, wm, wn, lane, acc);
  } else {
    store_wave<T, ACC, 4, true>(G, p, wm, wn, lane, acc);
  }
}

// f(0), .. f(N - 1) with their numbers as constants: fragments addressed by them are registers whatever is unrolled when
template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  each_of(std::make_integer_sequence<int, N>{}, f);
}

template <typename T, bool KA, bool KB, bool RAG>
__global__ __launch_bounds__(256, 1) void gemm16_square_kernel(const Gemm16P G) {
  constexpr int TN = 256, ST = 2, kWT = 256;                       // columns of a tile, stages, threads
  using SA = Wide<kWideM, KA, kWT>;
  using SB = Wide<TN, KB, kWT>;
  constexpr int FM = kWideM / 32, FN = TN / 32;
  constexpr int kStage = SA::Bytes + SB::Bytes, LD = SA::NP + SB::NP;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Place at_tile = place<TN>(G);
  const int m0 = at_tile.m0, n0 = at_tile.n0, kb = at_tile.kb, ke = at_tile.ke;
  const int steps = (ke - kb + kKS - 1) / kKS;
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = (wave >> 1) * FM, wn = (wave & 1) * FN;
  uint32_t oa[SA::NP], ob[SB::NP];
  auto offsets = [&](const int left) {
#pragma unroll
    for (int h = 0; h < SA::NP; ++h) oa[h] = SA::offset(G.lda, tid, h, G.M - m0, left);
#pragma unroll
    for (int h = 0; h < SB::NP; ++h) ob[h] = SB::offset(G.ldb, tid, h, G.N - n0, left);
  };
  offsets(kKS);
  const char* ta = (const char*)G.A + (KA ? (int64_t)kb * G.lda + m0 : (int64_t)m0 * G.lda + kb) * 2;
  const char* tb = (const char*)G.B + (KB ? (int64_t)kb * G.ldb + n0 : (int64_t)n0 * G.ldb + kb) * 2;
  const int64_t da = (KA ? kKS * G.lda : kKS) * 2, db = (KB ? kKS * G.ldb : kKS) * 2;
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * 1024;
  int next = 0;                      // the step that is asked for next, and its stage
  uint32_t stage = at;
  auto piece = [&](int h) {
    if (h < SA::NP) dma16(stage + h * (kWT * 16), oa[h], ta);
    else dma16(stage + SA::Bytes + (h - SA::NP) * (kWT * 16), ob[h - SA::NP], tb);
  };
  auto advance = [&]() {
    ta += da;
    tb += db;
    ++next;
    stage = stage == at + (ST - 1) * kStage ? at : stage + kStage;
  };
  typename SA::template Frags<FM> fa_at;
  typename SB::template Frags<FN> fb_at;
  fa_at.init(wm, lane);
  fb_at.init(wn, lane);
#pragma unroll
  for (int s = 0; s < ST; ++s)
    if (s < steps) {
      if (RAG && next == steps - 1) offsets(ke - kb - next * kKS);
#pragma unroll
      for (int h = 0; h < LD; ++h) piece(h);
      advance();
    }
  if (steps >= ST) wait_loads<LD*(ST - 1)>();
  else wait_loads<0>();
  barrier();
  const char* la = lds;
  uint4 fa[2][FM], fb[2][FN];
  constexpr int NM = FM * FN, FR = FM + FN, RS = NM * 3 / 4 / FR, DS = NM / LD;
  auto read = [&](auto Q, const char* from, auto F) {               // fragment F of index half Q: fb 0, fa 0 .., fb 1 ..
    constexpr int q = decltype(Q)::value, f = decltype(F)::value;
    if constexpr (f == 0) fb[q][0] = fb_at.get(from + SA::Bytes, 0, q);
    else if constexpr (f <= FM) fa[q][f - 1] = fa_at.get(from, f - 1, q);
    else if constexpr (f < FR) fb[q][f - FM] = fb_at.get(from + SA::Bytes, f - FM, q);
  };
  using zero = std::integral_constant<int, 0>;
  using one = std::integral_constant<int, 1>;
  each<FR>([&](auto f) { read(zero{}, la, f); });
  auto step = [&](auto MORE, const int s) {
    constexpr bool more = decltype(MORE)::value;
    const int left = ke - kb - s * kKS, g8 = (lane >> 4) * 8;
    if (RAG && s == steps - 1) {
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[0][j] = keep(fb[0][j], g8, left);
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[0][i] = keep(fa[0][i], g8, left);
      asm volatile("s_nop 4" ::: "memory");
    }
    __builtin_amdgcn_sched_barrier(0);
    each<NM>([&](auto at) {
      constexpr int t = decltype(at)::value;
      // (all read in the first three quarters: they have arrived when the products are through)
      if constexpr (t % RS == 0) read(one{}, la, std::integral_constant<int, t / RS>{});
      mma_acc<T>(acc[t % FM][t / FM], fb[0][t / FM], fa[0][t % FM]);
      __builtin_amdgcn_sched_barrier(0);
    });
    if (more) wait_loads<LD*(ST - 2)>();
    else wait_loads<0>();
    barrier();
    la = la == lds + (ST - 1) * kStage ? lds : la + kStage;
    if (RAG && s == steps - 1) {
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[1][j] = keep(fb[1][j], 32 + g8, left);
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[1][i] = keep(fa[1][i], 32 + g8, left);
      asm volatile("s_nop 4" ::: "memory");
    }
    if (RAG && more && next == steps - 1) offsets(ke - kb - next * kKS);
    __builtin_amdgcn_sched_barrier(0);
    each<NM>([&](auto at) {
      constexpr int t = decltype(at)::value;
      if constexpr (t % RS == 0) read(zero{}, la, std::integral_constant<int, t / RS>{});
      if (more && t % DS == 1 && t / DS < LD) piece(t / DS);
      mma_acc<T>(acc[t % FM][t / FM], fb[1][t / FM], fa[1][t % FM]);
      __builtin_amdgcn_sched_barrier(0);
    });
    if (more) advance();
  };
  int s = 0;
#pragma unroll 1
  for (; s + ST < steps; ++s) step(one{}, s);
#pragma unroll 1
  for (; s < steps; ++s) step(zero{}, s);
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  finish_wave<T, true, TN>(G, at_tile, wm, wn, lane, acc);
}

// A 256 x 128 tile by eight waves.
template <typename T, bool KA, bool KB, bool RAG>
struct Tall {
  static constexpr int TN = 128, ST = 3, kWT = 512;                // columns of a tile, stages, threads
  using SA = Wide<kWideM, KA, kWT>;
  using SB = Wide<TN, KB, kWT>;
  static constexpr int WN = 2, FM = kWideM / 16 * WN / 8, FN = TN / 16 / WN, KK = kKS / 32;   // waves along N, a wave's blocks each way
  static constexpr int kStage = SA::Bytes + SB::Bytes, LD = SA::NP + SB::NP;
  static constexpr int kLds = ST * kStage;

  // The sums of the tile whose first row / column start at ta / tb, over `len` indices; rooms: rows / columns to the end of
  // the matrix.
  static __device__ __forceinline__ void sums(char* lds, const char* ta, const char* tb, int64_t lda, int64_t ldb, int room_a,
                                              int room_b, int len, int tid, int wm, int wn, f32x4 (&acc)[FM][FN]) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int steps = (len + kKS - 1) / kKS;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint32_t oa[SA::NP], ob[SB::NP];
    auto offsets = [&](const int left) {
#pragma unroll
      for (int h = 0; h < SA::NP; ++h) oa[h] = SA::offset(lda, tid, h, room_a, left);
#pragma unroll
      for (int h = 0; h < SB::NP; ++h) ob[h] = SB::offset(ldb, tid, h, room_b, left);
    };
    offsets(kKS);
    const int64_t da = (KA ? kKS * lda : kKS) * 2, db = (KB ? kKS * ldb : kKS) * 2;
    const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * 1024;
    int next = 0;                    // the step that is asked for next, and its stage
    uint32_t stage = at;
    auto issue = [&]() {
      if (RAG && next == steps - 1) offsets(len - next * kKS);
#pragma unroll
      for (int h = 0; h < SA::NP; ++h) dma16(stage + h * (kWT * 16), oa[h], ta);
#pragma unroll
      for (int h = 0; h < SB::NP; ++h) dma16(stage + SA::Bytes + h * (kWT * 16), ob[h], tb);
      ta += da;
      tb += db;
      ++next;
      stage = stage == at + (ST - 1) * kStage ? at : stage + kStage;
    };
    typename SA::template Frags<FM> fa_at;
    typename SB::template Frags<FN> fb_at;
    fa_at.init(wm, lane);
    fb_at.init(wn, lane);
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
      if (s < steps) issue();
    if (steps >= ST - 1) wait_loads<LD*(ST - 2)>();
    else wait_loads<0>();
    barrier();
    // Two groups of four waves, one of each on every SIMD: while one reads its fragments the other multiplies.
    if (wave >= 4) barrier();
    const char* la = lds;
    for (int s = 0; s < steps; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (next < steps) issue();
      uint4 fa[KK][FM], fb[KK][FN];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[kk][j] = fb_at.get(la + SA::Bytes, j, kk);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[kk][i] = fa_at.get(la, i, kk);
      }
      la = la == lds + (ST - 1) * kStage ? lds : la + kStage;
      if (s + ST - 1 < steps) wait_loads<LD*(ST - 2)>();          // the next step's stage has arrived
      else wait_loads<0>();
      barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (RAG && s == steps - 1) {
        const int left = len - s * kKS, g8 = (lane >> 4) * 8;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
          for (int j = 0; j < FN; ++j) fb[kk][j] = keep(fb[kk][j], kk * 32 + g8, left);
#pragma unroll
          for (int i = 0; i < FM; ++i) fa[kk][i] = keep(fa[kk][i], kk * 32 + g8, left);
        }
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int i = 0; i < FM; ++i) acc[i][j] = mma16<T>(fb[kk][j], fa[kk][i], acc[i][j]);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      barrier();
    }
    if (wave < 4) barrier();
  }
};

template <typename T, bool KA, bool KB, bool RAG>
__global__ __launch_bounds__(512, 2) void gemm16_tall_kernel(const Gemm16P G) {
  using K = Tall<T, KA, KB, RAG>;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Place p = place<K::TN>(G);
  const int wm = (wave / K::WN) * K::FM, wn = (wave % K::WN) * K::FN;
  const char* ta = (const char*)G.A + (KA ? (int64_t)p.kb * G.lda + p.m0 : (int64_t)p.m0 * G.lda + p.kb) * 2;
  const char* tb = (const char*)G.B + (KB ? (int64_t)p.kb * G.ldb + p.n0 : (int64_t)p.n0 * G.ldb + p.kb) * 2;
  f32x4 acc[K::FM][K::FN];
  K::sums(lds, ta, tb, G.lda, G.ldb, G.M - p.m0, G.N - p.n0, p.ke - p.kb, tid, wm, wn, acc);
  finish_wave<T, false, K::TN>(G, p, wm, wn, tid & 63, acc);
}

// the tiles behind the first G.full: the parts' sums added in order
template <typename T, int TN>
__global__ __launch_bounds__(256) void gemm16_parts_kernel(const Gemm16P G) {
  constexpr int kTile = kWideM * TN;
  const int r = blockIdx.x / (kTile / 2048), at = (blockIdx.x % (kTile / 2048)) * 2048 + threadIdx.x * 8;
  const int rest = G.mt * G.nt - G.full;
  int m0, n0;
  tile_at<TN>(G, G.full + r, m0, n0);
  const int m = m0 + at / TN, n = n0 + at % TN;
  if (m >= G.M || n >= G.N) return;
  float v[8] = {};
  for (int z = 0; z < G.splits; ++z) {
    const float4* p = (const float4*)(G.part + (int64_t)(z * rest + r) * kTile + at);
    const float4 a = p[0], b = p[1];
    v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
    v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
  }
  finish16<T, 8>(G, m, n, v);
}

template <typename T, bool KA, bool KB, bool RAG>
void launch_wide(const Gemm16P& G, const WidePlan& p, hipStream_t s) {
  static uint64_t square_seen = 0, tall_seen = 0;
  const int blocks = p.full + (G.mt * G.nt - p.full) * p.splits;
  if (p.tn == 256) {
    constexpr int smem = 2 * (kWideM + 256) * kKS * 2;
    const auto kern = gemm16_square_kernel<T, KA, KB, RAG>;
    raise_lds_limit(&square_seen, smem, kern);
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), smem, s, G);
  } else {
    constexpr int smem = Tall<T, KA, KB, RAG>::kLds;
    const auto kern = gemm16_tall_kernel<T, KA, KB, RAG>;
    raise_lds_limit(&tall_seen, smem, kern);
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(512), smem, s, G);
  }
}
template <typename T>
void launch_orders(const Gemm16P& G, const WidePlan& p, int ka, int kb, hipStream_t s) {
  const bool rag = G.K % kKS != 0;
  if (ka && kb) rag ? launch_wide<T, true, true, true>(G, p, s) : launch_wide<T, true, true, false>(G, p, s);
  else if (ka) rag ? launch_wide<T, true, false, true>(G, p, s) : launch_wide<T, true, false, false>(G, p, s);
  else if (kb) rag ? launch_wide<T, false, true, true>(G, p, s) : launch_wide<T, false, true, false>(G, p, s);
  else rag ? launch_wide<T, false, false, true>(G, p, s) : launch_wide<T, false, false, false>(G, p, s);
  if (p.splits > 1) {
    const int rest = G.mt * G.nt - p.full;
    if (p.tn == 256) hipLaunchKernelGGL((gemm16_parts_kernel<T, 256>), dim3(rest * (kWideM * 256 / 2048)), dim3(256), 0, s, G);
    else hipLaunchKernelGGL((gemm16_parts_kernel<T, 128>), dim3(rest * (kWideM * 128 / 2048)), dim3(256), 0, s, G);
  }
}

}  // namespace

template <typename T>
void launch_wide_type(const Gemm16P& G, const WidePlan& p, int ka, int kb, hipStream_t s) {
  launch_orders<T>(G, p, ka, kb, s);
}

}  // namespace mega
