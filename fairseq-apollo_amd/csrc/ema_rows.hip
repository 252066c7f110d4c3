// Moving-average layer on the matrix cores for [B, D, L] rows of any activation type, parallel over time:
//   y = k * x + omega x  with the carried state, per channel (fairseq/modules/base_moving_average.py:120-172;
//   the reference's fused convolution serves fp32 / fp16 / bf16 alike, ops/fftconv_kernel.cu:214-269).
// A wave owns one block of 1024 tokens of a (batch, channel) row = 16 segments of 64 tokens = the 16 MFMA columns; per
// 32-token tile  y = K x + C h_start,  h_end = Q h_start + P x  with the K / P / C operand images of
// ema_image_kernel (csrc/ema_mfma.h).  fp32 / fp16 activations run on fp16 operands: x = x_hi + x_lo as two fp16
// terms (22 significant bits; one term for fp16 input), K, P and C as two fp16 terms, the states go into the C
// product as two terms: every product is formed as hi*hi + lo*hi + hi*lo (error ~ 2^-22), accumulation and the
// recurrences are fp32.  bf16 activations run on the bf16 operands of the other kernels (K, P two terms).
// A workgroup owns whole rows, a wave for each of their (at most 16) blocks and for both directions of a two-sided layer: x is
// read once, every wave leaves its block's end states from a zero start in LDS, and behind one barrier adds the earlier
// blocks' up with the powers of q^1024, starts its segments from the right state and writes y once.
#include "ema_mfma.h"
#include "tsn_common.h"

namespace mega {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kRBlk = 1024;               // tokens per block
constexpr int kRMost = 16;                // blocks of a row
constexpr int kRWaveLds = 4096;           // two 16-bit planes of the block, later y as fp32
constexpr int kRecF = 2 * kNS;            // floats of an end state: 16 complex values

struct RowsArgs {
  const void* x;         // [B, D, L] rows: element (b, d, t) at b * sxb + d * sxd + t
  void* y;
  int64_t sxb, sxd, syb, syd;
  const uint8_t* mask;   // [B, L] or null
  const uint4* image;    // [K][kImgSlots][64]
  const float* omega;    // [D]: residual of masked tokens (they do not enter the convolution), or null
  const float* h_in;     // [B, D, N, 2] or null
  float* h_out;          // [B, D, N, 2] or null
  int D, N, L, S, R;     // S: blocks of a row
  int is_complex;
};

__device__ __forceinline__ uint4 img_slot(const char* base, int slot, uint32_t lane_off) {
  return *(const uint4*)(base + slot * 1024 + lane_off);
}

__device__ __forceinline__ void load_c4(const char* base, int slot, uint32_t lane_off, float (&re)[4], float (&im)[4]) {
  const uint4 a = img_slot(base, slot, lane_off), b = img_slot(base, slot + 1, lane_off);
  re[0] = __uint_as_float(a.x); im[0] = __uint_as_float(a.y);
  re[1] = __uint_as_float(a.z); im[1] = __uint_as_float(a.w);
  re[2] = __uint_as_float(b.x); im[2] = __uint_as_float(b.y);
  re[3] = __uint_as_float(b.z); im[3] = __uint_as_float(b.w);
}

// the four states (2r, 2r+1, 8+2r, 9+2r) of row block r from table `tab` of the compact slot
__device__ __forceinline__ void load_cmp(const char* base, int tab, uint32_t r_off, float (&re)[4], float (&im)[4]) {
  const uint4 a = *(const uint4*)(base + kSlotCmp * 1024 + tab * 128 + r_off);
  const uint4 b = *(const uint4*)(base + kSlotCmp * 1024 + tab * 128 + 64 + r_off);
  re[0] = __uint_as_float(a.x); im[0] = __uint_as_float(a.y);
  re[1] = __uint_as_float(a.z); im[1] = __uint_as_float(a.w);
  re[2] = __uint_as_float(b.x); im[2] = __uint_as_float(b.y);
  re[3] = __uint_as_float(b.z); im[3] = __uint_as_float(b.w);
}

// one step of the inclusive scan of h_j = R h_{j-1} + e_j across the 16 lanes of a row
template <int CTRL>
__device__ __forceinline__ void scan_step(float (&er)[4], float (&ei)[4], const float (&rr)[4], const float (&ri)[4]) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float tr = dpp_f<CTRL>(er[u]), ti = dpp_f<CTRL>(ei[u]);
    er[u] = fmaf(tr, rr[u], fmaf(-ti, ri[u], er[u]));
    ei[u] = fmaf(ti, rr[u], fmaf(tr, ri[u], ei[u]));
  }
}

__device__ __forceinline__ void csquare(const float (&ar)[4], const float (&ai)[4], float (&br)[4], float (&bi)[4]) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    br[u] = ar[u] * ar[u] - ai[u] * ai[u];
    bi[u] = 2.f * ar[u] * ai[u];
  }
}

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;

// F16: fp16 operands (fp32 / fp16 activations), else bf16
template <bool F16>
__device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
  if (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// v as hi + lo in the operand type (16-bit patterns)
template <bool F16>
__device__ __forceinline__ void split16(float v, uint16_t* hi, uint16_t* lo) {
  if (F16) {
    const _Float16 h = (_Float16)v;
    *hi = __builtin_bit_cast(uint16_t, h);
    *lo = __builtin_bit_cast(uint16_t, (_Float16)(v - (float)h));
  } else {
    const __bf16 h = (__bf16)v;
    *hi = __builtin_bit_cast(uint16_t, h);
    *lo = __builtin_bit_cast(uint16_t, (__bf16)(v - (float)h));
  }
}

// byte offset of token i of the block inside a bf16 plane: segment row of 128 bytes, 16-byte chunks
// XOR-swizzled by the segment so that the B-operand reads of the 16 segments fall on different banks
__device__ __forceinline__ int plane_off(int i) {
  const int j = i >> 6, c8 = (i >> 3) & 7, e = i & 7;
  return j * 128 + ((c8 ^ (j >> 1)) << 4) + e * 2;
}

// eight consecutive tokens in the other order
__device__ __forceinline__ uint4 turned(uint4 v) {
  return make_uint4((v.w >> 16) | (v.w << 16), (v.z >> 16) | (v.z << 16), (v.y >> 16) | (v.y << 16), (v.x >> 16) | (v.x << 16));
}

// NX: terms of x; F16: fp16 operands; VEC: rows and mask are aligned for four tokens per access and L is a multiple of 4; BOTH:
// a two-sided layer (the direction back in time walks the row's blocks from behind, the tokens beyond L zeros in front
// of it, with coefficient rows D .. 2D - 1).
// What bounds it is a wave's chain (row in, products, scan, barrier, products, row out), so waves of many rows run beside each
// other.  1150 vector instructions and 72 products a wave of two directions are 8 us of 1 x 256 x 16384 (the rest: one round trip
// in, one out).  us, in two launches of a wave a direction and here: 1 x 256 x 16384 fp32 masked 23.7, 17.0; 8 x 1024 x 4096
// 180, 104; 8 x 128 x 3999 (its directions apart, partial sums in memory) 54, 19; one-sided 1 x 256 x 16384 16.5, 12.4.
template <typename T, int NX, bool F16, bool VEC, bool BOTH, int MAXW>
__global__ __launch_bounds__(64 * MAXW, MAXW == 4 ? 3 : 4) void ema_rows_kernel(const RowsArgs A) {
  constexpr int ND = BOTH ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) char lds[];   // [waves][kRWaveLds], then [waves][ND][kRecF] end states
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int waves = (int)blockDim.x >> 6, rows = waves / A.S;
  const int mine = wave / A.S, m = wave - mine * A.S;   // the row within the workgroup, the block of memory
  const int wrow = (int)blockIdx.x * rows + mine;
  const bool live = wrow < A.R;
  const int row = min(wrow, A.R - 1);                   // (waves meet at a barrier: one of no row repeats the last)
  const int b = row / A.D, d = row - b * A.D;
  const int j = lane & 15, r = lane >> 4;
  char* plane = lds + wave * kRWaveLds;                 // hi plane at 0, lo plane at 2048
  float* recs = (float*)(lds + waves * kRWaveLds);
  const T* xr = (const T*)A.x + (size_t)b * A.sxb + (size_t)d * A.sxd;
  const uint32_t loff = (uint32_t)lane * 16, roff = (uint32_t)r * 16;
  const uint8_t* mrow = A.mask ? A.mask + (size_t)b * A.L : nullptr;
  const int i0 = m * kRBlk;                             // first token of the block
  constexpr int kSP = F16 ? kSlotP16 : kSlotP, kSK = F16 ? kSlotK16 : kSlotK, kSC = F16 ? kSlotC16 : kSlotC;
  constexpr int NC = F16 ? 2 : 1;                       // terms of C and of the state operand
  const char* img[ND];
#pragma unroll
  for (int e = 0; e < ND; ++e) img[e] = (const char*)A.image + (size_t)(e * A.D + d) * kImgRowBytes;

  // ---- the block of x into LDS as two 16-bit planes (masked and out-of-range tokens as zeros); every load of
  // the block is requested before the first one is used, the operands of the first products with them
  constexpr int NL = VEC ? 4 : 8, W = VEC ? 4 : 1;      // accesses in flight, tokens of one
  uint4 P[ND][2][2];
#pragma unroll 1
  for (int k0 = 0; k0 < kRBlk / 64 / W; k0 += NL) {
    Vec<T, W> xq[NL];
    uint32_t mq[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int t = min(i0 + ((k0 + k) * 64 + lane) * W, A.L - W);
      xq[k] = *(const Vec<T, W>*)(xr + t);
      if constexpr (VEC) mq[k] = mrow ? *(const uint32_t*)(mrow + t) : 0u;
      else mq[k] = mrow ? mrow[t] : 0u;
    }
    if (VEC || k0) {                                    // (k0: the last round)
#pragma unroll
      for (int e = 0; e < ND; ++e)
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
          for (int mb = 0; mb < 2; ++mb) P[e][w][mb] = img_slot(img[e], kSP + 2 * w + mb, loff);
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int i = ((k0 + k) * 64 + lane) * W;
      const bool in = i0 + i < A.L;
      uint16_t hi[W], lo[W];
#pragma unroll
      for (int u = 0; u < W; ++u) {
        const bool masked = ((mq[k] >> (8 * u)) & 0xffu) != 0u;
        split16<F16>((in && !masked) ? to_float(xq[k].v[u]) : 0.f, &hi[u], &lo[u]);
      }
      const int o = plane_off(i);
      if constexpr (VEC) {
        *(uint2*)(plane + o) = make_uint2(hi[0] | ((uint32_t)hi[1] << 16), hi[2] | ((uint32_t)hi[3] << 16));
        if (NX > 1) *(uint2*)(plane + 2048 + o) = make_uint2(lo[0] | ((uint32_t)lo[1] << 16), lo[2] | ((uint32_t)lo[3] << 16));
      } else {
        *(uint16_t*)(plane + o) = hi[0];
        if (NX > 1) *(uint16_t*)(plane + 2048 + o) = lo[0];
      }
    }
  }
  __builtin_amdgcn_wave_barrier();                      // the wave's own LDS writes precede its reads
  // tokens 8 r .. 8 r + 7 of tile t of segment j, in direction e's order
  auto tokens = [&](int e, int t, int term) {
    const int jm = e ? 15 - j : j, c = e ? 7 - (4 * t + r) : 4 * t + r;
    const uint4 v = *(const uint4*)(plane + term * 2048 + jm * 128 + ((c ^ (jm >> 1)) << 4));
    return e ? turned(v) : v;
  };

  // ---- end states of the segments from a zero start: F after the first tile, E after the second
  float Fr[ND][4], Fi[ND][4], hr[ND][4], hi[ND][4];
  float Er[4], Ei[4];
#pragma unroll
  for (int e = 0; e < ND; ++e) {
    float Qr[4], Qi[4], Rr[4], Ri[4], R2r[4], R2i[4];
    load_cmp(img[e], kCmpQ32, roff, Qr, Qi);
    load_cmp(img[e], kCmpRS, roff, Rr, Ri);
    const int steps = __builtin_amdgcn_readfirstlane(*(const int*)(img[e] + kSlotCmp * 1024 + kCmpReach * 128));
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint4 Xh = tokens(e, t, 0);
      f32x4 S0 = {0.f, 0.f, 0.f, 0.f}, S1 = {0.f, 0.f, 0.f, 0.f};
      S0 = mfma<F16>(P[e][0][0], Xh, S0);
      S1 = mfma<F16>(P[e][0][1], Xh, S1);
      S0 = mfma<F16>(P[e][1][0], Xh, S0);
      S1 = mfma<F16>(P[e][1][1], Xh, S1);
      if (NX > 1) {
        const uint4 Xl = tokens(e, t, 1);
        S0 = mfma<F16>(P[e][0][0], Xl, S0);
        S1 = mfma<F16>(P[e][0][1], Xl, S1);
      }
      const float sr[4] = {S0[0], S0[2], S1[0], S1[2]};
      const float si[4] = {S0[1], S0[3], S1[1], S1[3]};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (t == 0) {
          Fr[e][u] = sr[u];
          Fi[e][u] = si[u];
        } else {
          Er[u] = fmaf(Qr[u], Fr[e][u], fmaf(-Qi[u], Fi[e][u], sr[u]));
          Ei[u] = fmaf(Qr[u], Fi[e][u], fmaf(Qi[u], Fr[e][u], si[u]));
        }
      }
    }
    // inclusive scan over the 16 segments by doubling; a step over d segments is skipped when |q|^(64 d) < 2^-24
    // for every state of the channel
    if (steps > 0) {
      scan_step<0x111>(Er, Ei, Rr, Ri);
      if (steps > 1) {
        csquare(Rr, Ri, R2r, R2i);
        scan_step<0x112>(Er, Ei, R2r, R2i);
        if (steps > 2) {
          csquare(R2r, R2i, Rr, Ri);
          scan_step<0x114>(Er, Ei, Rr, Ri);
          if (steps > 3) {
            csquare(Rr, Ri, R2r, R2i);
            scan_step<0x118>(Er, Ei, R2r, R2i);
          }
        }
      }
    }
    // lane 15 of a row holds the block's end state from a zero start; segment j starts from segment j - 1's
    if (j == 15) {
      float* rec = recs + (wave * ND + e) * kRecF;
      *(float4*)(rec + (2 * r) * 2) = make_float4(Er[0], Ei[0], Er[1], Ei[1]);
      *(float4*)(rec + (8 + 2 * r) * 2) = make_float4(Er[2], Ei[2], Er[3], Ei[3]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      hr[e][u] = dpp_f<0x111>(Er[u]);
      hi[e][u] = dpp_f<0x111>(Ei[u]);
    }
  }
  __syncthreads();

  // ---- y = K x + C h per tile and direction
  const int nn[4] = {2 * r, 2 * r + 1, 8 + 2 * r, 9 + 2 * r};
  f32x4 Y[ND][2][2];
#pragma unroll
  for (int e = 0; e < ND; ++e) {
    uint4 Kw[2][2], Cw[NC][2];
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) Kw[w][mb] = img_slot(img[e], kSK + 2 * w + mb, loff);
#pragma unroll
    for (int w = 0; w < NC; ++w)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) Cw[w][mb] = img_slot(img[e], kSC + 2 * w + mb, loff);
    float Qr[4], Qi[4];
    load_cmp(img[e], kCmpQ32, roff, Qr, Qi);
    // what the block inherits: h_start = sum_d (q^1024)^d T_{s-1-d} (+ (q^1024)^s h_in); lane (j, r) holds
    // the term d = j for its four states, the 16 lanes of a row add up
    const int s = e ? A.S - 1 - m : m;                  // blocks before this one
    const float* h_in = e ? nullptr : A.h_in;
    const int nterms = s + (h_in ? 1 : 0);
    float Cr[4] = {0.f, 0.f, 0.f, 0.f}, Ci[4] = {0.f, 0.f, 0.f, 0.f};
    if (nterms > 0) {
      float RWJr[4], RWJi[4], RJr[4], RJi[4], tr[4], ti[4];
      load_c4(img[e], kSlotRWJ, loff, RWJr, RWJi);      // (q^1024)^j of this lane's states
      load_c4(img[e], kSlotRJ, loff, RJr, RJi);
      const int look = __builtin_amdgcn_readfirstlane(*(const int*)(img[e] + kSlotCmp * 1024 + kCmpReach * 128 + 4));
#pragma unroll
      for (int u = 0; u < 4; ++u) tr[u] = ti[u] = 0.f;
      if (j < s) {
        const float* rec = recs + ((e ? wave + 1 + j : wave - 1 - j) * ND + e) * kRecF;
        const float4 a = *(const float4*)(rec + (2 * r) * 2), c = *(const float4*)(rec + (8 + 2 * r) * 2);
        tr[0] = a.x; ti[0] = a.y; tr[1] = a.z; ti[1] = a.w;
        tr[2] = c.x; ti[2] = c.y; tr[3] = c.z; ti[3] = c.w;
      } else if (h_in && j == s) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (nn[u] < A.N) {
            const size_t o = (((size_t)b * A.D + d) * A.N + nn[u]) * 2;
            tr[u] = h_in[o];
            ti[u] = A.is_complex ? h_in[o + 1] : 0.f;
          }
        }
      }
      const bool have = j < nterms && j < look;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float cr = RWJr[u] * tr[u] - RWJi[u] * ti[u];
        const float ci = RWJr[u] * ti[u] + RWJi[u] * tr[u];
        Cr[u] = group_sum<16>(have ? cr : 0.f);
        Ci[u] = group_sum<16>(have ? ci : 0.f);
      }
      // start state of segment j: segment j - 1's end plus (q^64)^j times the inherited state
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        hr[e][u] = fmaf(RJr[u], Cr[u], fmaf(-RJi[u], Ci[u], hr[e][u]));
        hi[e][u] = fmaf(RJr[u], Ci[u], fmaf(RJi[u], Cr[u], hi[e][u]));
      }
    }
    if (!BOTH && A.h_out && m == A.S - 1 && j == 15 && live) {
      // state after the last token: the block's own end state plus q^1024 times what it inherited
      float RWr[4], RWi[4];
      load_cmp(img[e], kCmpRW, roff, RWr, RWi);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (nn[u] < A.N) {
          const size_t o = (((size_t)b * A.D + d) * A.N + nn[u]) * 2;
          A.h_out[o] = fmaf(RWr[u], Cr[u], fmaf(-RWi[u], Ci[u], Er[u]));
          A.h_out[o + 1] = fmaf(RWr[u], Ci[u], fmaf(RWi[u], Cr[u], Ei[u]));
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint4 Xh = tokens(e, t, 0);
      uint16_t hh[8], hl[8];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        split16<F16>(hr[e][u], &hh[2 * u], &hl[2 * u]);
        split16<F16>(hi[e][u], &hh[2 * u + 1], &hl[2 * u + 1]);
      }
      const uint4 Hh = make_uint4(hh[0] | ((uint32_t)hh[1] << 16), hh[2] | ((uint32_t)hh[3] << 16),
                                  hh[4] | ((uint32_t)hh[5] << 16), hh[6] | ((uint32_t)hh[7] << 16));
      f32x4 Y0 = {0.f, 0.f, 0.f, 0.f}, Y1 = {0.f, 0.f, 0.f, 0.f};
      Y0 = mfma<F16>(Cw[0][0], Hh, Y0);
      Y1 = mfma<F16>(Cw[0][1], Hh, Y1);
      Y0 = mfma<F16>(Kw[0][0], Xh, Y0);
      Y1 = mfma<F16>(Kw[0][1], Xh, Y1);
      Y0 = mfma<F16>(Kw[1][0], Xh, Y0);
      Y1 = mfma<F16>(Kw[1][1], Xh, Y1);
      {
        // the states as two terms in either operand type (one bf16 term leaves 2^-9 of sum |gamma q h| at the first
        // tokens of every tile, which shows where the states cancel in the sum over the states)
        const uint4 Hl = make_uint4(hl[0] | ((uint32_t)hl[1] << 16), hl[2] | ((uint32_t)hl[3] << 16),
                                    hl[4] | ((uint32_t)hl[5] << 16), hl[6] | ((uint32_t)hl[7] << 16));
        if (NC > 1) {
          Y0 = mfma<F16>(Cw[NC - 1][0], Hh, Y0);
          Y1 = mfma<F16>(Cw[NC - 1][1], Hh, Y1);
        }
        Y0 = mfma<F16>(Cw[0][0], Hl, Y0);
        Y1 = mfma<F16>(Cw[0][1], Hl, Y1);
      }
      if (NX > 1) {
        const uint4 Xl = tokens(e, t, 1);
        Y0 = mfma<F16>(Kw[0][0], Xl, Y0);
        Y1 = mfma<F16>(Kw[0][1], Xl, Y1);
      }
      Y[e][t][0] = Y0;
      Y[e][t][1] = Y1;
      if (t == 0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float nr = fmaf(Qr[u], hr[e][u], fmaf(-Qi[u], hi[e][u], Fr[e][u]));
          hi[e][u] = fmaf(Qr[u], hi[e][u], fmaf(Qi[u], hr[e][u], Fi[e][u]));
          hr[e][u] = nr;
        }
      }
    }
  }
  // ---- y through LDS (fp32; the wave's x is used up; the 16-byte pieces of a segment's 256 bytes are XOR-swizzled by the
  // segment so that the 16 segments' stores fall on different banks) and out in whole runs of tokens
  float* ys = (float*)plane;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      *(float4*)(ys + j * 64 + (((t * 8 + h * 4 + r) ^ j) & 15) * 4) = make_float4(Y[0][t][h][0], Y[0][t][h][1], Y[0][t][h][2], Y[0][t][h][3]);
  if constexpr (BOTH) {
    __builtin_amdgcn_wave_barrier();
    // in the order of memory: walking piece (j, c) is piece (15 - j, 15 - c) there, its four tokens turned
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int jm = 15 - j, cm = 15 - (t * 8 + h * 4 + r);
        float4* at = (float4*)(ys + jm * 64 + ((cm ^ jm) & 15) * 4);
        const float4 o = *at;
        *at = make_float4(o.x + Y[1][t][h][3], o.y + Y[1][t][h][2], o.z + Y[1][t][h][1], o.w + Y[1][t][h][0]);
      }
  }
  __builtin_amdgcn_wave_barrier();
  T* yr = (T*)A.y + (size_t)b * A.syb + (size_t)d * A.syd;
  const bool resid = A.omega && A.mask;                  // masked tokens keep their residual omega x
  const float om = resid ? A.omega[d] : 0.f;
#pragma unroll 1
  for (int k0 = 0; k0 < kRBlk / 64 / W; k0 += NL) {
    Vec<T, W> xo[NL];
    uint32_t mq[NL];
    if (resid) {
#pragma unroll
      for (int k = 0; k < NL; ++k) {
        const int t = min(i0 + ((k0 + k) * 64 + lane) * W, A.L - W);
        xo[k] = *(const Vec<T, W>*)(xr + t);
        if constexpr (VEC) mq[k] = *(const uint32_t*)(mrow + t);
        else mq[k] = mrow[t];
      }
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int i = ((k0 + k) * 64 + lane) * W, w = i0 + i;
      const float* at = ys + (i & ~63) + (((((i & 63) >> 2) ^ (i >> 6)) & 15) << 2) + (i & 3);
      float v[W];
      if constexpr (VEC) {
        const float4 q = *(const float4*)at;
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
      } else {
        v[0] = *at;
      }
      Vec<T, W> o;
#pragma unroll
      for (int u = 0; u < W; ++u) {
        if (resid) v[u] += (mq[k] >> (8 * u)) & 0xffu ? om * to_float(xo[k].v[u]) : 0.f;
        o.v[u] = from_float<T>(v[u]);
      }
      if (live && w < A.L) *(Vec<T, W>*)(yr + w) = o;
    }
  }
}

template <typename T, int NX, bool F16, bool VEC, bool BOTH>
int launch_rows_v(const RowsArgs& A, hipStream_t s) {
  static uint64_t attr_seen = 0;
  // two directions want 150 registers: workgroups of few waves may have them (8 x 256 x 1024, two-sided 8.6 us, 9.9 at 128);
  // one direction is quicker with more waves beside each other (4 x 1024 x 2048 fp16 15.3, 16.8).  Longer rows have up to 16
  // waves a workgroup and so 128 registers: with four tokens an access 9 of them (fp32), 10 (fp16) or 4 (bf16) live in scratch
  // with two directions, 4 with one (fp32, fp16).
  auto kern = ema_rows_kernel<T, NX, F16, VEC, BOTH, kRMost>;
  if constexpr (BOTH) {
    if (A.S <= 4) kern = ema_rows_kernel<T, NX, F16, VEC, BOTH, 4>;
  }
  const int rows = A.S < 4 ? 4 / A.S : 1, waves = rows * A.S;     // workgroups of three waves and more
  constexpr int each = kRWaveLds + (BOTH ? 2 : 1) * kRecF * 4;
  if (waves * each > 64 * 1024) raise_lds_limit(&attr_seen, kRMost * each, ema_rows_kernel<T, NX, F16, VEC, BOTH, kRMost>);
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(A.R, rows)), dim3(64 * waves), waves * each, s, A);
  MEGA_CHECK_LAUNCH("ema_fwd (rows on the matrix cores)");
  return MEGA_OK;
}

// four tokens per access when every row and the mask start on such a boundary
template <typename T>
bool rows_vec_ok(const RowsArgs& A) {
  const size_t al = 4 * sizeof(T);
  return A.L % 4 == 0 && A.L >= 4 && ((uintptr_t)A.x % al) == 0 && ((uintptr_t)A.y % al) == 0 &&
         A.sxb % 4 == 0 && A.sxd % 4 == 0 && A.syb % 4 == 0 && A.syd % 4 == 0 &&
         (!A.mask || ((uintptr_t)A.mask % 4) == 0);
}

template <typename T, int NX, bool F16>
int launch_rows(const RowsArgs& A, bool both, hipStream_t s) {
  const bool vec = rows_vec_ok<T>(A);
  if (both) return vec ? launch_rows_v<T, NX, F16, true, true>(A, s) : launch_rows_v<T, NX, F16, false, true>(A, s);
  return vec ? launch_rows_v<T, NX, F16, true, false>(A, s) : launch_rows_v<T, NX, F16, false, false>(A, s);
}

}  // namespace

// [B, D, L] rows on both sides (time contiguous), at most 16 blocks of 1024 tokens, ndim <= 16, no truncation
bool ema_rows_covers(int dtype, int64_t sxb, int64_t sxd, int64_t sxl, int64_t syb, int64_t syd, int64_t syl,
                     int64_t B, int64_t D, int64_t N, int64_t L, int64_t Lk, const float* h_out) {
  if (N > kNS || Lk > 0 || sxl != 1 || syl != 1 || L < 64) return false;
  if (ceil_div(L, kRBlk) > kRMost) return false;
  if (h_out && L % kRBlk != 0) return false;           // the state after the last token of a partial block
  if (B * D >= (int64_t)1 << 26) return false;          // the grids stay below 2^31 workgroups
  (void)dtype; (void)sxb; (void)sxd; (void)syb; (void)syd;
  return true;
}

int ema_rows_run(const void* x, void* y, int dtype, int64_t sxb, int64_t sxd, int64_t syb, int64_t syd,
                 const void* image, int is_complex, const float* omega, const uint8_t* mask, const float* h_in,
                 float* h_out, int64_t B, int64_t D, int64_t N, int64_t L, int bidirectional, hipStream_t s) {
  RowsArgs A;
  A.x = x; A.y = y; A.sxb = sxb; A.sxd = sxd; A.syb = syb; A.syd = syd; A.mask = mask;
  A.image = (const uint4*)image; A.D = (int)D; A.N = (int)N; A.L = (int)L;
  A.S = (int)ceil_div(L, kRBlk); A.R = (int)(B * D); A.is_complex = is_complex;
  A.omega = mask ? omega : nullptr; A.h_in = h_in; A.h_out = h_out;
  switch (dtype) {
    case MEGA_F32: return launch_rows<float, 2, true>(A, bidirectional != 0, s);
    case MEGA_F16: return launch_rows<f16_t, 1, true>(A, bidirectional != 0, s);
    default: return launch_rows<bf16_t, 1, false>(A, bidirectional != 0, s);
  }
}

}  // namespace mega
