// TimestepNorm -> moving-average layer in one kernel (gfx950, bf16 / fp16 / fp32 activations, 32 to 128 channels per
// norm group, ndim <= 16, optional padding mask, rows of any length up to 16 blocks): what MovingAverageGatedAttention.forward does at
// fairseq/modules/moving_average_gated_attention.py:304-315 (x = norm(x); mx = move(x^T)) with
// TimestepNorm per fairseq/csrc/ops/timestep_norm.cc:218-316 and the layer per
// fairseq/modules/base_moving_average.py:120-172.  x is read once, xn (the norm's output, which the
// layer also feeds to v_proj) and y are written once.
//
// A workgroup (16 waves) owns one (batch row, up to 64 channels of a norm group, block of 1024 tokens): with 64
// channels of 16 bits or 32 of fp32 whole 128-byte lines of x, xn and -- with [B, D, L] rows -- y.  A wider group is
// shared by two to four workgroups, each of which reads the group's whole lines for the moments.  fp32 / fp16
// activations take the moving average's products on fp16 operands of two terms, as ema_rows.hip does (fp32 activations
// as two 16-bit planes of LDS, y back over them as the halves of its words).  The blocks are aligned to the end of the row: a row that is
// not a whole number of blocks starts inside block 0, behind virtual tokens that count as padding.
//   1. load the block, per-token moments of the group (packed dot products + DPP), Welford scan over
//      the block's tokens (padding weighs nothing), publish the block aggregate, fold the earlier blocks'
//      aggregates of the same (row, group) and the prior state into the carry-in, finish mean / rstd per token;
//   2. normalise from registers, store xn (zeros at padding), and stage xn (bf16, as the layer sees it) into LDS
//      transposed to channel rows;
//   3. per channel (4 per wave), with the operand images of ema_image_kernel:
//        phase A: end states of the 16 segments (64 tokens = 2 tiles each) from a zero start on the
//                 matrix cores, scanned across the 16 lanes of a DPP row; the block's end state from a
//                 zero start is parked in LDS and published;
//      look-back: the earlier blocks' end states (and the caller's carried state) folded into the
//                 block's start state, h_start = sum_d (q^1024)^d E_{s-1-d}, parked over the end states;
//        phase B: the segment scan again, segment start state = what the segment before left + (q^64)^j h_start,
//                 y_tile = K x_tile + C h (h as one bf16 term, two for slow poles and few states), bf16, back into LDS over x, and
//                 out as whole rows.
// Blocks map to workgroup ids time-major and workgroups are dispatched in id order, so a block only
// waits for blocks dispatched before it; every wait is bounded and poisons the block's outputs with
// NaN (and sets the error word of the workspace header) when it gives up.
#include <type_traits>

#include "ema_mfma.h"
#include "tsn_common.h"

// Phase markers: a profiling build defines MEGA_FTR(k) to stamp a clock per workgroup; no-ops here.
#ifndef MEGA_FTR
#define MEGA_FTR(k)
#define MEGA_FTR_END()
#endif
#ifndef MEGA_FTR2
#define MEGA_FTR2(k)
#endif

// Held-back block starts of a one-round launch: ticks of 10 ns per block index (mod 4), and the least share of the
// compute units the launch has to fill (1 / MEGA_FUSED_STAGGER_FILL) for them to be used.
#ifndef MEGA_FUSED_STAGGER
#define MEGA_FUSED_STAGGER 60
#endif
#ifndef MEGA_FUSED_STAGGER_FILL
#define MEGA_FUSED_STAGGER_FILL 4
#endif
#ifndef MEGA_FUSED_STAGGER_BLOCKS
#define MEGA_FUSED_STAGGER_BLOCKS 4
#endif
#ifndef MEGA_FUSED_TWO_TERMS
#define MEGA_FUSED_TWO_TERMS 0
#endif

namespace mega {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kFW = 16;                       // waves per workgroup
constexpr int kFT = kFW * 64;                 // threads
constexpr int kFSeg = 1024;                   // tokens per block: 16 segments x 2 tiles x 32
constexpr int kFRow = kFSeg * 2;              // bytes of one channel row of a 16-bit plane in LDS
constexpr int kFMaxBlocks = 16;               // terms of the look-back sum (earlier blocks + the carried state): one per lane of a row
constexpr int kFTabs = 2;                     // per-state multiplier tables kept in LDS: q^32, q^64

static_assert(kSEGT == 2, "the fused kernel uses the q^64 segment multipliers of the image");

// What follows from the activation type and the CW channels of a workgroup (PARTS workgroups share a norm group).
template <typename T, int CW, int PARTS>
struct Geo {
  static constexpr bool F16 = !__is_same(T, bf16_t);          // operands of the moving average: fp16 or bf16
  static constexpr int NX = sizeof(T) == 4 ? 2 : 1;           // 16-bit terms of x, a plane of the tile each
  static constexpr int NC = F16 ? 2 : kNWC;                   // terms of the C operand
  static constexpr int VPP = 16 / (int)sizeof(T);             // values of a 16-byte piece
  static constexpr int PPT = CW / VPP;                        // pieces of a token
  static constexpr int PL = PPT <= 4 ? 4 : 8;                 // lanes of a token (those beyond PPT idle in the norm)
  static constexpr int TPR = kFT / PL;                        // tokens per round of loads
  static constexpr int NLD = kFSeg / TPR;                     // rounds = pieces per thread
  static constexpr int CPW = CW / kFW;                        // channels per wave
  static constexpr int GC = CW * PARTS;                       // channels per norm group
  static constexpr int Plane = CW * kFRow + (CW / 4) * 16;
  static constexpr int Tile = NX * Plane;
  static constexpr int RecW = 4 + CW * kNS * 2;               // 64-bit words per block record: n, mean, var, pad, end states
  static constexpr size_t Smem = (size_t)Tile + 2 * kFSeg * 4 + 64 + (size_t)kFTabs * CW * 128 + CW * 8;
  static_assert(CW % kFW == 0 && CW <= 64 && PPT <= 8, "one to four channels per wave, at most 128 bytes of a token");
  static_assert(Smem <= 160 * 1024, "LDS of one workgroup");
};

struct FusedArgs {
  const void* x;         // [B, L, D]
  void* xn;              // [B, L, D]
  void* y;               // strides (syb, syd, syl): [B, D, L] rows (syl == 1) or [B, L, D] (syd == 1)
  int64_t syb, syd, syl;
  const int64_t* prev_count;
  const float* prev_mean;
  const float* prev_var;
  int64_t* count;
  float* mean;
  float* var;
  const float* gamma;    // [D] (weight + 1)
  const float* beta;     // [D]
  const uint8_t* mask;   // [B, L], nonzero = padding: no part in the statistics, xn = 0; or null
  const uint4* image;    // [D][kImgSlots][64]
  const float* h_in;     // [B, D, N, 2] or null
  float* h_out;          // [B, D, N, 2] or null
  float* cummean;        // [B, L, G] running mean / rstd of every token, kept for the norm's backward pass; or null
  float* cumrstd;
  TsnHeader* hdr;
  unsigned long long* rec;   // [B * D / CW][S + 1][RecW]; slot S: the caller's carried state, put there by block 0
  int B, L, D, G, N, S;
  int pad;               // S * 1024 - L virtual tokens in front of every row: the block grid ends at the row's last token
  float eps;
  int is_complex;
  int xcd_map;
  int stagger;           // start of block s held back by (s & 3) * stagger ticks of 10 ns (0: all start at once)
  LookbackLaunch lb;     // status word, poll limit, test hook
};

__device__ __forceinline__ int row_base(int c) { return c * kFRow + (c >> 2) * 16; }

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}

// a pair of values in the 16-bit operand type, rounded to nearest
template <bool F16>
__device__ __forceinline__ uint32_t pack16(float lo, float hi) {
  if constexpr (F16) {
    const f16x2_t v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
  } else {
    const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
}

// the two values of a packed pair
template <bool F16>
__device__ __forceinline__ float2 unpack16(uint32_t w) {
  if constexpr (F16) {
    const f16x2_t v = __builtin_bit_cast(f16x2_t, w);
    return make_float2((float)v[0], (float)v[1]);
  } else {
    return make_float2(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u));
  }
}

template <bool F16>
__device__ __forceinline__ f32x4 mma(uint4 a, uint4 b, f32x4 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ float lane_bcast(float v, int src_lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src_lane << 2, __builtin_bit_cast(int, v)));
}

// one step of the inclusive scan of h_j = R h_{j-1} + e_j across the 16 lanes of a row: lanes take the
// value SH lanes to the left (zero outside the row) times R^SH
template <int CTRL>
__device__ __forceinline__ void scan_step(float (&er)[4], float (&ei)[4], const float (&rr)[4], const float (&ri)[4]) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float tr = dpp_f<CTRL>(er[u]), ti = dpp_f<CTRL>(ei[u]);
    const float nri = -ri[u];
    er[u] = fmaf(tr, rr[u], er[u]);
    er[u] = fmaf(ti, nri, er[u]);
    ei[u] = fmaf(ti, rr[u], ei[u]);
    ei[u] = fmaf(tr, ri[u], ei[u]);
  }
}

__device__ __forceinline__ void csquare(const float (&ar)[4], const float (&ai)[4], float (&br)[4], float (&bi)[4]) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    br[u] = ar[u] * ar[u] - ai[u] * ai[u];
    bi[u] = 2.f * ar[u] * ai[u];
  }
}

// activations leave once and are not read again by this kernel: streaming (non-temporal) stores
#ifndef MEGA_FUSED_NT
#define MEGA_FUSED_NT 1
#endif
__device__ __forceinline__ void store_stream(uint4* p, uint4 v) {
#if MEGA_FUSED_NT
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(__builtin_bit_cast(u32x4, v), (u32x4*)p);
#else
  *p = v;
#endif
}

// slot `slot` of an operand image: uniform base, 32-bit lane offset (scalar-base addressing)
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

// the four states of row block r from table `tab` of the compact slot: two 16-byte pieces that the 16 lanes of
// a row share (one line per table leaves the cache, not a slot)
__device__ __forceinline__ void load_cmp(const char* base, int tab, uint32_t r_off, float (&re)[4], float (&im)[4]) {
  const uint4 a = *(const uint4*)(base + kSlotCmp * 1024 + tab * 128 + r_off);
  const uint4 b = *(const uint4*)(base + kSlotCmp * 1024 + tab * 128 + 64 + r_off);
  re[0] = __uint_as_float(a.x); im[0] = __uint_as_float(a.y);
  re[1] = __uint_as_float(a.z); im[1] = __uint_as_float(a.w);
  re[2] = __uint_as_float(b.x); im[2] = __uint_as_float(b.y);
  re[3] = __uint_as_float(b.z); im[3] = __uint_as_float(b.w);
}

// the same from the copy of tables 0..1 in LDS; row: table * channels + channel
__device__ __forceinline__ void lds_cmp(const char* s_tab, int row, uint32_t r_off, float (&re)[4], float (&im)[4]) {
  const float4 a = *(const float4*)(s_tab + row * 128 + r_off);
  const float4 b = *(const float4*)(s_tab + row * 128 + 64 + r_off);
  re[0] = a.x; im[0] = a.y; re[1] = a.z; im[1] = a.w;
  re[2] = b.x; im[2] = b.y; re[3] = b.z; im[3] = b.w;
}

// LOUT 0: y as [B, D, L] rows; 1: y as [B, L, D].  CW: channels of a workgroup; PARTS: workgroups that share a norm
// group: each reads the group's whole lines for the moments (all add in the same order, so all arrive at the same
// statistics to the last bit) and keeps its own CW channels.
// STAG: the start of block s is held back by s * A.stagger ticks (an instance of its own: the launches that do not
// hold anything back run the code without the wait).
template <typename T, int CW, int PARTS, int LOUT, bool STAG>
__global__ __launch_bounds__(kFT) void norm_ema_fused_kernel(const FusedArgs A) {
  using Gm = Geo<T, CW, PARTS>;
  constexpr bool F16 = Gm::F16;
  constexpr int NX = Gm::NX, NC = Gm::NC, VPP = Gm::VPP, PL = Gm::PL, TPR = Gm::TPR, NLD = Gm::NLD, CPW = Gm::CPW;
  constexpr bool FINE = NX > 1;              // (merges of running statistics)
  constexpr int kParts = PARTS, GC = Gm::GC, kPlane = Gm::Plane, kRecW = Gm::RecW;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* tile = smem;
  float* s_gm = (float*)(smem + Gm::Tile);    // [kFSeg] group mean of a token, later the running mean
  float* s_gv = s_gm + kFSeg;                 // [kFSeg] group variance, later the running rstd
  float* s_wt = s_gv + kFSeg;                 // [4][4] totals of the four scanning waves
  float* s_end = s_gm;                        // [CW][kNS][2] block end states from a zero start (after step 2)
  char* s_tab = (char*)(s_wt + 16);           // [kFTabs][CW][kNS] complex: q^32, q^64 of every channel
  uint2* s_reach = (uint2*)(s_tab + kFTabs * CW * 128);   // [CW] reach of every channel's slowest pole

  const T* const gx = (const T*)A.x;
  T* const gxn = (T*)A.xn;
  T* const gy = (T*)A.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: channel rows and image addresses stay scalar
  const int G = A.G;
  const int U = G * kParts;                              // workgroups per (batch row, block)
  const int BU = A.B * U;
  const int s = (int)blockIdx.x / BU, local = (int)blockIdx.x - s * BU;
  int b, unit;
  if (A.xcd_map) {
    // consecutive workgroup ids go to the 8 XCDs in turn: keep a group's blocks (and with them the operand
    // images of its channels and the lines its two halves share) on one XCD, U / 8 units per XCD
    const int up = U >> 3, xcd = local & 7, slot = local >> 3;
    unit = xcd * up + slot % up;
    b = slot / up;
  } else {
    b = local / U;
    unit = local - b * U;
  }
  const int g = unit / kParts, part = unit - g * kParts;
  const int cb = g * GC + part * CW;                     // the workgroup's first channel
  const uint32_t tag = A.hdr->epoch + 1u;
  // The blocks are aligned to the end of the row: block 0 starts `pad` virtual tokens before the first one (they
  // count as padding: no statistics, zeros into the moving average, nothing stored), so the last block ends at the
  // last token and the state handed back is the state after it.
  const int t0 = s * kFSeg - A.pad;
  const bool front = s == 0 && A.pad > 0;                // uniform: this block holds virtual tokens
  // 16-byte piece of the token's line, token 0 .. TPR - 1 of a round: the lanes of tokens 2m and 2m + 1 are 8 apart
  const int lp = tid & (PL - 1);
  const bool act = Gm::PPT == PL || lp < Gm::PPT;
  const int piece = act ? lp : 0;
  const int tokl = PL == 8 ? tid >> 3 : ((tid >> 4) << 2) | ((tid >> 1) & 2) | ((tid >> 3) & 1);
  // addresses of the block's lines: a uniform base per round of tokens plus one 32-bit lane offset
  const int64_t xblk = ((int64_t)b * A.L + t0) * A.D + (int64_t)cb;      // (negative offsets inside a front block are never used)
  const uint32_t toff = (uint32_t)tokl * (uint32_t)A.D + piece * VPP;
  const size_t brow = (size_t)b * G + g;                 // statistics of the group
  const size_t rrow = brow * kParts + part;              // records of the workgroup (its own copy of the statistics too)
  unsigned long long* const myrec = A.rec + (rrow * (A.S + 1) + s) * kRecW;
  bool poison = false;

  MEGA_FTR(0);
  // A launch of a single round has every workgroup of the chip asking for its block at the same moment, and every
  // block after a row's first then waits for the records of the blocks before it.  Blocks 1..3 of every four ask a
  // little later each (constant 100 MHz clock, a bounded wait): the requests spread out, and the later start is time
  // the block would have spent waiting for those records.
  if (STAG && s != 0) {
    const uint64_t t_end = wall_clock64() + (uint64_t)(s * A.stagger);
    while (wall_clock64() < t_end) __builtin_amdgcn_s_sleep(4);
  }
  // ---- everything the norm needs from memory is requested before the block itself
  const Moments prior = {(float)A.prev_count[b], A.prev_mean[brow], A.prev_var[brow]};
  float gam[VPP], bet[VPP];
  load_params<VPP>(A.gamma + cb + piece * VPP, gam);
  load_params<VPP>(A.beta + cb + piece * VPP, bet);
  uint4 xv[NLD];
  uint4 xo[kParts > 1 ? NLD : 1];
  // the thread's pieces of the lines that begin at element `base`; virtual tokens and idle lanes read as zeros
  auto load_lines = [&](const int64_t base, uint4 (&v)[NLD]) {
    if (!front) {
#pragma unroll
      for (int k = 0; k < NLD; ++k) {
        v[k] = Gm::PPT == PL || act ? *(const uint4*)(gx + base + (int64_t)k * TPR * A.D + toff) : make_uint4(0u, 0u, 0u, 0u);
      }
    } else {
#pragma unroll
      for (int k = 0; k < NLD; ++k)
        v[k] = act && k * TPR + tokl >= A.pad ? *(const uint4*)(gx + base + (int64_t)k * TPR * A.D + toff) : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  const int64_t gblk = xblk - (int64_t)part * CW;        // first channel of the group
  load_lines(xblk, xv);
  // the other half of the group's lines, for the moments only (the workgroup of that half reads the same lines on
  // the same XCD)
  if constexpr (kParts == 2) load_lines(gblk + (1 - part) * CW, xo);
  // padding flags of the thread's tokens (bit k: token k * TPR + tokl): the caller's mask and the virtual
  // tokens of a front block
  uint32_t mbits = 0;
  if (!front) {
    if (A.mask) {
      const uint8_t* mrow = A.mask + (int64_t)b * A.L + t0 + tokl;
#pragma unroll
      for (int k = 0; k < NLD; ++k) mbits |= (mrow[k * TPR] != 0 ? 1u : 0u) << k;
    }
  } else {
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      const bool real = k * TPR + tokl >= A.pad;
      const bool padded = !real || (A.mask && A.mask[(int64_t)b * A.L + t0 + k * TPR + tokl] != 0);
      mbits |= (padded ? 1u : 0u) << k;
    }
  }

  // the per-state multipliers of the workgroup's channels (two lines per channel) go to LDS once
  {
    static_assert(kCmpQ32 == 0 && kCmpRS == 1 && kFTabs == 2, "tables 0..1 of the compact slot are staged");
    const char* ibase = (const char*)A.image + (size_t)cb * kImgRowBytes + kSlotCmp * 1024;
    static_assert(kFTabs * CW * 8 <= kFT, "one piece a thread");
    if (tid < kFTabs * CW * 8) {                    // (table, channel, 16-byte piece)
      const int t = tid / (CW * 8), rem = tid - t * (CW * 8), c = rem >> 3, pc = rem & 7;
      *(uint4*)(s_tab + (t * CW + c) * 128 + pc * 16) = *(const uint4*)(ibase + (size_t)c * kImgRowBytes + t * 128 + pc * 16);
    }
    // and how far every channel's slowest pole reaches (asked for here, used after the norm: no wave waits for it)
    if (tid < CW) s_reach[tid] = *(const uint2*)(ibase + (size_t)tid * kImgRowBytes + kCmpReach * 128);
  }

  // ---- the caller's carried state joins the records the later look-ups read: slot S of the row, written by block 0
  if (s == 0 && A.h_in && tid < CW * 16) {
    const int c = tid >> 4, n = tid & 15;
    float2 v = make_float2(0.f, 0.f);
    if (n < A.N) {
      v = *(const float2*)(A.h_in + (((size_t)b * A.D + cb + c) * A.N + n) * 2);
      if (!A.is_complex) v.y = 0.f;
    }
    unsigned long long* e = A.rec + (rrow * (A.S + 1) + A.S) * kRecW + 4 + ((size_t)c * kNS + n) * 2;
    put_rec(e, tagged(__float_as_uint(v.x), tag));
    put_rec(e + 1, tagged(__float_as_uint(v.y), tag));
  }

  // ---- moments of every token's group (the PL lanes of a line)
  auto keep_moments = [&](const int k, const float m, const float v) {
    if (lp == 0) {
      const bool pad = (mbits >> k) & 1u;
      s_gm[k * TPR + tokl] = pad ? 0.f : m;                         // (whatever x holds there)
      s_gv[k * TPR + tokl] = pad ? -1.f : v;                        // a negative variance marks padding
    }
  };
  if constexpr (NX == 1 && CW == 32 && kParts > 1) {
    // Quarters of 64 channels' lines: the sums of four lanes each, added as the wider workgroups' eight lanes are (the
    // statistics of a row do not depend on how its launch was split).
    float sm[2][NLD], sq[2][NLD];
    auto add_quarter = [&](const int i, const uint4 (&v)[NLD]) {   // i: which four pieces of a line
#pragma unroll
      for (int k = 0; k < NLD; ++k) {
        const uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        float s = 0.f, q = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s = dot2_ones<T>(w[e], s);
          q = dot2_self<T>(w[e], q);
        }
        sm[i & 1][k] = i < 2 ? s : sm[i & 1][k] + s;
        sq[i & 1][k] = i < 2 ? q : sq[i & 1][k] + q;
      }
    };
    if constexpr (kParts == 2) {
      if (part == 0) {
        add_quarter(0, xv);
        add_quarter(1, xo);
      } else {
        add_quarter(0, xo);
        add_quarter(1, xv);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kParts; ++i) {
        load_lines(gblk + i * CW, xo);
        add_quarter(i, xo);
      }
    }
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      const float m = (group_sum<PL>(sm[0][k]) + group_sum<PL>(sm[1][k])) * (1.0f / GC);
      const float v = fmaxf((group_sum<PL>(sq[0][k]) + group_sum<PL>(sq[1][k])) * (1.0f / GC) - m * m, 0.f);
      keep_moments(k, m, v);
    }
  } else if constexpr (NX == 1) {
    // sum and sum of squares by packed dot products; E[x^2] - mean^2 in fp32 resolves more than the inputs carry
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      const uint32_t w[4] = {xv[k].x, xv[k].y, xv[k].z, xv[k].w};
      float sm = 0.f, sq = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sm = dot2_ones<T>(w[i], sm);
        sq = dot2_self<T>(w[i], sq);
      }
      if constexpr (kParts == 2) {
        const uint32_t wo[4] = {xo[k].x, xo[k].y, xo[k].z, xo[k].w};
        float so = 0.f, qo = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          so = dot2_ones<T>(wo[i], so);
          qo = dot2_self<T>(wo[i], qo);
        }
        // lower half first in both workgroups
        sm = part == 0 ? sm + so : so + sm;
        sq = part == 0 ? sq + qo : qo + sq;
      }
      const float m = group_sum<PL>(sm) * (1.0f / GC);
      const float v = fmaxf(group_sum<PL>(sq) * (1.0f / GC) - m * m, 0.f);
      keep_moments(k, m, v);
    }
  } else {
    // fp32: the mean of a part first, then its squares around that mean; the later parts of a group (in the order of
    // their channels) by how far their means lie from the first part's
    static_assert(Gm::PPT == PL, "every lane of a line holds values");
    float gmean[NLD], gdist[NLD], gvar[NLD];
    auto add_part = [&](const int i, const uint4 (&v)[NLD]) {     // i: parts before this one
#pragma unroll
      for (int k = 0; k < NLD; ++k) {
        const float f[4] = {__uint_as_float(v[k].x), __uint_as_float(v[k].y), __uint_as_float(v[k].z), __uint_as_float(v[k].w)};
        const float m = group_sum<PL>((f[0] + f[1]) + (f[2] + f[3])) * (1.0f / CW);
        float q = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float d = f[e] - m;
          q = fmaf(d, d, q);
        }
        q = group_sum<PL>(q);
        if (i == 0) {
          gmean[k] = m;
          gdist[k] = 0.f;
          gvar[k] = q;
        } else {
          const float d = m - gmean[k];
          gdist[k] += d;
          gvar[k] += fmaf(d * d, (float)CW, q);
        }
      }
    };
    if constexpr (kParts == 1) {
      add_part(0, xv);
    } else if constexpr (kParts == 2) {
      if (part == 0) {
        add_part(0, xv);
        add_part(1, xo);
      } else {
        add_part(0, xo);
        add_part(1, xv);
      }
    } else {
#pragma unroll 1
      for (int i = 0; i < kParts; ++i) {       // (the workgroup's own part again: one order for all, and registers for one)
        load_lines(gblk + i * CW, xo);
        add_part(i, xo);
      }
    }
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      if constexpr (kParts == 1) {
        keep_moments(k, gmean[k], fmaxf(gvar[k] * (1.0f / GC), 0.f));       // (NaN is no padding: it counts, as in the other widths)
      } else {
        const float shift = gdist[k] * (1.0f / kParts);
        keep_moments(k, gmean[k] + shift, fmaxf(fmaf(-shift, shift, gvar[k] * (1.0f / GC)), 0.f));
      }
    }
  }
  __syncthreads();
  MEGA_FTR(1);

  // ---- running statistics: waves 0..3 scan 256 tokens each (4 per lane), the wave totals meet in LDS
  Moments pref[4], lane_exc = {0.f, 0.f, 0.f};
  if (wave < 4) {
    const float4 m4 = *(const float4*)(s_gm + wave * 256 + lane * 4);
    const float4 v4 = *(const float4*)(s_gv + wave * 256 + lane * 4);
    const float mm[4] = {m4.x, m4.y, m4.z, m4.w}, vv[4] = {v4.x, v4.y, v4.z, v4.w};
    // padding counts for nothing: weight 0 (the merges keep the other side's statistics)
    Moments st = {vv[0] >= 0.f ? 1.f : 0.f, mm[0], fmaxf(vv[0], 0.f)};
    pref[0] = st;
#pragma unroll
    for (int u = 1; u < 4; ++u) {
      st = merge<FINE>(st, Moments{vv[u] >= 0.f ? 1.f : 0.f, mm[u], fmaxf(vv[u], 0.f)});
      pref[u] = st;
    }
    const Moments inc = row_scan<FINE>(st);
    const Moments exc = dpp_m<0x111>(inc);
    Moments acc = {0.f, 0.f, 0.f}, rp = {0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const Moments t = {__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, inc.n), 16 * r + 15)),
                         __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, inc.mean), 16 * r + 15)),
                         __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, inc.var), 16 * r + 15))};
      if ((lane >> 4) == r) rp = acc;
      acc = merge<FINE>(acc, t);
    }
    lane_exc = merge<FINE>(rp, exc);
    if (lane == 0) {
      s_wt[wave * 4] = acc.n;
      s_wt[wave * 4 + 1] = acc.mean;
      s_wt[wave * 4 + 2] = acc.var;
    }
  }
  __syncthreads();
  if (wave < 4) {
    Moments wpre = {0.f, 0.f, 0.f}, tot = {0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w == wave) wpre = tot;
      tot = merge<FINE>(tot, Moments{s_wt[w * 4], s_wt[w * 4 + 1], s_wt[w * 4 + 2]});
    }
    if (wave == 0 && lane == 0 && !(A.lb.withhold_first && s == 0)) {
      put_rec(myrec, tagged((uint32_t)tot.n, tag));
      put_rec(myrec + 1, tagged(__float_as_uint(tot.mean), tag));
      put_rec(myrec + 2, tagged(__float_as_uint(tot.var), tag));
    }
    MEGA_FTR(2);
    // earlier blocks of this (row, group): lane i fetches block i's aggregate
    Moments accp = {0.f, 0.f, 0.f};
    if (s > 0) {
      const unsigned long long* rp = A.rec + (rrow * (A.S + 1) + (lane < s ? lane : s - 1)) * kRecW;
      unsigned long long w0, w1, w2;
      uint32_t spins = 0;
      for (;;) {
        w0 = get_rec(rp);
        w1 = get_rec(rp + 1);
        w2 = get_rec(rp + 2);
        const bool ok = (uint32_t)(w0 >> 32) == tag && (uint32_t)(w1 >> 32) == tag && (uint32_t)(w2 >> 32) == tag;
        if (__all(ok)) break;
        if (++spins > A.lb.spin_limit) {
          poison = true;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      for (int i = 0; i < s; ++i) {
        const Moments t = {(float)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)w0, i),
                           __builtin_bit_cast(float, __builtin_amdgcn_readlane((int)(uint32_t)w1, i)),
                           __builtin_bit_cast(float, __builtin_amdgcn_readlane((int)(uint32_t)w2, i))};
        accp = merge<FINE>(accp, t);
      }
    }
    MEGA_FTR(3);
    Moments carry = merge<FINE>(prior, accp);
    if (poison) {
      carry.mean = __builtin_nanf("");
      if (lane == 0) report_give_up(A.hdr, A.lb.status);
    }
    const Moments base = merge<FINE>(carry, merge<FINE>(wpre, lane_exc));
    Moments full = base;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      full = merge<FINE>(base, pref[u]);
      const float rstd = __builtin_amdgcn_rsqf(full.var + A.eps);
      s_gm[wave * 256 + lane * 4 + u] = full.mean;
      s_gv[wave * 256 + lane * 4 + u] = rstd;
      // training: the statistics the norm's backward pass reads (a padded token holds the carried ones)
      if (A.cummean && part == 0) {
        const int64_t tok = (int64_t)t0 + wave * 256 + lane * 4 + u;
        if (tok >= 0) {
          const int64_t o = ((int64_t)b * A.L + tok) * A.G + g;
          A.cummean[o] = full.mean;
          A.cumrstd[o] = rstd;
        }
      }
    }
    if (s == A.S - 1 && wave == 3 && lane == 63 && part == 0) {
      A.mean[brow] = full.mean;
      A.var[brow] = full.var;
      // tokens that count: whole numbers below 2^24, exact in the float sums
      if (g == 0) A.count[b] = poison ? (int64_t)-1 : A.prev_count[b] + (int64_t)(accp.n + tot.n);
    }
  }
  __syncthreads();

  // operand loaders of the moving-average phases (one register set: a channel's operands are requested as soon
  // as the previous channel's have been used, and travel under the rest of that channel's work)
  const uint32_t loff0 = (uint32_t)lane * 16;
  const uint32_t koff0 = (uint32_t)(((lane & 15) - 8 * (lane >> 4) + 24) * 16);
  constexpr int kSP = F16 ? kSlotP16 : kSlotP, kSC = F16 ? kSlotC16 : kSlotC;
  auto load_p = [&](const int c, uint4 (&P)[kNWP][2]) {
    const char* img = (const char*)A.image + (size_t)(cb + c) * kImgRowBytes;
    uint32_t loff = loff0;
    asm volatile("" : "+v"(loff));
#pragma unroll
    for (int w = 0; w < kNWP; ++w)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) P[w][mb] = img_slot(img, kSP + 2 * w + mb, loff);
  };
  auto load_kc = [&](const int c, uint4 (&K)[kNWK][2], uint4 (&C)[NC][2]) {
    const char* img = (const char*)A.image + (size_t)(cb + c) * kImgRowBytes;
    uint32_t loff = loff0;
    asm volatile("" : "+v"(loff));
    if constexpr (F16) {
#pragma unroll
      for (int w = 0; w < kNWK; ++w)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) K[w][mb] = img_slot(img, kSlotK16 + 2 * w + mb, loff);
    } else {
      // K from the slot that holds each distinct vector once: 7 lines per term leave the cache instead of 16
      uint32_t koff = koff0;
      asm volatile("" : "+v"(koff));
#pragma unroll
      for (int w = 0; w < kNWK; ++w)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) K[w][mb] = *(const uint4*)(img + ((kSlotKT + w) * 1024 + mb * 256) + koff);
    }
#pragma unroll
    for (int w = 0; w < NC; ++w)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) C[w][mb] = img_slot(img, kSC + 2 * w + mb, loff);
  };
  // the P operand of the wave's first channel travels under the normalisation
  uint4 Pa[kNWP][2];
  load_p(wave, Pa);

  // ---- normalise from registers and stage xn (as the layer sees it) transposed: channel rows of 16 segments x
  // 128 bytes, 16-byte chunk c of segment j at chunk c ^ (j >> 1) (the 16 lanes of a matrix-core operand load then
  // cover all banks); the lanes of tokens (2m, 2m+1) swap halves so that each writes dwords (even token | odd token
  // << 16) of four channels.  fp32: the two 16-bit terms of x are the halves, a plane each.
  {
    const int odd = tokl & 1;
    const uint32_t sel_lo = odd ? 0x01000504u : 0x05040100u;
    const uint32_t sel_hi = odd ? 0x03020706u : 0x07060302u;
    const int tl = tokl & ~1;
    char* wbase = tile + (NX == 1 ? row_base(piece * 8 + odd * 4) : odd * kPlane + row_base(piece * 4)) + (tl >> 6) * 128 +
                  ((tl & 7) >> 1) * 4;
    const int c8 = (tl & 63) >> 3;
    // weight + 1 = 1 and bias = 0 for every channel of the group (the module's initial values): the affine step
    // is skipped, one multiply-add per element less (a wave sees all channels, so the branch is uniform)
    bool plain = true;
#pragma unroll
    for (int i = 0; i < VPP; ++i) plain = plain && gam[i] == 1.f && bet[i] == 0.f;
    const bool ident = __all(plain);
    auto stage = [&](auto IDENT, auto MASKED, auto FRONT) {
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      const int tok = k * TPR + tokl;
      const float m = s_gm[tok], r = s_gv[tok];
      const float mr = m * r;
      const uint32_t w[4] = {xv[k].x, xv[k].y, xv[k].z, xv[k].w};
      uint32_t o[4], h[4];               // what leaves as xn, and the halves the moving average takes
      const bool pad = decltype(MASKED)::value && ((mbits >> k) & 1u);      // padding leaves as zeros, whatever x holds there
      if constexpr (NX == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float2 v = unpack16<F16>(w[i]);
          const float lo = fmaf(v.x, r, -mr), hi = fmaf(v.y, r, -mr);
          o[i] = decltype(IDENT)::value ? pack16<F16>(lo, hi)
                                        : pack16<F16>(fmaf(lo, gam[2 * i], bet[2 * i]), fmaf(hi, gam[2 * i + 1], bet[2 * i + 1]));
          o[i] = pad ? 0u : o[i];
          h[i] = o[i];
        }
      } else {
        float f[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f[i] = fmaf(__uint_as_float(w[i]), r, -mr);
          if (!decltype(IDENT)::value) f[i] = fmaf(f[i], gam[i], bet[i]);
          f[i] = pad ? 0.f : f[i];
          o[i] = __float_as_uint(f[i]);
          lo[i] = f[i] - (float)(_Float16)f[i];
        }
        h[0] = pack16<true>(f[0], f[1]);
        h[1] = pack16<true>(f[2], f[3]);
        h[2] = pack16<true>(lo[0], lo[1]);
        h[3] = pack16<true>(lo[2], lo[3]);
      }
      if (act && (!decltype(FRONT)::value || tok >= A.pad))                // virtual tokens have no place in xn
        store_stream((uint4*)(gxn + xblk + (int64_t)k * TPR * A.D + toff), make_uint4(o[0], o[1], o[2], o[3]));
      const uint32_t s0 = odd ? h[0] : h[2], s1 = odd ? h[1] : h[3];
      const uint32_t r0 = dpp_u<0x128>(s0), r1 = dpp_u<0x128>(s1);       // row_ror:8 = the partner token's lane
      const uint32_t m0 = odd ? h[2] : h[0], m1 = odd ? h[3] : h[1];
      if (act) {
        char* wp = wbase + k * (TPR * 2) + ((c8 ^ ((k * TPR + tl) >> 7)) << 4);
        *(uint32_t*)(wp) = __builtin_amdgcn_perm(r0, m0, sel_lo);
        *(uint32_t*)(wp + kFRow) = __builtin_amdgcn_perm(r0, m0, sel_hi);
        *(uint32_t*)(wp + 2 * kFRow) = __builtin_amdgcn_perm(r1, m1, sel_lo);
        *(uint32_t*)(wp + 3 * kFRow) = __builtin_amdgcn_perm(r1, m1, sel_hi);
      }
    }
    };
    if (front) {
      if (ident) {
        stage(std::true_type{}, std::true_type{}, std::true_type{});
      } else {
        stage(std::false_type{}, std::true_type{}, std::true_type{});
      }
    } else if (A.mask) {
      if (ident) {
        stage(std::true_type{}, std::true_type{}, std::false_type{});
      } else {
        stage(std::false_type{}, std::true_type{}, std::false_type{});
      }
    } else if (ident) {
      stage(std::true_type{}, std::false_type{}, std::false_type{});
    } else {
      stage(std::false_type{}, std::false_type{}, std::false_type{});
    }
  }
  __syncthreads();

  MEGA_FTR(4);
  // ---- moving average.  MFMA lane layout: column j = lane & 15 is segment j, r = lane >> 4 holds the
  // states (2r, 2r+1, 8+2r, 9+2r) of the 32-row state products.
  const int j = lane & 15, r = lane >> 4;
  const int nn[4] = {2 * r, 2 * r + 1, 8 + 2 * r, 9 + 2 * r};
  const bool last_block = s == A.S - 1;
  const int nterms = s + (A.h_in ? 1 : 0);
  const uint32_t roff0 = (uint32_t)r * 16;
  // how far the channels' slowest poles reach (figures of the operand image, uniform per wave and channel)
  int nsteps[CPW], nlook[CPW];
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    const uint2 rw = s_reach[wave + kFW * i];
    nsteps[i] = __builtin_amdgcn_readfirstlane((int)rw.x);
    nlook[i] = __builtin_amdgcn_readfirstlane((int)rw.y);
  }

  // the wave's own row leaves as whole lines ([B, D, L] rows)
  auto store_row = [&](const int c) {
    // LDS operations of one wave are performed in order: the lanes' writes above are visible to the
    // reads below without waiting for anything else (a release fence would also wait for the wave's
    // outstanding global stores)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const char* rb = tile + row_base(c);
    T* yr = gy + (int64_t)b * A.syb + (int64_t)(cb + c) * A.syd + t0;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int q = k * 64 + lane;                 // 16-byte chunk of the row: segment q >> 3, chunk q & 7
      const char* at = rb + (q >> 3) * 128 + (((q & 7) ^ (q >> 4)) << 4);
      const uint4 v = *(const uint4*)at;
      // (a front block: the row begins inside it, at a multiple of 8)
      if constexpr (NX == 1) {
        if (q * 8 >= -t0) store_stream((uint4*)(yr + q * 8), v);
      } else {
        const uint4 u = *(const uint4*)(at + kPlane);          // the low halves of the same eight values
        if (q * 8 >= -t0) {
          store_stream((uint4*)(yr + q * 8),
                       make_uint4(__builtin_amdgcn_perm(v.x, u.x, 0x05040100u), __builtin_amdgcn_perm(v.x, u.x, 0x07060302u),
                                  __builtin_amdgcn_perm(v.y, u.y, 0x05040100u), __builtin_amdgcn_perm(v.y, u.y, 0x07060302u)));
          store_stream((uint4*)(yr + q * 8 + 4),
                       make_uint4(__builtin_amdgcn_perm(v.z, u.z, 0x05040100u), __builtin_amdgcn_perm(v.z, u.z, 0x07060302u),
                                  __builtin_amdgcn_perm(v.w, u.w, 0x05040100u), __builtin_amdgcn_perm(v.w, u.w, 0x07060302u)));
        }
      }
    }
  };

  // End states of channel c's 16 segments from a zero start (P products; F = the state after a segment's first
  // tile), scanned across the row by doubling: E becomes the state after segment j with the block started from
  // zero.  A step over d segments is skipped (uniform branch) when |q|^(64 d) < 2^-24 for every state of the
  // channel: what it would add is below fp32 resolution.
  auto segment_scan = [&](const int c, const int steps, const uint4 (&P)[kNWP][2], const char* row, const float (&Qr)[4], const float (&Qi)[4],
                          float (&Er)[4], float (&Ei)[4], float (&Fr)[4], float (&Fi)[4], const uint32_t roff) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const char* at = row + (((4 * t + r) ^ (j >> 1)) << 4);
      const uint4 X = *(const uint4*)at;
      f32x4 S0 = {0.f, 0.f, 0.f, 0.f}, S1 = {0.f, 0.f, 0.f, 0.f};
      if constexpr (NX > 1) {                     // (the small terms of a sum first)
        const uint4 Xl = *(const uint4*)(at + kPlane);
        S0 = mma<F16>(P[0][0], Xl, S0);
        S1 = mma<F16>(P[0][1], Xl, S1);
      }
#pragma unroll
      for (int w = 0; w < kNWP; ++w) {
        const int v = F16 ? kNWP - 1 - w : w;
        S0 = mma<F16>(P[v][0], X, S0);
        S1 = mma<F16>(P[v][1], X, S1);
      }
      const float sr[4] = {S0[0], S0[2], S1[0], S1[2]};
      const float si[4] = {S0[1], S0[3], S1[1], S1[3]};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (t == 0) {
          Fr[u] = sr[u];
          Fi[u] = si[u];
        } else {
          Er[u] = fmaf(Qr[u], Fr[u], fmaf(-Qi[u], Fi[u], sr[u]));
          Ei[u] = fmaf(Qr[u], Fi[u], fmaf(Qi[u], Fr[u], si[u]));
        }
      }
    }
    if (steps > 0) {
      float Rr[4], Ri[4], R2r[4], R2i[4];
      lds_cmp(s_tab, kCmpRS * CW + c, roff, Rr, Ri);
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
  };

  // ---- phase A, what the later blocks wait for: the block's end state from a zero start (lane 15 of every row
  // after the scan), parked in LDS and published
  MEGA_FTR(5);
  // it goes before the other waves' phase B
  __builtin_amdgcn_s_setprio(2);
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    const int c = wave + kFW * i;
    uint32_t roff = roff0;
    asm volatile("" : "+v"(roff));
    float Qr[4], Qi[4];
    lds_cmp(s_tab, kCmpQ32 * CW + c, roff, Qr, Qi);
    const char* row = tile + row_base(c) + j * 128;
    float Er[4], Ei[4], Fr[4], Fi[4];
    segment_scan(c, nsteps[i], Pa, row, Qr, Qi, Er, Ei, Fr, Fi, roff);
    if (j == 15) {
      *(float4*)(s_end + (c * kNS + 2 * r) * 2) = make_float4(Er[0], Ei[0], Er[1], Ei[1]);
      *(float4*)(s_end + (c * kNS + 8 + 2 * r) * 2) = make_float4(Er[2], Ei[2], Er[3], Ei[3]);
    }
    // the next channel's P operand (after the last channel: the first one's again, for phase B)
    __builtin_amdgcn_sched_barrier(0);
    load_p(i + 1 < CPW ? wave + kFW * (i + 1) : wave, Pa);
    __builtin_amdgcn_sched_barrier(0);
    MEGA_FTR(6 + i);
  }
  if (!last_block && !(A.lb.withhold_first && s == 0)) {
    // the wave's channels x 16 states x (re, im): two words per lane (four channels: every lane)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    if (CPW == 4 || (lane >> 4) < CPW) {
      const int cp = wave + kFW * (lane >> 4);
      const float2 v = *(const float2*)(s_end + (cp * kNS + (lane & 15)) * 2);
      unsigned long long* e = myrec + 4 + ((size_t)cp * kNS + (lane & 15)) * 2;
      put_rec(e, tagged(__float_as_uint(v.x), tag));
      put_rec(e + 1, tagged(__float_as_uint(v.y), tag));
    }
  }
  __builtin_amdgcn_s_setprio(0);

  // the operands of phase B's first channel travel under the wait for the earlier blocks
  uint4 Ka[kNWK][2], Ca[NC][2];
  load_kc(wave, Ka, Ca);
  float Jr[4] = {0.f, 0.f, 0.f, 0.f}, Ji[4] = {0.f, 0.f, 0.f, 0.f};
  auto load_j = [&](const int c) {
    const char* img = (const char*)A.image + (size_t)(cb + c) * kImgRowBytes;
    uint32_t loff = loff0;
    asm volatile("" : "+v"(loff));
    load_c4(img, kSlotRJ, loff, Jr, Ji);             // (q^64)^j
  };
  load_j(wave);

  // ---- start state of the block: h_start = sum_{d >= 0} (q^1024)^d E_{s-1-d}, E_{-1} being the caller's carried
  // state (slot S of the row's records).  Lane (j, r) works for channel wave + 16 (j >> 2) (idle when the wave has no
  // such channel) and takes the terms d = (j & 3) + 4 k; the four lanes of a quad add up.
  const int ci = j >> 2;
  const bool cown = CPW == 4 || ci < CPW;
  const int cl = wave + kFW * (cown ? ci : 0);
  float Cr[4] = {0.f, 0.f, 0.f, 0.f}, Ci[4] = {0.f, 0.f, 0.f, 0.f};
  if (nterms > 0) {
    const int chl = cb + cl;
    int look = 0;                                  // blocks back that still reach this lane's channel
#pragma unroll
    for (int i = 0; i < CPW; ++i) look = ci == i ? nlook[i] : look;
    const char* wimg = (const char*)A.image + (size_t)chl * kImgRowBytes;
    int maxlook = 0;
#pragma unroll
    for (int i = 0; i < CPW; ++i) maxlook = nlook[i] > maxlook ? nlook[i] : maxlook;
    const int nrounds = nterms < maxlook ? nterms : maxlook;
    for (int d0 = 0; d0 < nrounds; d0 += 4) {
      const int d = d0 + (j & 3);
      const bool have = d < nterms && d < look;
      const int slot = have ? (d < s ? s - 1 - d : A.S) : 0;
      const unsigned long long* e = A.rec + (rrow * (A.S + 1) + slot) * kRecW + 4 + (size_t)cl * kNS * 2 + 4 * r;
      float Wr[4], Wi[4];
      load_c4(wimg, kSlotRWJ, (uint32_t)(((r << 4) | (have ? d : 0)) * 16), Wr, Wi);      // (q^1024)^d
      unsigned long long w[8];
      uint32_t spins = 0;
      for (;;) {
        bool ok = true;
#pragma unroll
        for (int u = 0; u < 4; ++u) {              // states (2r, 2r+1) and (8+2r, 9+2r): two runs of four words
          w[u] = have ? get_rec(e + u) : tagged(0u, tag);
          w[4 + u] = have ? get_rec(e + 16 + u) : tagged(0u, tag);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) ok &= (uint32_t)(w[u] >> 32) == tag;
        if (__all(ok)) break;
        if (++spins > A.lb.spin_limit) {
          poison = true;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float er = __uint_as_float((uint32_t)w[2 * u]), ei = __uint_as_float((uint32_t)w[2 * u + 1]);
        Cr[u] = fmaf(Wr[u], er, fmaf(-Wi[u], ei, Cr[u]));
        Ci[u] = fmaf(Wr[u], ei, fmaf(Wi[u], er, Ci[u]));
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      Cr[u] = group_sum<4>(Cr[u]);
      Ci[u] = group_sum<4>(Ci[u]);
    }
    if (poison) {
      Cr[0] = __builtin_nanf("");
      if (lane == 0) report_give_up(A.hdr, A.lb.status);
    }
  }
  // h_start (zero when nothing comes in) is parked over the wave's own end states, which have left; the last block
  // first returns the state after its last token: end state from a zero start + (q^1024) h_start
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  if (last_block && A.h_out && (j & 3) == 0 && cown) {
    const int ch = cb + cl;
    float Rr[4], Ri[4];
    load_cmp((const char*)A.image + (size_t)ch * kImgRowBytes, kCmpRW, roff0, Rr, Ri);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (nn[u] < A.N) {
        const float er = s_end[(cl * kNS + nn[u]) * 2], ei = s_end[(cl * kNS + nn[u]) * 2 + 1];
        const size_t o = (((size_t)b * A.D + ch) * A.N + nn[u]) * 2;
        A.h_out[o] = fmaf(Rr[u], Cr[u], fmaf(-Ri[u], Ci[u], er));
        A.h_out[o + 1] = fmaf(Rr[u], Ci[u], fmaf(Ri[u], Cr[u], ei));
      }
    }
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  if ((j & 3) == 0 && cown) {
    *(float4*)(s_end + (cl * kNS + 2 * r) * 2) = make_float4(Cr[0], Ci[0], Cr[1], Ci[1]);
    *(float4*)(s_end + (cl * kNS + 8 + 2 * r) * 2) = make_float4(Cr[2], Ci[2], Cr[3], Ci[3]);
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  MEGA_FTR(10);

  // ---- phase B per channel: the segment scan again (cheaper than keeping four channels' scans in registers across
  // the wait), start state of segment j = what segment j - 1 left + (q^64)^j h_start, then
  // y_tile = K x_tile + C h (h: the state at the tile's first token, carried into the product as two bf16 terms where
  // one would show; at a segment's second tile h = q^32 h + F), bf16,
  // back into LDS over x, and out as whole rows.
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    const int c = wave + kFW * i;
    // One bf16 term for the states leaves an error of 2^-9 of sum |gamma q h| at the first tokens of every tile.  It
    // shows where the states dwarf y (slow poles: |q|^128 >= 2^-24 for some state of the channel), in layers of few
    // states, whose rounding errors do not average out in the sum over the states, and in real-valued layers, whose
    // input weights alternate in sign along the states so that the states cancel by construction: those take a
    // second term (hi + lo), and fp16 operands always do.  MEGA_FUSED_TWO_TERMS=1 gives every channel the second term (+ 0.7 us at the headline
    // shape).
    const bool two_terms = F16 || MEGA_FUSED_TWO_TERMS || nsteps[i] >= 2 || A.N <= 8 || !A.is_complex;
    uint32_t roff = roff0;
    asm volatile("" : "+v"(roff));
    char* row = tile + row_base(c) + j * 128;
    float hr[4], hi[4], Fr[4], Fi[4];
    {
      float Qr[4], Qi[4];
      lds_cmp(s_tab, kCmpQ32 * CW + c, roff, Qr, Qi);
      segment_scan(c, nsteps[i], Pa, row, Qr, Qi, hr, hi, Fr, Fi, roff);
    }
    MEGA_FTR2(0);
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < CPW) load_p(wave + kFW * (i + 1), Pa);
    __builtin_amdgcn_sched_barrier(0);
    {
      const float4 b0 = *(const float4*)(s_end + (c * kNS + 2 * r) * 2);
      const float4 b1 = *(const float4*)(s_end + (c * kNS + 8 + 2 * r) * 2);
      const float br[4] = {b0.x, b0.z, b1.x, b1.z}, bi[4] = {b0.y, b0.w, b1.y, b1.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float sr = dpp_f<0x111>(hr[u]), si = dpp_f<0x111>(hi[u]);
        hr[u] = fmaf(Jr[u], br[u], fmaf(-Ji[u], bi[u], sr));
        hi[u] = fmaf(Jr[u], bi[u], fmaf(Ji[u], br[u], si));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < CPW) load_j(wave + kFW * (i + 1));
    __builtin_amdgcn_sched_barrier(0);
    MEGA_FTR2(1);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      asm volatile("" ::: "memory");              // x again from LDS: cheaper than eight registers across the scan
      const char* xat = row + (((4 * t + r) ^ (j >> 1)) << 4);
      const uint4 X = *(const uint4*)xat;
      f32x4 Y0 = {0.f, 0.f, 0.f, 0.f}, Y1 = {0.f, 0.f, 0.f, 0.f};
      uint32_t hp[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) hp[u] = pack16<F16>(hr[u], hi[u]);
      const uint4 Hop = make_uint4(hp[0], hp[1], hp[2], hp[3]);
      auto low_states = [&]() {
        uint32_t hl[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float2 v = unpack16<F16>(hp[u]);
          hl[u] = pack16<F16>(hr[u] - v.x, hi[u] - v.y);
        }
        const uint4 Hlo = make_uint4(hl[0], hl[1], hl[2], hl[3]);
#pragma unroll
        for (int w = 0; w < kNWC; ++w) {
          Y0 = mma<F16>(Ca[w][0], Hlo, Y0);
          Y1 = mma<F16>(Ca[w][1], Hlo, Y1);
        }
      };
      if constexpr (F16) {                        // the small terms of the sum first
        low_states();
        Y0 = mma<F16>(Ca[NC - 1][0], Hop, Y0);
        Y1 = mma<F16>(Ca[NC - 1][1], Hop, Y1);
        if constexpr (NX > 1) {
          const uint4 Xl = *(const uint4*)(xat + kPlane);
          Y0 = mma<F16>(Ka[0][0], Xl, Y0);
          Y1 = mma<F16>(Ka[0][1], Xl, Y1);
        }
#pragma unroll
        for (int w = kNWK - 1; w >= 0; --w) {
          Y0 = mma<F16>(Ka[w][0], X, Y0);
          Y1 = mma<F16>(Ka[w][1], X, Y1);
        }
        Y0 = mma<F16>(Ca[0][0], Hop, Y0);
        Y1 = mma<F16>(Ca[0][1], Hop, Y1);
      } else {
#pragma unroll
        for (int w = 0; w < kNWK; ++w) {
          Y0 = mma<F16>(Ka[w][0], X, Y0);
          Y1 = mma<F16>(Ka[w][1], X, Y1);
        }
#pragma unroll
        for (int w = 0; w < NC; ++w) {
          Y0 = mma<F16>(Ca[w][0], Hop, Y0);
          Y1 = mma<F16>(Ca[w][1], Hop, Y1);
        }
        if (two_terms) low_states();
      }
      if (t == 0) {
        float Qr[4], Qi[4];
        lds_cmp(s_tab, kCmpQ32 * CW + c, roff, Qr, Qi);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float nr = fmaf(Qr[u], hr[u], fmaf(-Qi[u], hi[u], Fr[u]));
          hi[u] = fmaf(Qr[u], hi[u], fmaf(Qi[u], hr[u], Fi[u]));
          hr[u] = nr;
        }
      }
      // y over x (fp32: the upper and lower halves of its words, a plane each): tokens 32 t + 4 r + {0..3} and
      // 32 t + 16 + 4 r + {0..3} of segment j
      char* y0 = row + (((4 * t + (r >> 1)) ^ (j >> 1)) << 4) + (r & 1) * 8;
      char* y1 = row + (((4 * t + 2 + (r >> 1)) ^ (j >> 1)) << 4) + (r & 1) * 8;
      if constexpr (NX == 1) {
        *(uint2*)y0 = make_uint2(pack16<F16>(Y0[0], Y0[1]), pack16<F16>(Y0[2], Y0[3]));
        *(uint2*)y1 = make_uint2(pack16<F16>(Y1[0], Y1[1]), pack16<F16>(Y1[2], Y1[3]));
      } else {
        auto halves = [](const float a, const float c, const uint32_t sel) {
          return __builtin_amdgcn_perm(__float_as_uint(c), __float_as_uint(a), sel);
        };
        *(uint2*)y0 = make_uint2(halves(Y0[0], Y0[1], 0x07060302u), halves(Y0[2], Y0[3], 0x07060302u));
        *(uint2*)y1 = make_uint2(halves(Y1[0], Y1[1], 0x07060302u), halves(Y1[2], Y1[3], 0x07060302u));
        *(uint2*)(y0 + kPlane) = make_uint2(halves(Y0[0], Y0[1], 0x05040100u), halves(Y0[2], Y0[3], 0x05040100u));
        *(uint2*)(y1 + kPlane) = make_uint2(halves(Y1[0], Y1[1], 0x05040100u), halves(Y1[2], Y1[3], 0x05040100u));
      }
      MEGA_FTR2(2 + t);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < CPW) load_kc(wave + kFW * (i + 1), Ka, Ca);
    __builtin_amdgcn_sched_barrier(0);
    MEGA_FTR2(4);
    if (LOUT == 0) store_row(c);
    __builtin_amdgcn_sched_barrier(0);
    MEGA_FTR(11 + i);
  }
  if (LOUT == 1) {
    // [B, L, D]: the inverse of the staging step, whole lines of 64 channels per token
    __syncthreads();
    const int odd = tokl & 1;
    const uint32_t sel_keep = odd ? 0x07060302u : 0x05040100u;
    const uint32_t sel_give = odd ? 0x05040100u : 0x07060302u;
    const int tl = tokl & ~1;
    const char* rbase = tile + (NX == 1 ? row_base(piece * 8 + odd * 4) : odd * kPlane + row_base(piece * 4)) +
                        (tl >> 6) * 128 + ((tl & 7) >> 1) * 4;
    const int c8 = (tl & 63) >> 3;
    T* yb = gy + (int64_t)b * A.syb + (int64_t)(cb + piece * VPP) * A.syd;
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      const int tok = k * TPR + tokl;
      const char* rp = rbase + k * (TPR * 2) + ((c8 ^ ((k * TPR + tl) >> 7)) << 4);
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = *(const uint32_t*)(rp + e * kFRow);
      const uint32_t keep0 = __builtin_amdgcn_perm(w[1], w[0], sel_keep);
      const uint32_t keep1 = __builtin_amdgcn_perm(w[3], w[2], sel_keep);
      const uint32_t got0 = dpp_u<0x128>(__builtin_amdgcn_perm(w[1], w[0], sel_give));
      const uint32_t got1 = dpp_u<0x128>(__builtin_amdgcn_perm(w[3], w[2], sel_give));
      // the even token's lane kept (and got the partner's view of) the first half: channels 0..3 of eight, or the
      // upper halves of four words
      const uint32_t f0 = odd ? got0 : keep0, f1 = odd ? got1 : keep1, l0 = odd ? keep0 : got0, l1 = odd ? keep1 : got1;
      uint4 o;
      if constexpr (NX == 1) {
        o = make_uint4(f0, f1, l0, l1);
      } else {
        o.x = __builtin_amdgcn_perm(f0, l0, 0x05040100u);
        o.y = __builtin_amdgcn_perm(f0, l0, 0x07060302u);
        o.z = __builtin_amdgcn_perm(f1, l1, 0x05040100u);
        o.w = __builtin_amdgcn_perm(f1, l1, 0x07060302u);
      }
      if (act && t0 + tok >= 0) store_stream((uint4*)(yb + (int64_t)(t0 + tok) * A.syl), o);
    }
  }

  MEGA_FTR_END();
  // ---- retire: the last workgroup to finish opens the next epoch
  if (tid == 0) {
    const uint32_t total = gridDim.x;
    const uint32_t k = blockIdx.x & 31u;
    const uint32_t quota = (total - k + 31u) / 32u;
    if (atomicAdd(&A.hdr->done1[k], 1u) == quota - 1u) {
      publish_u32(&A.hdr->done1[k], 0u);
      const uint32_t classes = total < 32u ? total : 32u;
      if (atomicAdd(&A.hdr->done2, 1u) == classes - 1u) {
        publish_u32(&A.hdr->done2, 0u);
        publish_u32(&A.hdr->epoch, tag == 0xffffffffu ? 0u : tag);
      }
    }
  }
}

// records of B * D channels in workgroups of cw
size_t fused_ws_bytes(int64_t B, int64_t D, int64_t S, int cw) {
  return align_up(sizeof(TsnHeader), 256) + align_up((size_t)(B * ceil_div(D, cw)) * (S + 1) * (4 + cw * kNS * 2) * 8, 256);
}

// Channels of a workgroup for norm groups of gc channels, 0: no instance.  16-bit rows of a block fill the LDS with 64
// channels, fp32 rows (two planes) with 32; a group that does not fit is shared by equal parts of a multiple of 16.  Only the widths
// below have instances, each measured against the two operators; others (16, 24, 80, 112, 160 and more) run as two operators.
// The two operators one after the other (norm, transposition, rows kernels, transposition) take, against one launch
// here, with y in x's layout: fp16 3 x 1501 x 768 in 48s 79 us, 26 here; fp16 4 x 4096 x 1024 in 64s 101 us, 34; fp16
// 2 x 8192 x 2048 in 128s 249 us, 76; fp32 4 x 4096 x 1024 138 us, 53 (3.8 TB/s); fp32 2 x 8192 x 2048 in four parts
// 364 us, 134; fp32 1 x 300 x 512 in 32s 51 us, 24 (the host's call).  bf16 in the widths beside 64 and 128 (norm, then
// the streaming kernel): 4 x 4096 x 768 in 48s 54 us, 40; 8 x 2048 x 512 in 32s 32 us, 24; 2 x 1333 x 1536 37 us, 25.
// 16-bit groups of 64 and 128 channels go to workgroups of 32 where even those are no more than the compute units: the
// launch lasts one workgroup's chain, which half the channels shorten (the moments' lines are read by every workgroup of
// the group): bf16 2 x 2991 x 1024 32.1 us of device time with 64, 28.1 with 32; 4 x 2048 x 1024 30.0, 26.1; the bf16
// values are the same bit for bit, of fp16 ones about two in a million differ by a unit in the last place (whether the
// compiler rounds fma and conversion once or twice differs from instance to instance).
int fused_channels(int dtype, int64_t gc, int64_t rows_blocks_channels) {
  const bool wide = dtype == MEGA_F32;
  if (!wide && (gc == 64 || gc == 128) && rows_blocks_channels <= (int64_t)32 * device_cu_count()) return 32;
  switch (gc) {
    case 32: return 32;
    case 48: return wide ? 16 : 48;
    case 64: return wide ? 32 : 64;
    case 96: return wide ? 32 : 48;
    case 128: return wide ? 32 : 64;
    default: return 0;
  }
}

template <typename T, int CW, int PARTS, int LOUT, bool STAG>
void fused_launch(const FusedArgs& A, dim3 grid, hipStream_t s) {
  static uint64_t attr_seen = 0;
  const auto kern = norm_ema_fused_kernel<T, CW, PARTS, LOUT, STAG>;
  constexpr size_t smem = Geo<T, CW, PARTS>::Smem;
  raise_lds_limit(&attr_seen, (int)smem, kern);
  hipLaunchKernelGGL(kern, grid, dim3(kFT), smem, s, A);
}

template <typename T, int CW, int PARTS>
void fused_launch_layout(const FusedArgs& A, int lout, dim3 grid, hipStream_t s) {
  if constexpr (__is_same(T, bf16_t) && CW == 64) {
    if (A.stagger > 0)
      return lout ? fused_launch<T, CW, PARTS, 1, true>(A, grid, s) : fused_launch<T, CW, PARTS, 0, true>(A, grid, s);
  }
  return lout ? fused_launch<T, CW, PARTS, 1, false>(A, grid, s) : fused_launch<T, CW, PARTS, 0, false>(A, grid, s);
}

template <typename T>
void fused_launch_width(const FusedArgs& A, int gc, int cw, int lout, dim3 grid, hipStream_t s) {
  if constexpr (sizeof(T) == 4) {
    switch (gc) {
      case 32: return fused_launch_layout<T, 32, 1>(A, lout, grid, s);
      case 48: return fused_launch_layout<T, 16, 3>(A, lout, grid, s);
      case 64: return fused_launch_layout<T, 32, 2>(A, lout, grid, s);
      case 96: return fused_launch_layout<T, 32, 3>(A, lout, grid, s);
      default: return fused_launch_layout<T, 32, 4>(A, lout, grid, s);
    }
  } else {
    switch (gc) {
      case 32: return fused_launch_layout<T, 32, 1>(A, lout, grid, s);
      case 48: return fused_launch_layout<T, 48, 1>(A, lout, grid, s);
      case 64:
        return cw == 32 ? fused_launch_layout<T, 32, 2>(A, lout, grid, s) : fused_launch_layout<T, 64, 1>(A, lout, grid, s);
      case 96: return fused_launch_layout<T, 48, 2>(A, lout, grid, s);
      default:
        return cw == 32 ? fused_launch_layout<T, 32, 4>(A, lout, grid, s) : fused_launch_layout<T, 64, 2>(A, lout, grid, s);
    }
  }
}

// state: 1: a state comes in, 2: one is handed on (bits).
// No call is less accurate here than as two operators.  fp32 / fp16 rows of at least 64 tokens go through the rows kernels
// there, whose operands are the same two fp16 terms (errors of y 1.6e-7 here, 1.9e-7 there, fp32, 2 x 700 x 512); shorter
// ones, and those that hand a state on behind a partial block, through the fp32 recurrence of ema_scan.hip: 1.3e-7 here
// and 0.8e-7 there at 2 x 40 x 256, and a channel whose norm weight is 1e-3 of the others' 7e-5 and 4e-7.  bf16 in the
// widths beside 64 and 128 likewise below 256 tokens (errors of y 1.9e-3 and 1.66e-3, 2 x 200; of the state 2.4e-6 and
// 1e-7, 2 x 40), and the streaming kernel's states behind a partial block are closer than the ones here (1.96e-6, 2.4e-6).
bool fused_sizes(int dtype, int64_t B, int64_t L, int64_t D, int64_t G, int64_t N, int state, bool rows) {
  if (G <= 0 || D <= 0 || D % G || N > kNS || N <= 0 || L <= 0) return false;
  const int64_t gc = D / G;
  const int cw = fused_channels(dtype, gc, B * D * ceil_div(L, kFSeg));
  if (cw == 0 || ceil_div(L, kFSeg) + (state & 1) > kFMaxBlocks) return false;
  const bool bf16_lines = dtype == MEGA_BF16 && (gc == 64 || gc == 128);
  if (!bf16_lines && (L < (dtype == MEGA_BF16 ? 256 : 64) || (state != 0 && L % kFSeg != 0))) return false;
  // a ragged first block (the block grid is aligned to the end of the row): no carried state in (it would have to
  // enter in the middle of a block), and rows in time must begin at a multiple of 8 inside it
  if (L % kFSeg != 0 && ((state & 1) || (rows && L % 8 != 0))) return false;
  return B * (D / cw) * ceil_div(L, kFSeg) < (int64_t)1 << 31;
}

bool fused_covers(int dtype, int64_t B, int64_t L, int64_t D, int64_t G, int64_t N, const void* x, const void* xn,
                  const void* y, int64_t syb, int64_t syd, int64_t syl, const float* h_in, const float* h_out) {
  if (!fused_sizes(dtype, B, L, D, G, N, (h_in ? 1 : 0) | (h_out ? 2 : 0), syl == 1)) return false;
  if (((uintptr_t)x % 16) || ((uintptr_t)xn % 16) || ((uintptr_t)y % 16)) return false;
  const bool rows = syl == 1 && syd % 8 == 0 && syb % 8 == 0;
  const bool lines = syd == 1 && syl % 8 == 0 && syb % 8 == 0;
  return rows || lines;
}

}  // namespace
}  // namespace mega

using namespace mega;

// workspace (zero once, then owned by these calls): launch header + the records of whichever route a shape takes
extern "C" size_t mega_norm_ema_fwd_workspace_bytes(int64_t B, int64_t L, int64_t D, int64_t G, int64_t N) {
  (void)N;
  if (B <= 0 || L <= 0 || D <= 0 || G <= 0) return 256;
  const size_t fused = fused_ws_bytes(B, D, ceil_div(L, kFSeg), 16);      // (the narrowest workgroups: the most records)
  const size_t tsn = mega_timestep_norm_workspace_bytes(MEGA_BF16, B, L, D, G);
  return fused > tsn ? fused : tsn;
}

// 1: a call of these sizes (dense operands on 16 bytes) is one launch of the one-kernel route, for any activation type
extern "C" int mega_norm_ema_fwd_one_kernel(int dtype, int64_t B, int64_t L, int64_t D, int64_t G, int64_t N, int carried,
                                            int rows_out) {
  return fused_sizes(dtype, B, L, D, G, N, carried, rows_out != 0) && mega_ema_image_bytes(D, N, 0) > 0 ? 1 : 0;
}

// scratch (no initialisation, contents never survive a call): the moving average's own workspace when the two
// operators run one after the other, or room for kernel generation when no image is passed
extern "C" size_t mega_norm_ema_fwd_scratch_bytes(int64_t B, int64_t L, int64_t D, int64_t G, int64_t N) {
  (void)G;
  if (B <= 0 || L <= 0 || D <= 0 || N <= 0) return 256;
  const size_t ema = mega_ema_fwd_workspace_bytes(B, D, N, L, 0, 0);
  const size_t img = mega_ema_image_bytes(D, N, 0);
  return align_up(ema > img ? ema : img, 256);
}

extern "C" int mega_norm_ema_fwd_train(const void* x, void* xn, void* y, int dtype, int64_t syb, int64_t syd,
                                       int64_t syl, const int64_t* prev_count, const float* prev_mean,
                                       const float* prev_var, const float* norm_gamma, const float* norm_beta,
                                       const uint8_t* mask, double eps, int64_t* count, float* mean, float* var,
                                       float* cummean, float* cumrstd, const float* p, const float* q,
                                       const float* gamma, int is_complex, const float* omega, const float* h_in,
                                       float* h_out, int64_t B, int64_t L, int64_t D, int64_t G, int64_t N,
                                       const void* image, void* workspace, size_t workspace_bytes, void* scratch,
                                       size_t scratch_bytes, void* stream) {
  if (const int rc = lookback_pending("norm_ema_fwd")) return rc;
  MEGA_REQUIRE((cummean == nullptr) == (cumrstd == nullptr), MEGA_ERR_ARG,
               "norm_ema_fwd: cummean and cumrstd go together");
  MEGA_REQUIRE(dtype == MEGA_F32 || dtype == MEGA_BF16 || dtype == MEGA_F16, MEGA_ERR_ARG,
               "norm_ema_fwd: unknown dtype %d", dtype);
  MEGA_REQUIRE(B >= 0 && L >= 0 && D > 0 && G > 0 && N > 0 && D % G == 0, MEGA_ERR_ARG,
               "norm_ema_fwd: bad shape B=%ld L=%ld D=%ld G=%ld N=%ld", (long)B, (long)L, (long)D, (long)G, (long)N);
  if (B == 0) return MEGA_OK;
  const size_t need = mega_norm_ema_fwd_workspace_bytes(B, L > 0 ? L : 1, D, G, N);
  MEGA_REQUIRE(workspace && workspace_bytes >= need, MEGA_ERR_WORKSPACE, "norm_ema_fwd: workspace of %zu bytes needed",
               need);
  hipStream_t s = (hipStream_t)stream;
  const int64_t S = ceil_div(L > 0 ? L : 1, kFSeg);
  char* w = (char*)workspace;
  const bool one_kernel = L > 0 && (image || mega_ema_image_bytes(D, N, 0) > 0) &&
                          fused_covers(dtype, B, L, D, G, N, x, xn, y, syb, syd, syl, h_in, h_out);
  if (!one_kernel || !image) {
    const size_t sneed = mega_norm_ema_fwd_scratch_bytes(B, L > 0 ? L : 1, D, G, N);
    MEGA_REQUIRE(scratch && scratch_bytes >= sneed, MEGA_ERR_WORKSPACE, "norm_ema_fwd: scratch of %zu bytes needed",
                 sneed);
  }
  if (one_kernel) {
    MEGA_REQUIRE(x && xn && y && prev_count && prev_mean && prev_var && norm_gamma && norm_beta && count && mean &&
                     var && p && q && gamma && omega,
                 MEGA_ERR_ARG, "norm_ema_fwd: null pointer argument");
    MEGA_REQUIRE(!ranges_overlap(prev_count, (size_t)B * 8, count, (size_t)B * 8) &&
                     !ranges_overlap(prev_mean, (size_t)B * G * 4, mean, (size_t)B * G * 4) &&
                     !ranges_overlap(prev_var, (size_t)B * G * 4, var, (size_t)B * G * 4),
                 MEGA_ERR_ARG, "norm_ema_fwd: count / mean / var must not overlap prev_count / prev_mean / prev_var");
    MEGA_REQUIRE(!h_in || !h_out || !ranges_overlap(h_in, (size_t)B * D * N * 8, h_out, (size_t)B * D * N * 8),
                 MEGA_ERR_ARG, "norm_ema_fwd: h_out must not overlap h_in (every block reads h_in, the last writes h_out)");
    const void* img = image;
    if (!img) {
      // no cached image: kernel generation runs with every call
      const int rc = ema_image_build(p, q, gamma, is_complex, omega, D, N, 0, 1, scratch, s, (dtype == MEGA_BF16 ? kImgPC | kImgKT : kImgF16) | kImgBlocks);
      if (rc) return rc;
      img = scratch;
    }
    FusedArgs A;
    A.x = x; A.xn = xn; A.y = y; A.syb = syb; A.syd = syd; A.syl = syl;
    A.prev_count = prev_count; A.prev_mean = prev_mean; A.prev_var = prev_var; A.count = count; A.mean = mean;
    A.var = var; A.gamma = norm_gamma; A.beta = norm_beta; A.mask = mask; A.image = (const uint4*)img; A.h_in = h_in; A.h_out = h_out;
    A.cummean = cummean; A.cumrstd = cumrstd;
    A.hdr = (TsnHeader*)w; A.rec = (unsigned long long*)(w + align_up(sizeof(TsnHeader), 256));
    A.B = (int)B; A.L = (int)L; A.D = (int)D; A.G = (int)G; A.N = (int)N; A.S = (int)S; A.eps = (float)eps;
    A.pad = (int)(S * kFSeg - L);
    A.is_complex = is_complex;
    const int gc = (int)(D / G), cw = fused_channels(dtype, gc, B * D * S);
    A.xcd_map = (D / cw) % 8 == 0 ? 1 : 0;
    A.lb = lookback_launch(true);
    const dim3 grid((unsigned)(B * (D / cw) * S));
    // held-back starts only where the launch is one round of workgroups (one per compute unit) and fills most of it
    const int cus = device_cu_count();
    A.stagger = (S > 1 && S <= MEGA_FUSED_STAGGER_BLOCKS && (int64_t)grid.x <= cus &&
                 (int64_t)grid.x * MEGA_FUSED_STAGGER_FILL >= cus * (MEGA_FUSED_STAGGER_FILL - 1))
                    ? MEGA_FUSED_STAGGER
                    : 0;
    const int lout = syl == 1 ? 0 : 1;
    switch (dtype) {
      case MEGA_F32: fused_launch_width<float>(A, gc, cw, lout, grid, s); break;
      case MEGA_F16: fused_launch_width<f16_t>(A, gc, cw, lout, grid, s); break;
      default: fused_launch_width<bf16_t>(A, gc, cw, lout, grid, s); break;
    }
    MEGA_CHECK_LAUNCH("norm_ema_fwd");
    return lookback_verify("norm_ema_fwd", s);
  }
  // outside the one-kernel envelope: the two operators one after the other
  // (x -> xn by the norm, xn read through its transposed view by the moving average); the norm keeps its
  // launch header and tile records in the same workspace (same header, same protocol)
  int rc = mega_group_timestep_norm_fwd(x, xn, dtype, prev_count, prev_mean, prev_var, norm_gamma, norm_beta, mask, B, L,
                                        D, G, eps, count, mean, var, nullptr, cummean, cumrstd, workspace,
                                        workspace_bytes, stream);
  if (rc) return rc;
  return mega_ema_fwd(xn, y, dtype, L * D, 1, D, syb, syd, syl, p, q, gamma, is_complex, omega, mask, h_in, h_out, B, D,
                      N, L, 0, 0, 1, image, scratch, scratch_bytes, stream);
}

extern "C" int mega_norm_ema_fwd(const void* x, void* xn, void* y, int dtype, int64_t syb, int64_t syd, int64_t syl,
                                 const int64_t* prev_count, const float* prev_mean, const float* prev_var,
                                 const float* norm_gamma, const float* norm_beta, const uint8_t* mask, double eps,
                                 int64_t* count, float* mean, float* var, const float* p, const float* q,
                                 const float* gamma, int is_complex, const float* omega, const float* h_in,
                                 float* h_out, int64_t B, int64_t L, int64_t D, int64_t G, int64_t N,
                                 const void* image, void* workspace, size_t workspace_bytes, void* scratch,
                                 size_t scratch_bytes, void* stream) {
  return mega_norm_ema_fwd_train(x, xn, y, dtype, syb, syd, syl, prev_count, prev_mean, prev_var, norm_gamma, norm_beta,
                                 mask, eps, count, mean, var, nullptr, nullptr, p, q, gamma, is_complex, omega, h_in,
                                 h_out, B, L, D, G, N, image, workspace, workspace_bytes, scratch, scratch_bytes, stream);
}
