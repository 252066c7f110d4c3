// Gradient of a small vocabulary's embedding table: dw[v] = sum of dy[t] over the tokens t with id v, zeros for the padding
// id and for ids that do not occur (torch's embedding backward; its sort, segment search and sums are 19 launches, 112 us for
// 8192 tokens of 1024 channels in bf16 on 264 rows, here 2, 36 us).
//
// A wave owns 64 columns and a run of tokens, and the whole table's sums of them in LDS: a token is one 128-byte line (16-bit
// types) and one addition per lane, in the order of the tokens; nobody else touches the wave's sums.  Four tokens are read, added
// and written back together, equal ids among them taking the sum so far from each other (one by one each waits for the LDS;
// its own atomic additions take 50 us instead of 29).  The runs' sums go to
// memory and a second kernel adds them in order.  What bounds it is a run's chain through the LDS,
// two waves on a compute unit (loads of the next tokens beside the additions changed nothing), so the runs are as many as give
// every compute unit two, of at least 64 tokens.
#include "common.h"

namespace mega {
namespace {

constexpr int kEgAhead = 16;          // tokens on their way from memory
constexpr int kEgRows = 318;          // of a table: two workgroups on a compute unit's 160 KB
constexpr int kEgTurn = 4;            // tokens that one wait for the LDS serves

struct EmbedGradP {
  const int64_t* ids;  // [T]
  const void* dy;      // [T][D]
  float* part;         // [runs][V][D]
  void* dw;            // [V][D]
  int64_t T, run;
  int V, D, padding, runs;
};

template <typename T>
__global__ __launch_bounds__(64) void embed_grad_kernel(const EmbedGradP P) {
  extern __shared__ float sums[];                                  // [V + 1][64]; the last row: ids beyond the table
  const int lane = threadIdx.x, d = blockIdx.x * 64 + lane;
#pragma unroll 8
  for (int v = 0; v <= P.V; ++v) sums[v * 64 + lane] = 0.f;
  const int64_t t0 = (int64_t)blockIdx.y * P.run, t1 = min(P.T, t0 + P.run);
  if (d < P.D) {
    const T* dy = (const T*)P.dy + d;
    int64_t t = t0;
    for (; t + kEgAhead <= t1; t += kEgAhead) {
      T x[kEgAhead];
      int64_t id[kEgAhead];
#pragma unroll
      for (int u = 0; u < kEgAhead; ++u) {
        x[u] = dy[(t + u) * P.D];
        id[u] = P.ids[t + u];
      }
#pragma unroll
      for (int u = 0; u < kEgAhead; u += kEgTurn) {
        int at[kEgTurn];
        float s[kEgTurn];
#pragma unroll
        for (int e = 0; e < kEgTurn; ++e) {
          at[e] = (uint64_t)id[u + e] < (uint64_t)P.V ? (int)id[u + e] : P.V;
          s[e] = sums[at[e] * 64 + lane];
        }
#pragma unroll
        for (int e = 0; e < kEgTurn; ++e) {
#pragma unroll
          for (int f = 0; f < e; ++f) s[e] = at[f] == at[e] ? s[f] : s[e];     // (the last of them)
          s[e] += to_float(x[u + e]);
        }
#pragma unroll
        for (int e = 0; e < kEgTurn; ++e) sums[at[e] * 64 + lane] = s[e];
      }
    }
    for (; t < t1; ++t) {
      const int64_t id = P.ids[t];
      if ((uint64_t)id < (uint64_t)P.V) sums[(int)id * 64 + lane] += to_float(dy[t * P.D]);
    }
    float* part = P.part + (int64_t)blockIdx.y * P.V * P.D + d;
#pragma unroll 8
    for (int v = 0; v < P.V; ++v) part[(int64_t)v * P.D] = sums[v * 64 + lane];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void embed_grad_sum_kernel(const EmbedGradP P) {
  const int64_t total = (int64_t)P.V * P.D, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  float s = 0.f;
#pragma unroll 8
  for (int r = 0; r < P.runs; ++r) s += P.part[r * total + i];
  ((T*)P.dw)[i] = from_float<T>(i / P.D == P.padding ? 0.f : s);
}

void plan(int64_t T, int64_t D, int64_t* run, int* runs) {
  const int64_t want = ceil_div(2 * device_cu_count(), ceil_div(D, 64)), most = ceil_div(T, 64);
  const int64_t n = want < most ? want : most;
  *run = ceil_div(T, n);
  *runs = (int)ceil_div(T, *run);
}

template <typename T>
void launch(const EmbedGradP& P, hipStream_t s) {
  static uint64_t seen = 0;
  const int smem = (P.V + 1) * 256;
  if (smem > 64 * 1024) raise_lds_limit(&seen, (kEgRows + 1) * 256, embed_grad_kernel<T>);
  hipLaunchKernelGGL(embed_grad_kernel<T>, dim3((unsigned)ceil_div(P.D, 64), (unsigned)P.runs), dim3(64), smem, s, P);
  hipLaunchKernelGGL(embed_grad_sum_kernel<T>, dim3((unsigned)ceil_div((int64_t)P.V * P.D, 256)), dim3(256), 0, s, P);
}

}  // namespace
}  // namespace mega

using namespace mega;

// Tables whose 64 columns of fp32 sums fit the LDS with two workgroups on a compute unit; 0 otherwise
extern "C" size_t mega_embedding_grad_workspace_bytes(int64_t T, int64_t V, int64_t D) {
  if (T <= 0 || V <= 0 || D <= 0 || V > kEgRows || T >= (int64_t)1 << 31 || D >= (int64_t)1 << 20) return 0;
  int64_t run;
  int runs;
  plan(T, D, &run, &runs);
  return (size_t)runs * V * D * 4;
}

extern "C" int mega_embedding_grad(const int64_t* ids, const void* dy, void* dw, int dtype, int64_t T, int64_t V, int64_t D,
                                   int64_t padding_id, void* workspace, size_t workspace_bytes, void* stream) {
  MEGA_REQUIRE(dtype == MEGA_F32 || dtype == MEGA_BF16 || dtype == MEGA_F16, MEGA_ERR_ARG, "embedding_grad: unknown dtype %d", dtype);
  const size_t need = mega_embedding_grad_workspace_bytes(T, V, D);
  MEGA_REQUIRE(need, MEGA_ERR_UNSUPPORTED, "embedding_grad: 1 to 318 rows, fewer than 2^31 tokens of fewer than 2^20 channels");
  MEGA_REQUIRE(ids && dy && dw, MEGA_ERR_ARG, "embedding_grad: null pointer argument");
  MEGA_REQUIRE(workspace && workspace_bytes >= need && (uintptr_t)workspace % 4 == 0, MEGA_ERR_WORKSPACE,
               "embedding_grad: workspace of %zu bytes needed", need);
  EmbedGradP P = {ids, dy, (float*)workspace, dw, T, 0, (int)V, (int)D, (int)(padding_id >= 0 && padding_id < V ? padding_id : -1), 0};
  plan(T, D, &P.run, &P.runs);
  if (dtype == MEGA_BF16) launch<bf16_t>(P, (hipStream_t)stream);
  else if (dtype == MEGA_F16) launch<f16_t>(P, (hipStream_t)stream);
  else launch<float>(P, (hipStream_t)stream);
  MEGA_CHECK_LAUNCH("embedding_grad");
  return MEGA_OK;
}
