// attention_wide.hip: the long products of 16-bit attention with its weights in memory
#pragma once

#include "common.h"

namespace mega {

// One product per (row, head); element (m, k) of A, (n, k) of B at m * ld + k, or stored K-major k * ld + m.  Batch entry
// z = zo nin + zi starts at zo * s + zi * si of each operand.
struct AttnWideP {
  const void *A, *B;
  void* C;
  int64_t lda, ldb, ldc, sa, sb, sc, sai, sbi, sci;
  int nin, batches, M, N, K;
  int mt, nt;
  int tiles;           // of a batch entry
  int xcd;             // whole batch entries go to one XCD each (their number is a multiple of eight)
  // the score gradient: C = alpha E (A B^T - rowdot) where n <= m (causal) or everywhere
  const void* E;
  const float* rowdot; // [batches][M]
  int64_t lde, se, sei;
  float alpha;
  int causal;
};

// dS = alpha w (dy v^T - rowdot): both operands along k; causal: tiles that touch n <= m only
// y = P v: P along k, v K-major; causal: k ends with the tile's rows
// dv = w^T dy: both K-major; causal: k starts with the tile's rows
enum AttnWide { kScoreGrad, kValues, kValueGrad };

// whether the wide tiles take it: leading dimensions (elements) within a tile's 32-bit offsets, grids within their limit
bool attention_wide_takes(const AttnWideP& P, AttnWide kind);
void attention_wide_launch(AttnWideP P, AttnWide kind, bool bf16, hipStream_t s);

// The weights themselves: P [batches][L][L] = softmax(scale q k^T) over the visible keys, zeros behind them (causal): to the
// end of the row, or of the 256 columns that hold the diagonal
struct AttnWeightsP {
  const void *q, *k;   // [B][L][Nh][H1]
  void* P;
  int L, Nh, H1, batches;
  float scale;
  int causal, zero_all;
  int xcd, qt;         // tiles of queries
};
bool attention_weights_takes(const AttnWeightsP& A);
void attention_weights_launch(AttnWeightsP A, bool bf16, hipStream_t s);

}  // namespace mega
