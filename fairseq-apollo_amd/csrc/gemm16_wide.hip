// Wide-tile products: the plan, and the bf16 kernels (gemm16_wide_f16.hip: the same for fp16, a unit of its own so that both
// compile side by side).
#include "gemm16_wide.h"

namespace mega {

extern template void launch_wide_type<f16_t>(const Gemm16P&, const WidePlan&, int, int, hipStream_t);

// The tile and the split with the least estimated time.  Whole rounds of tiles (one on each compute unit) run unsplit; what is
// left over is split along the reduction over the idle units, into fp32 partial sums that a second kernel adds up.  In us:
// 1.4 a step and 10 a round with square tiles, 0.85 and 6 with tall ones, 5 and its traffic at 4 TB/s for the second kernel.
// High by 5 - 25 % of what warm operands take, for both kinds alike (8192 x 4352 x 1024 94.8, 77.3; 8192 x 2816 x 1024 58.8, 47.4;
// 8192 x 2048 x 2048 54.8, 52.0; 5000 x 1024 x 2048 33.2, 26.1), nearer with operands from memory (88.4, 61.5, -, 31.3): fit to
// compare plans, with each other and with the 64 x 64 tiles' estimate, not to tell times.  The parts take up to 200 MB of a call's
// workspace (192 tiles beside whole rounds, in four).
WidePlan gemm16_wide_plan(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = device_cu_count(), steps = ceil_div(K, kKS);
  WidePlan best = {};
  double least = 1e300;
  for (int tn = 256; tn >= 128; tn -= 128) {
    const double step = tn == 256 ? 1.4 : 0.85, round = tn == 256 ? 10 : 6;
    const int64_t tiles = ceil_div(M, kWideM) * ceil_div(N, tn), rest = tiles % cus;
    const double whole = (double)(tiles / cus) * (steps * step + round);
    for (int64_t want = 1; want <= 16 && (want == 1 || (rest && want * 4 <= steps)); ++want) {
      const int64_t len = ceil_div(steps, want), parts = ceil_div(steps, len);
      const double us = whole + (rest ? (double)ceil_div(rest * parts, cus) * (len * step + round) : 0.) +
                        (parts > 1 ? 5 + (double)rest * kWideM * tn * (4 * parts + 2) / 4e6 : 0.);
      if (us < least) {
        least = us;
        best = {us, tn, (int)parts, (int)(parts > 1 ? tiles - rest : tiles), (int)len * kKS, parts > 1 ? (size_t)(rest * parts) * kWideM * tn * 4 : 0};
      }
    }
  }
  return best;
}

void gemm16_wide_launch(Gemm16P G, const WidePlan& p, bool bf16, int ka, int kb, void* parts, hipStream_t s) {
  G.mt = (int)ceil_div(G.M, kWideM);
  G.nt = (int)ceil_div(G.N, p.tn);
  G.full = p.full;
  G.splits = p.splits;
  G.kstep = p.kstep;
  G.part = p.splits > 1 ? (float*)parts : nullptr;
  if (bf16) launch_wide_type<bf16_t>(G, p, ka, kb, s);
  else launch_wide_type<f16_t>(G, p, ka, kb, s);
}

}  // namespace mega
