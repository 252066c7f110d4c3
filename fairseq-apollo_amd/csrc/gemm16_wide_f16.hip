// Wide-tile products of fp16 operands.
#include "gemm16_wide.h"

namespace mega {

template void launch_wide_type<f16_t>(const Gemm16P&, const WidePlan&, int, int, hipStream_t);

}  // namespace mega
