// Instantiations of the two-product launch, f16 operands.
#include "gemm_pair.hpp"

namespace brk {
int gemm_pair_f16(const gemm16::GemmArgs& w, const gemm16::Problem& pw, long long batch_w, const gemm16::GemmArgs& x,
                 const gemm16::Problem& px, long long batch_x, int kernel, const gemm16::ColumnSums& sums,
                 const gemm16::PartialSums& later, hipStream_t st) {
    return gemm16::launch_pair<BR_GEMM_F16>(w, pw, batch_w, x, px, batch_x, kernel, sums, later, st);
}
}  // namespace brk
