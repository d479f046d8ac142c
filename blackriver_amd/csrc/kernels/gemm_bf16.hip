// bf16-multiplicand instantiations of the MFMA GEMM templates.
#include "gemm_dtl16.hpp"

namespace brk {
int gemm16_tiles_bf16(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, long long batch, hipStream_t st) {
    return gemm16::launch_dtl<BR_GEMM_BF16>(g, p, kernel, batch, st);
}
int gemm16_pair_bf16(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, int slot, hipStream_t st) {
    return gemm16::launch_dtl_pair<BR_GEMM_BF16>(g, p, kernel, slot, st);
}
}  // namespace brk
