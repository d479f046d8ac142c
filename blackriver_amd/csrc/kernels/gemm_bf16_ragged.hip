// bf16-multiplicand instantiations of the GEMM templates for small and ragged products, and of the register-staged
// kernel for operands none of the direct-to-LDS kernels takes.
#include "gemm_dtl16.hpp"
#include "gemm_flex.hpp"

namespace brk {
int gemm16_ragged_bf16(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, long long batch, hipStream_t st) {
    using namespace gemm16;
    if (kernel == kTile256) return launch_dtl_ragged<BR_GEMM_BF16, 256, 256, 64, 128, 2>(g, p, batch, st);
    if (kernel == kTile256x128) return launch_dtl_ragged<BR_GEMM_BF16, 256, 128, 64, 64, 3>(g, p, batch, st);
    if (kernel == kTile128) return launch_dtl_ragged<BR_GEMM_BF16, 128, 128, 64, 64, 2>(g, p, batch, st);
    return launch_flex<BR_GEMM_BF16>(g, p, kernel, batch, st);
}
int gemm16_registers_bf16(const gemm16::GemmArgs& g, const gemm16::Problem& p, long long batch, hipStream_t st) {
    return gemm16::launch<BR_GEMM_BF16>(g, p, batch, st);
}
}  // namespace brk
