// fp32 instantiations of the small-tile GEMM template.
#include "gemm_flex.hpp"

namespace brk {
namespace {
template <bool WORDS>
int launch(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, long long batch, hipStream_t st) {
    using namespace gemm16;
    if (fp32_waves(kernel, g.m, g.n, g.k, batch) == 8)
        return kernel == kFlex32 ? launch_flex_fp32<32, 32, 8, WORDS>(g, p, batch, st) : launch_flex_fp32<32, 64, 8, WORDS>(g, p, batch, st);
    if (kernel == kFlex64) return launch_flex_fp32<64, 64, 4, WORDS>(g, p, batch, st);
    if (kernel == kFlex32x64) return launch_flex_fp32<32, 64, 4, WORDS>(g, p, batch, st);
    return launch_flex_fp32<32, 32, 4, WORDS>(g, p, batch, st);
}
}  // namespace
int gemm_fp32(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, bool words, long long batch, hipStream_t st) {
    return words ? launch<true>(g, p, kernel, batch, st) : launch<false>(g, p, kernel, batch, st);
}
}  // namespace brk
