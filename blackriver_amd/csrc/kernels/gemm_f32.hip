// fp32 instantiations of the small-tile GEMM template.
#include "gemm_flex.hpp"

namespace brk {
namespace {
template <bool WORDS>
int launch(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, long long batch, hipStream_t st) {
    using namespace gemm16;
    // Where a CU has at most one workgroup of the small tiles, eight waves walk along K instead of four, two to a SIMD.
    // Four / eight, us: 32 x 32 tiles, [128 x 512] K = 512 5.5 / 5.2, [200 x 768] K = 768 7.6 / 6.7, [64 x 2048] K = 8192 49 / 37;
    // 32 x 64, [512 x 1024] K = 4096 37.8 / 34.2, K = 1024 11.9 / 13.2.  With more tiles than CUs eight are 5-40 % slower.
    if constexpr (!WORDS) {
        const long long tiles = ceil_div(g.m, 32) * ceil_div(g.n, kCost[kernel].bn) * batch;
        if (kernel == kFlex32 && tiles <= 256 && g.k >= kFp32EightWaves) return launch_flex_fp32<32, 32, 8, WORDS>(g, p, batch, st);
        if (kernel == kFlex32x64 && tiles <= 256 && g.k >= 3072) return launch_flex_fp32<32, 64, 8, WORDS>(g, p, batch, st);
    }
    if (kernel == kFlex64) return launch_flex_fp32<64, 64, 4, WORDS>(g, p, batch, st);
    if (kernel == kFlex32x64) return launch_flex_fp32<32, 64, 4, WORDS>(g, p, batch, st);
    return launch_flex_fp32<32, 32, 4, WORDS>(g, p, batch, st);
}
}  // namespace
int gemm_fp32(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, bool words, long long batch, hipStream_t st) {
    return words ? launch<true>(g, p, kernel, batch, st) : launch<false>(g, p, kernel, batch, st);
}
}  // namespace brk
