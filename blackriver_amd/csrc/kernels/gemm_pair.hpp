// Two small products in one launch, and a column sum beside them.
//
// The backward pass of a linear layer multiplies its output gradient twice, dW = dy^T x and dx = dy W, and sums its
// columns; the backward pass of attention does the like with the probabilities and with the scores' gradient.  None of
// these reads what another writes.  Up to a few hundred tokens each is a launch of 4-10 us that leaves most of the chip
// idle, and most of that time is the launch, the first loads and the merging of the waves' sums.  Here the workgroups of
// all of them are one launch: a workgroup's number says which product it belongs to.  Every tile is summed as
// gemm_flex_kernel sums it (gemm_flex.hpp).
//
// Measured, both products as two launches / as one (fp16, us): 63 tokens, 384 -> 384 features 7.4 / 4.1; 140 tokens,
// 384 -> 1536 10.3 / 6.3; 516 tokens, 640 -> 640 11.2 / 6.9; 885 tokens, 640 -> 2560 26.4 / 18.3; attention heads of 48
// tokens 6.9 / 3.7; fp32, 212 tokens, 896 -> 3584 48.9 / 37.9.  A block of 2 x 32 tokens of 256 features, forward and
// backward, 101 -> 87 us; 4 x 250 tokens of 1024 on the operator chain 450 -> 423.
#pragma once
#include "gemm_flex.hpp"

namespace brk {
namespace gemm16 {

// Column sums of a dense [rows, cols] matrix of the products' type (a bias gradient); x == null: none.
struct ColumnSums {
    const void* x = nullptr;
    float* out = nullptr;
    int rows = 0, cols = 0;
    float scale = 1.0f;
};
constexpr int kSumLanes = 8;   // 16-byte granules of a row one workgroup sums

template <int CT>
__device__ __forceinline__ void sum_strip(const ColumnSums& s, int strip, float* lds) {
    constexpr int kVec = CT == BR_GEMM_F32 ? 4 : 8, kRows = 256 / kSumLanes, kAhead = 4;
    const int lane = threadIdx.x % kSumLanes, first = threadIdx.x / kSumLanes;
    const int col = (strip * kSumLanes + lane) * kVec;
    float acc[kVec];
#pragma unroll
    for (int j = 0; j < kVec; j++) acc[j] = 0.f;
    if (col < s.cols) {
        const u32x4* x = static_cast<const u32x4*>(s.x) + col / kVec;
        const int pitch = s.cols / kVec;
        for (int r = first; r < s.rows; r += kAhead * kRows) {
            u32x4 v[kAhead];
            // rows past the last one read that row: all loads leave before the first is used
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const int at = r + u * kRows;
                v[u] = x[(long long)(at < s.rows ? at : s.rows - 1) * pitch];
            }
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                if (r + u * kRows >= s.rows) break;
                if constexpr (CT == BR_GEMM_F32) {
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[j] += __uint_as_float(v[u][j]);
                } else {
                    typedef std::conditional_t<CT == BR_GEMM_F16, f16x8, bf16x8> T8;
                    const T8 h = __builtin_bit_cast(T8, v[u]);
#pragma unroll
                    for (int j = 0; j < kVec; j++) acc[j] += (float)h[j];
                }
            }
        }
    }
    // the row slots of a wave meet by lane exchanges, the waves through LDS
#pragma unroll
    for (int d = kSumLanes; d < 64; d *= 2)
#pragma unroll
        for (int j = 0; j < kVec; j++) acc[j] += __shfl_xor(acc[j], d);
    constexpr int kWidth = kSumLanes * kVec;
    if ((threadIdx.x & 63) < kSumLanes) {
#pragma unroll
        for (int j = 0; j < kVec; j++) lds[(threadIdx.x >> 6) * kWidth + lane * kVec + j] = acc[j];
    }
    __syncthreads();
    const int at = strip * kWidth + threadIdx.x;
    if (threadIdx.x < kWidth && at < s.cols)
        s.out[at] = (lds[threadIdx.x] + lds[kWidth + threadIdx.x] + lds[2 * kWidth + threadIdx.x] + lds[3 * kWidth + threadIdx.x]) * s.scale;
}

// What a LayerNorm backward has left to add up: `arrays` of `parts` partial rows of cols4 quads, one behind the other.
// In a launch of their own these sums take 4 us, nearly all of it the launch; beside the products next to nothing: the
// forward and backward pass of a block 82.7 -> 79.3 us on [64 x 256] and 135.1 -> 132.8 on [78 x 1024]; no difference on
// [1000 x 1024], where the products fill the chip (366.8 and 366.5).
struct PartialSums {
    const flex_f32x4* partials = nullptr;   // null: none
    flex_f32x4* out[3] = {nullptr, nullptr, nullptr};
    int arrays = 0, parts = 0, cols4 = 0;
    float scale = 1.0f;
    int groups() const { return partials ? arrays * ((cols4 + 15) / 16) : 0; }
};
// 16 quads of columns of one array, in the order of ln_bwd_finalize_x4 (layernorm.hip): 64 slices of the parts, folded
// 8 at a time.
__device__ __forceinline__ void add_partials(const PartialSums& s, int group, flex_f32x4* lds) {
    constexpr int kSlices = 64;
    const int per = (s.cols4 + 15) / 16, array = group / per, q = threadIdx.x & 15, g = threadIdx.x >> 4;
    const int c4 = (group - array * per) * 16 + q;
    const flex_f32x4* part = s.partials + (long long)array * s.parts * s.cols4;
    flex_f32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = 0.f;
        if (c4 < s.cols4)
            for (int p = g + 16 * k; p < s.parts; p += kSlices) v[k] += part[(long long)p * s.cols4 + c4];
        lds[(g + 16 * k) * 16 + q] = v[k];
    }
    __syncthreads();
    if (g < 8) {
        for (int k = g + 8; k < kSlices; k += 8) v[0] += lds[k * 16 + q];
    }
    __syncthreads();
    if (g < 8) lds[g * 16 + q] = v[0];
    __syncthreads();
    if (g == 0 && c4 < s.cols4) {
        for (int k = 1; k < 8; k++) v[0] += lds[k * 16 + q];
        flex_f32x4* const out = array == 0 ? s.out[0] : array == 1 ? s.out[1] : s.out[2];
        out[c4] = v[0] * s.scale;
    }
}

// Workgroups [0, n1) run `a`, [n1, n1 + n2) run `b`, those after them the column sums and the partial sums.  AK1 .. BK2:
// which operands are row-contiguous.
template <int CT, int BM, int BN, int KW, int ST, bool AK1, bool BK1, typename TC1, bool AK2, bool BK2, typename TC2>
__global__ __launch_bounds__(KW * 64, CT == BR_GEMM_F32 ? 2 : 1) void gemm_flex_pair_kernel(GemmArgs a, GemmArgs b, unsigned n1, unsigned n2, unsigned n3, ColumnSums sums,
                                                                                       PartialSums later) {
    static_assert(KW == 4, "the column sums are four waves'");
    static_assert(flex_lds_bytes<BM, BN, KW, ST>() >= 64 * 16 * sizeof(flex_f32x4), "add_partials' slices");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[flex_lds_bytes<BM, BN, KW, ST>()];
    const unsigned id = blockIdx.x;
    if (id < n1) flex_product<CT, BM, BN, KW, ST, AK1, BK1, TC1, false, false, false>(a, id, n1, lds);
    else if (id < n1 + n2) flex_product<CT, BM, BN, KW, ST, AK2, BK2, TC2, false, false, false>(b, id - n1, n2, lds);
    else if (id < n1 + n2 + n3) sum_strip<CT>(sums, (int)(id - n1 - n2), reinterpret_cast<float*>(lds));
    else add_partials(later, (int)(id - n1 - n2 - n3), reinterpret_cast<flex_f32x4*>(lds));
}

// `w`: C of fp32, both operands row-contiguous.  `x`: A k-contiguous.  The one whose workgroups walk further along K
// starts first.
template <int CT, int BM, int BN, int KW, int ST, bool BK2, typename TC2>
int launch_pair_layout(const GemmArgs& w, const GemmArgs& x, unsigned nw, unsigned nx, const ColumnSums& sums,
                       const PartialSums& later, hipStream_t st) {
    const unsigned strip = kSumLanes * (CT == BR_GEMM_F32 ? 4 : 8);
    const unsigned extra = sums.x ? ((unsigned)sums.cols + strip - 1) / strip : 0;
    if ((long long)nw + nx + extra + later.groups() > 0x7fffffffLL / (KW * 64)) return BR_ERR_TODO;
    const unsigned grid = nw + nx + extra + (unsigned)later.groups();
    if (x.k >= w.k)
        gemm_flex_pair_kernel<CT, BM, BN, KW, ST, false, BK2, TC2, true, true, float><<<grid, KW * 64, 0, st>>>(x, w, nx, nw, extra, sums, later);
    else
        gemm_flex_pair_kernel<CT, BM, BN, KW, ST, true, true, float, false, BK2, TC2><<<grid, KW * 64, 0, st>>>(w, x, nw, nx, extra, sums, later);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

template <int CT, int BM, int BN, int KW, int ST>
int launch_pair_config(GemmArgs w, const Problem& pw, long long batch_w, GemmArgs x, const Problem& px, long long batch_x,
                       const ColumnSums& sums, const PartialSums& later, hipStream_t st) {
    const long long nw = flex_tiles<BM, BN>(w, pw, batch_w), nx = flex_tiles<BM, BN>(x, px, batch_x);
    if (nw < 0 || nx < 0) return BR_ERR_TODO;
    if constexpr (CT != BR_GEMM_F32) {
        using T = std::conditional_t<CT == BR_GEMM_F16, __half, __hip_bfloat16>;
        if (px.c_dtype != BR_F32) {
            if (px.b_kstr) return launch_pair_layout<CT, BM, BN, KW, ST, true, T>(w, x, (unsigned)nw, (unsigned)nx, sums, later, st);
            return launch_pair_layout<CT, BM, BN, KW, ST, false, T>(w, x, (unsigned)nw, (unsigned)nx, sums, later, st);
        }
    }
    if (px.b_kstr) return launch_pair_layout<CT, BM, BN, KW, ST, true, float>(w, x, (unsigned)nw, (unsigned)nx, sums, later, st);
    return launch_pair_layout<CT, BM, BN, KW, ST, false, float>(w, x, (unsigned)nw, (unsigned)nx, sums, later, st);
}

template <int CT>
int launch_pair(const GemmArgs& w, const Problem& pw, long long batch_w, const GemmArgs& x, const Problem& px,
                long long batch_x, int kernel, const ColumnSums& sums, const PartialSums& later, hipStream_t st) {
    constexpr int ST32 = CT == BR_GEMM_F32 ? 1 : 2;   // as each is launched by itself
    if (kernel == kFlex64) return launch_pair_config<CT, 64, 64, 4, 1>(w, pw, batch_w, x, px, batch_x, sums, later, st);
    if (kernel == kFlex32x64) return launch_pair_config<CT, 32, 64, 4, 1>(w, pw, batch_w, x, px, batch_x, sums, later, st);
    return launch_pair_config<CT, 32, 32, 4, ST32>(w, pw, batch_w, x, px, batch_x, sums, later, st);
}

}  // namespace gemm16
}  // namespace brk
