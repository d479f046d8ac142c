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

// The workgroup's first four waves add up the rows, whatever it has: with the rows dealt to eight waves, whose sums meet one after
// the other, the result was up to 8 % further from 64 bits ([2048] from 200 rows 1.87e-8, from four waves 1.79e-8).
template <int CT>
__device__ __forceinline__ void sum_strip(const ColumnSums& s, int strip, float* lds) {
    constexpr int kVec = CT == BR_GEMM_F32 ? 4 : 8, kThreads = 256, kRows = kThreads / kSumLanes, kAhead = 4;
    const int lane = threadIdx.x % kSumLanes, first = threadIdx.x / kSumLanes;
    const int col = (strip * kSumLanes + lane) * kVec;
    float acc[kVec];
#pragma unroll
    for (int j = 0; j < kVec; j++) acc[j] = 0.f;
    if (threadIdx.x < kThreads && col < s.cols) {
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
    if (threadIdx.x < kThreads && (threadIdx.x & 63) < kSumLanes) {
#pragma unroll
        for (int j = 0; j < kVec; j++) lds[(threadIdx.x >> 6) * kWidth + lane * kVec + j] = acc[j];
    }
    __syncthreads();
    const int at = strip * kWidth + threadIdx.x;
    if (threadIdx.x < kWidth && at < s.cols) {
        float sum = lds[threadIdx.x];
#pragma unroll
        for (int w = 1; w < kThreads / 64; w++) sum += lds[w * kWidth + threadIdx.x];
        s.out[at] = sum * s.scale;
    }
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
template <int THREADS>
__device__ __forceinline__ void add_partials(const PartialSums& s, int group, flex_f32x4* lds) {
    constexpr int kSlices = 64;
    const int per = (s.cols4 + 15) / 16, array = group / per, q = threadIdx.x & 15, g = threadIdx.x >> 4;
    const int c4 = (group - array * per) * 16 + q;
    const flex_f32x4* part = s.partials + (long long)array * s.parts * s.cols4;
    constexpr int kEach = kSlices * 16 / THREADS, kStride = THREADS / 16;   // slices of a thread
    flex_f32x4 v[kEach];
#pragma unroll
    for (int k = 0; k < kEach; k++) {
        v[k] = 0.f;
        if (c4 < s.cols4)
            for (int p = g + kStride * k; p < s.parts; p += kSlices) v[k] += part[(long long)p * s.cols4 + c4];
        lds[(g + kStride * k) * 16 + q] = v[k];
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
    else add_partials<KW * 64>(later, (int)(id - n1 - n2 - n3), reinterpret_cast<flex_f32x4*>(lds));
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

// ---- weight gradients from few tokens -------------------------------------------
// 128 x 128 tiles of a product with both operands row-contiguous and an fp32 C: eight waves of 64 x 32, K steps of 64 in two
// buffers that all of them load.
//
// Why: the gradient of a weight from 16 to 300 tokens is many tiles of one to five K steps.  Dealt to four waves along K, most of
// them wait for the one that has the step, and a 32 x 64 tile costs its launch, a load's latency and the merging of four sums
// for 8 KB of C: 2048 workgroups for [4096 x 1024], three rounds of them.  256 of these tiles run in one, beside the
// other product, whose walk along K (up to 16 steps of four waves, 12 us) is what the launch then waits for: on eight waves half
// that.  What bounds it: below 6 us launch, first loads and the walk; [4096 x 1024] and its weight are 25 MB, 5 us of the 9 to 13.
template <int CT>
__device__ __forceinline__ void wide_product(const GemmArgs& g, unsigned id, unsigned groups, unsigned char* lds_raw) {
    constexpr int BM = 128, BN = 128, KT = 64, FM = 2, WM = 64, WN = 32;
    using T = FlexTile<CT, BM, true, false>;
    constexpr int kEach = T::kInstr / 8, kLoads = 2 * kEach, kStageBytes = 2 * T::kBytes;
    static_assert(T::kStep == KT && T::kInstr % 8 == 0 && 8 * WM * WN * 4 == 2 * kStageBytes, "the tile at the end fills both buffers");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave >> 2) * WM, wn = (wave & 3) * WN;
    long long batch;
    int tm, tn;
    tile_coords(g, id, groups, batch, tm, tn);
    const int row0 = __builtin_amdgcn_readfirstlane(tm) * BM, col0 = __builtin_amdgcn_readfirstlane(tn) * BN;
    const int b = __builtin_amdgcn_readfirstlane((int)batch), k = (int)g.k, steps = (k + KT - 1) / KT;
    const unsigned char* a_src = static_cast<const unsigned char*>(g.a) + 2 * (b * g.sa + row0);
    const unsigned char* b_src = static_cast<const unsigned char*>(g.b) + 2 * (b * g.sb + col0);
    // where the operands end, rounded up to the granule the last element lies in
    const long long a_end = (((k - 1) * g.lda + g.m - row0) * 2 + 15) & ~15LL, b_end = (((k - 1) * g.ldb + g.n - col0) * 2 + 15) & ~15LL;
    const long long a_step = g.lda * (2LL * KT), b_step = g.ldb * (2LL * KT);
    unsigned a_off[kEach], b_off[kEach];
#pragma unroll
    for (int q = 0; q < kEach; q++) {
        a_off[q] = T::source_offset(wave * kEach + q, lane, g.lda);
        b_off[q] = T::source_offset(wave * kEach + q, lane, g.ldb);
    }
    lds_byte* const lds = (lds_byte*)lds_raw;
    const unsigned lds0 = (unsigned)(unsigned long long)lds;
    auto issue = [&](int step, int stage) {
        const buffer_rsrc ra = buffer_from(a_src + step * a_step, a_end - step * a_step), rb = buffer_from(b_src + step * b_step, b_end - step * b_step);
        const unsigned dst = lds0 + (unsigned)stage * kStageBytes;
#pragma unroll
        for (int q = 0; q < kEach; q++) T::load(dst, wave * kEach + q, a_off[q], ra);
#pragma unroll
        for (int q = 0; q < kEach; q++) T::load(dst + T::kBytes, wave * kEach + q, b_off[q], rb);
    };
    // K is walked as the four waves of a small tile do, one after the other: steps 0, 4, 8, .., then 1, 5, ..; each of the four is a
    // sum of its own and then added to the others.  The bits are a small tile's.  (One sum that all of K goes through has up to 1.5
    // times the error: [1024 x 4096] from 300 tokens 1.14e-7 against 64 bits, so 7.6e-8.)
    auto after = [&](int step) { return step + 4 < steps ? step + 4 : (step & 3) + 1; };
    f32x16 acc[FM][1], all[FM][1];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[i][0][v] = all[i][0][v] = 0.f;
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) all[i][0][v] += acc[i][0][v];
    };
    int ahead = 0;   // the next step to load
    for (int t = 0; t < 2 && t < steps; t++, ahead = after(ahead)) issue(ahead, t);
    for (int t = 0, step = 0; t < steps; t++, step = after(step)) {
        // the step is in once at most the loads of the step after it are outstanding
        if (t + 1 < steps) wait_vmem<kLoads>();
        else wait_vmem<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const lds_byte* tile = lds + (t & 1) * kStageBytes;
        u32x4 fa[4][FM], fb[4];
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
#pragma unroll
            for (int i = 0; i < FM; i++) fa[ks][i] = T::fragment(tile, T::frag_offset(wm + i * 32, ks, lane));
            fb[ks] = T::fragment(tile + T::kBytes, T::frag_offset(wn, ks, lane));
        }
        const bool fresh = step < 4;   // the next of the four sums
        if (fresh) fold();             // while the fragments are on their way
        // the buffer takes the step after the next one (or, at the end, the sums) once every wave has read it
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (t + 2 < steps) {
            issue(ahead, t & 1);
            ahead = after(ahead);
        }
        if (fresh) {
#pragma unroll
            for (int i = 0; i < FM; i++) acc[i][0] = Cvt<CT>::mfma(fb[0], fa[0][i], f32x16{});
        } else {
#pragma unroll
            for (int i = 0; i < FM; i++) acc[i][0] = Cvt<CT>::mfma(fb[0], fa[0][i], acc[i][0]);
        }
#pragma unroll
        for (int ks = 1; ks < 4; ks++)
#pragma unroll
            for (int i = 0; i < FM; i++) acc[i][0] = Cvt<CT>::mfma(fb[ks], fa[ks][i], acc[i][0]);
    }
    fold();
    // by way of LDS, a part of each wave's own, to whole lines of C
    lds_byte* const mine = lds + wave * (WM * WN * 4);
    flex_park<WM, WN>(all, mine, lane);
    __builtin_amdgcn_wave_barrier();
    float* const c_base = static_cast<float*>(g.c) + b * g.sc;
    const lds_f32x4* const sums = (const lds_f32x4*)mine;
#pragma unroll
    for (int it = 0; it < WM * WN / 256; it++) {
        const int r = it * 8 + (lane >> 3), c = lane & 7;
        flex_f32x4 s = sums[r * 8 + (c ^ (r & 7))];
        s *= g.alpha;
        const int row = row0 + wm + r, col = col0 + wn + c * 4;
        if (row >= g.m) continue;
        float* const to = c_base + row * g.ldc + col;
        const int left = (int)(g.n - col);
        if (left >= 4 && g.vec_c) {
            *reinterpret_cast<float4*>(to) = make_float4(s.x, s.y, s.z, s.w);
        } else {
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (u < left) to[u] = s[u];
        }
    }
}

// gemm_flex_pair_kernel with the weight gradient `w` on such tiles, x on 32 x 32 ones whose K is dealt to eight waves.
// x first: its workgroups walk further along K.
template <int CT, bool BK2, typename TC2>
__global__ __launch_bounds__(512, 4) void gemm_wide_pair_kernel(GemmArgs x, GemmArgs w, unsigned nx, unsigned nw, unsigned n3, ColumnSums sums, PartialSums later) {
    constexpr int kBytes = flex_lds_bytes<32, 32, 8, 1>();
    static_assert(kBytes == 4 * FlexTile<CT, 128, true, false>::kBytes && kBytes >= 64 * 16 * sizeof(flex_f32x4), "LDS of all parts");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kBytes];
    const unsigned id = blockIdx.x;
    if (id < nx) flex_product<CT, 32, 32, 8, 1, false, BK2, TC2, false, false, false>(x, id, nx, lds);
    else if (id < nx + nw) wide_product<CT>(w, id - nx, nw, lds);
    else if (id < nx + nw + n3) sum_strip<CT>(sums, (int)(id - nx - nw), reinterpret_cast<float*>(lds));
    else add_partials<512>(later, (int)(id - nx - nw - n3), reinterpret_cast<flex_f32x4*>(lds));
}

template <int CT>
int launch_wide_pair(GemmArgs w, const Problem& pw, long long batch_w, GemmArgs x, const Problem& px, long long batch_x,
                     const ColumnSums& sums, const PartialSums& later, hipStream_t st) {
    const long long nw = flex_tiles<128, 128>(w, pw, batch_w), nx = flex_tiles<32, 32>(x, px, batch_x);
    if (nw < 0 || nx < 0) return BR_ERR_TODO;
    const unsigned extra = sums.x ? ((unsigned)sums.cols + kSumLanes * 8 - 1) / (kSumLanes * 8) : 0;
    if (nw + nx + extra + later.groups() > 0x7fffffffLL / 512) return BR_ERR_TODO;
    const unsigned grid = (unsigned)(nw + nx + extra + later.groups());
    using T = std::conditional_t<CT == BR_GEMM_F16, __half, __hip_bfloat16>;
    if (px.c_dtype != BR_F32 && px.b_kstr)
        gemm_wide_pair_kernel<CT, true, T><<<grid, 512, 0, st>>>(x, w, (unsigned)nx, (unsigned)nw, extra, sums, later);
    else if (px.c_dtype != BR_F32)
        gemm_wide_pair_kernel<CT, false, T><<<grid, 512, 0, st>>>(x, w, (unsigned)nx, (unsigned)nw, extra, sums, later);
    else if (px.b_kstr)
        gemm_wide_pair_kernel<CT, true, float><<<grid, 512, 0, st>>>(x, w, (unsigned)nx, (unsigned)nw, extra, sums, later);
    else
        gemm_wide_pair_kernel<CT, false, float><<<grid, 512, 0, st>>>(x, w, (unsigned)nx, (unsigned)nw, extra, sums, later);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

template <int CT>
int launch_pair(const GemmArgs& w, const Problem& pw, long long batch_w, const GemmArgs& x, const Problem& px,
                long long batch_x, int kernel, const ColumnSums& sums, const PartialSums& later, hipStream_t st) {
    constexpr int ST32 = CT == BR_GEMM_F32 ? 1 : 2;   // as each is launched by itself
    if constexpr (CT != BR_GEMM_F32)
        if (kernel == kPairWide) return launch_wide_pair<CT>(w, pw, batch_w, x, px, batch_x, sums, later, st);
    if (kernel == kFlex64) return launch_pair_config<CT, 64, 64, 4, 1>(w, pw, batch_w, x, px, batch_x, sums, later, st);
    if (kernel == kFlex32x64) return launch_pair_config<CT, 32, 64, 4, 1>(w, pw, batch_w, x, px, batch_x, sums, later, st);
    return launch_pair_config<CT, 32, 32, 4, ST32>(w, pw, batch_w, x, px, batch_x, sums, later, st);
}

}  // namespace gemm16
}  // namespace brk
