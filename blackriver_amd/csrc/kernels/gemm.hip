// Strided-batched GEMM entry point of the C ABI.
//
//   C[b][i,j] = alpha * sum_p opA[b][i,p] * opB[b][p,j] (+ C) (+ bias[j])
//
// 16-bit multiplicands (fp16 / bf16, fp32 accumulation) go to the kernel
// templates in gemm_dtl16.hpp and gemm_flex.hpp (both operands stored in the
// MFMA type, aligned: direct-to-LDS loads; gemm_plan.hpp chooses between them)
// and gemm_mfma16.hpp (fp32 operands converted on load, unaligned rows).  This
// file holds the argument checking, the staging of fp32 and of unaligned
// operands into a caller's workspace so that they too can take the
// direct-to-LDS kernels, and a kernel for fp32 products of many whole tiles from a
// short K, and for those whose leading dimensions are too long for the 32-bit
// offsets of the one in gemm_flex.hpp (128x128x16 tiles, 4 wave64s x 2x2 MFMA
// blocks, register prefetch + LDS double buffering).
#include "common.hpp"

#include <hip/hip_bf16.h>

#include <stdlib.h>
#include <string.h>

#include "gemm_dtl16.hpp"
#include "gemm_pair.hpp"

using namespace brk;

namespace brk {
#define BR_GEMM16_ENTRIES(T)                                                                                             \
    int gemm16_tiles_##T(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, long long batch, hipStream_t st);  \
    int gemm16_pair_##T(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, int slot, hipStream_t st);          \
    int gemm16_ragged_##T(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, long long batch, hipStream_t st); \
    int gemm16_registers_##T(const gemm16::GemmArgs& g, const gemm16::Problem& p, long long batch, hipStream_t st);
BR_GEMM16_ENTRIES(f16)
BR_GEMM16_ENTRIES(bf16)
#undef BR_GEMM16_ENTRIES
int gemm_fp32(const gemm16::GemmArgs& g, const gemm16::Problem& p, int kernel, bool words, long long batch, hipStream_t st);
#define BR_GEMM_PAIR_ENTRY(T)                                                                                            \
    int gemm_pair_##T(const gemm16::GemmArgs& w, const gemm16::Problem& pw, long long batch_w, const gemm16::GemmArgs& x,    \
                      const gemm16::Problem& px, long long batch_x, int kernel, const gemm16::ColumnSums& sums,                   \
                      const gemm16::PartialSums& later, hipStream_t st);
BR_GEMM_PAIR_ENTRY(f16)
BR_GEMM_PAIR_ENTRY(bf16)
BR_GEMM_PAIR_ENTRY(f32)
#undef BR_GEMM_PAIR_ENTRY
}  // namespace brk

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
using gemm16::GemmArgs;

constexpr int BM = 128, BN = 128;
constexpr int kThreads = 256;

// m varies fastest so that neighbouring workgroups share one panel of B
__device__ __forceinline__ void tile_coords32(const GemmArgs& g, long long& batch, int& tm, int& tn) {
    const unsigned tiles_m = (unsigned)g.tiles_m, per_batch = tiles_m * (unsigned)g.tiles_n, id = blockIdx.x;
    const unsigned entry = id < per_batch ? 0 : id / per_batch;
    const unsigned rem = id - entry * per_batch;
    batch = entry;
    tn = (int)(rem / tiles_m);
    tm = (int)(rem - tn * tiles_m);
}

// ---- fp32 operands on v_mfma_f32_32x32x2_f32 ------------------------------
// Same tiling with BK = 16 fp32 values per step; LDS rows padded to 20 floats.
constexpr int BK32 = 16;
constexpr int kPitch32 = BK32 + 4;

template <bool KSTR>
struct TileLoader32 {
    float4 r[2];
    __device__ __forceinline__ void fetch(const float* base, long long ld, long long row0, long long rows,
                                          long long k0, long long kdim, bool vec) {
        const int t = threadIdx.x;
        if (!KSTR) {
            const int c = t & 3, r0 = t >> 2;  // 4 k-values per chunk, 64 rows per pass
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const long long row = row0 + r0 + 64 * p;
                const long long off = row * ld + k0 + c * 4;
                if (vec && row < rows && k0 + c * 4 + 4 <= kdim) {
                    r[p] = *reinterpret_cast<const float4*>(base + off);
                } else {
                    float w[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) w[e] = (row < rows && k0 + c * 4 + e < kdim) ? base[off + e] : 0.f;
                    r[p] = make_float4(w[0], w[1], w[2], w[3]);
                }
            }
        } else {
            const int r4 = t & 31, kg = t >> 5;  // 4 rows x 2 k-values per thread
            const long long row = row0 + 4 * r4;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const long long kidx = k0 + 2 * kg + kk;
                const long long off = kidx * ld + row;
                if (vec && row + 4 <= rows && kidx < kdim) {
                    r[kk] = *reinterpret_cast<const float4*>(base + off);
                } else {
                    float w[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) w[e] = (row + e < rows && kidx < kdim) ? base[off + e] : 0.f;
                    r[kk] = make_float4(w[0], w[1], w[2], w[3]);
                }
            }
        }
    }
    __device__ __forceinline__ void commit(float* tile) const {
        const int t = threadIdx.x;
        if (!KSTR) {
            const int c = t & 3, r0 = t >> 2;
#pragma unroll
            for (int p = 0; p < 2; p++) *reinterpret_cast<float4*>(tile + (r0 + 64 * p) * kPitch32 + c * 4) = r[p];
        } else {
            const int r4 = t & 31, kg = t >> 5;
            const float a[4] = {r[0].x, r[0].y, r[0].z, r[0].w};
            const float b[4] = {r[1].x, r[1].y, r[1].z, r[1].w};
#pragma unroll
            for (int e = 0; e < 4; e++)
                *reinterpret_cast<float2*>(tile + (4 * r4 + e) * kPitch32 + 2 * kg) = make_float2(a[e], b[e]);
        }
    }
};

template <bool A_KSTR, bool B_KSTR>
__global__ __launch_bounds__(kThreads) void gemm_mfma32_kernel(GemmArgs g) {
    __shared__ __attribute__((aligned(16))) float lds_a[2][BM * kPitch32];
    __shared__ __attribute__((aligned(16))) float lds_b[2][BN * kPitch32];
    long long batch;
    int tm, tn;
    tile_coords32(g, batch, tm, tn);
    const long long row0 = (long long)tm * BM, col0 = (long long)tn * BN;
    const float* a_base = static_cast<const float*>(g.a) + batch * g.sa;
    const float* b_base = static_cast<const float*>(g.b) + batch * g.sb;
    TileLoader32<A_KSTR> la;
    TileLoader32<B_KSTR> lb;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lrow = lane & 31, lk = (lane >> 5) * 4;

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    const long long nk = (g.k + BK32 - 1) / BK32;
    la.fetch(a_base, g.lda, row0, g.m, 0, g.k, g.vec_a);
    lb.fetch(b_base, g.ldb, col0, g.n, 0, g.k, g.vec_b);
    la.commit(lds_a[0]);
    lb.commit(lds_b[0]);
    __syncthreads();
    for (long long kt = 0; kt < nk; kt++) {
        const int cur = (int)(kt & 1);
        if (kt + 1 < nk) {
            la.fetch(a_base, g.lda, row0, g.m, (kt + 1) * BK32, g.k, g.vec_a);
            lb.fetch(b_base, g.ldb, col0, g.n, (kt + 1) * BK32, g.k, g.vec_b);
        }
        const float* ta = lds_a[cur] + (wm * 64 + lrow) * kPitch32 + lk;
        const float* tb = lds_b[cur] + (wn * 64 + lrow) * kPitch32 + lk;
#pragma unroll
        for (int ks = 0; ks < BK32 / 8; ks++) {
            // a lane holds k = ks*8 + (lane/32)*4 + s for s = 0..3; MFMA number s
            // multiplies slot s of both halves of the wave, i.e. two distinct k
            float4 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                fa[i] = *reinterpret_cast<const float4*>(ta + i * 32 * kPitch32 + ks * 8);
                fb[i] = *reinterpret_cast<const float4*>(tb + i * 32 * kPitch32 + ks * 8);
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].x, fb[j].x, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].y, fb[j].y, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].z, fb[j].z, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].w, fb[j].w, acc[i][j], 0, 0, 0);
                }
        }
        if (kt + 1 < nk) {
            la.commit(lds_a[cur ^ 1]);
            lb.commit(lds_b[cur ^ 1]);
        }
        __syncthreads();
    }
    float* c_base = static_cast<float*>(g.c) + batch * g.sc;
    const float* old_base = g.addend ? static_cast<const float*>(g.addend) + batch * g.sc : c_base;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const long long col = col0 + wn * 64 + j * 32 + lrow;
        if (col >= g.n) continue;
        const float bias = g.bias ? g.bias[batch * g.sbias + col] : 0.f;
#pragma unroll
        for (int i = 0; i < 2; i++) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const long long row = row0 + wm * 64 + i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
                if (row < g.m) {
                    float* p = c_base + row * g.ldc + col;
                    float o = g.alpha * acc[i][j][v] + bias;
                    if (g.accumulate) o += old_base[row * g.ldc + col];
                    *p = o;
                }
            }
        }
    }
}

long long elem_size(int dtype) { return dtype == BR_F32 ? 4 : 2; }

// The product of `rows` x `cols` elements of C from (row, col) on; multiples of 8, so that operands stay aligned.
GemmArgs part_of(GemmArgs g, const gemm16::Problem& p, long long row, long long col, long long rows, long long cols) {
    const long long at = elem_size(p.c_dtype) * (row * g.ldc + col);
    g.m = rows;
    g.n = cols;
    g.a = static_cast<const unsigned char*>(g.a) + 2 * (p.a_kstr ? row : row * g.lda);
    g.b = static_cast<const unsigned char*>(g.b) + 2 * (p.b_kstr ? col : col * g.ldb);
    g.c = static_cast<unsigned char*>(g.c) + at;
    if (g.c2) g.c2 = static_cast<unsigned char*>(g.c2) + at;
    if (g.addend) g.addend = static_cast<const unsigned char*>(g.addend) + at;
    if (g.bias) g.bias += col;
    return g;
}

// A 16-bit product by its plan, operands already checked by dtl_applies.  g.splits > 1: slices of K as batch entries.
int run_plan(GemmArgs g, const gemm16::Problem& p, const gemm16::Plan& plan, long long batch, int compute, hipStream_t st) {
    using namespace gemm16;
    const bool f16 = compute == BR_GEMM_F16;
    const KernelCost& tile = kCost[plan.kernel];
    if (!is_flex(plan.kernel) && g.ldc >= kEdgeColumns && (g.m % tile.bm != 0 || g.n % tile.bn != 0)) {
        // Partial large tiles of a C this wide are beyond their epilogue's offsets: whole tiles as planned, the columns
        // and the rows that are left on small tiles, which address C in 64 bits.
        const long long m_in = g.m / tile.bm * tile.bm, n_in = g.n / tile.bn * tile.bn;
        const Plan small{flex_kernel(g.m, g.n - n_in > 0 ? g.n - n_in : g.n, g.k, batch)};
        Plan whole = plan;
        whole.pair = false;
        whole.tail_from = 0;
        int rc = BR_OK;
        if (m_in > 0 && n_in > 0) rc = run_plan(part_of(g, p, 0, 0, m_in, n_in), p, whole, batch, compute, st);
        if (rc == BR_OK && n_in < g.n) rc = run_plan(part_of(g, p, 0, n_in, g.m, g.n - n_in), p, small, batch, compute, st);
        if (rc == BR_OK && m_in < g.m && n_in > 0) rc = run_plan(part_of(g, p, m_in, 0, g.m - m_in, n_in), p, small, batch, compute, st);
        return rc;
    }
    if (plan.pair && g.partials) {
        const int slot = split_slot_of(st);
        if (slot >= 0) return f16 ? gemm16_pair_f16(g, p, plan.kernel, slot, st) : gemm16_pair_bf16(g, p, plan.kernel, slot, st);
    }
    if (plan.tail_from > 0) {
        // whole rounds of 256x256 tiles, then the columns left over on 256x128 tiles (see column_tail)
        const GemmArgs head = part_of(g, p, 0, 0, g.m, plan.tail_from);
        const GemmArgs tail = part_of(g, p, 0, plan.tail_from, g.m, g.n - plan.tail_from);
        const int rc = f16 ? gemm16_tiles_f16(head, p, kTile256, 1, st) : gemm16_tiles_bf16(head, p, kTile256, 1, st);
        if (rc != BR_OK) return rc;
        return f16 ? gemm16_tiles_f16(tail, p, kTile256x128Groups, 1, st) : gemm16_tiles_bf16(tail, p, kTile256x128Groups, 1, st);
    }
    // a bias of its own for every batch entry: not on two groups of waves (see gemm_dtl16.hpp)
    const int kernel = plan.kernel == kTile256x128Groups && g.sbias != 0 && batch > 1 ? kTile256x128 : plan.kernel;
    // the loads have to be checked against the end of K: K, or a slice of it, is no whole number of steps
    const bool ragged = (g.k % 64 != 0 && kernel != kTile128Half) || g.splits > 1;
    if (ragged || is_flex(kernel))
        return f16 ? gemm16_ragged_f16(g, p, kernel, batch, st) : gemm16_ragged_bf16(g, p, kernel, batch, st);
    return f16 ? gemm16_tiles_f16(g, p, kernel, batch, st) : gemm16_tiles_bf16(g, p, kernel, batch, st);
}

// What products have beyond br_hip_gemm's arguments.
struct Extra {
    long long bias_stride = 0;          // between batch entries
    const float* addend = nullptr;      // with `sum`: sum = C + addend beside C (one batch entry, fp32)
    float* sum = nullptr;
    bool summed = false;                // out: the product's kernel has written `sum`
};

// br_hip_gemm with the tensor an accumulating product adds to named separately (null = c itself).  `planned`: what a
// caller with a workspace has planned (null: plan here, nothing split); `padded`: see gemm16::Problem.
int gemm_impl(int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha, const void* a, int a_dtype,
              int64_t lda, int64_t stride_a, const void* b, int b_dtype, int64_t ldb, int64_t stride_b, int accumulate,
              const void* addend, void* c, int c_dtype, int64_t ldc, int64_t stride_c, const float* bias, int64_t batch,
              int compute, br_stream_t stream, const gemm16::Plan* planned = nullptr, bool padded = false,
              float* partials = nullptr, size_t partial_bytes = 0, Extra* extra = nullptr) {
    if (m < 0 || n < 0 || k < 0 || batch < 0) return BR_ERR_ATTR;
    if (m == 0 || n == 0 || batch == 0) return BR_OK;
    if (!a || !b) return BR_ERR_INPUT;
    if (!c) return BR_ERR_OUTPUT;
    // minimal leading dimensions for the stated layouts
    if (lda < (trans_a ? m : k) || ldb < (trans_b ? k : n) || ldc < n) return BR_ERR_ATTR;
    const int native = compute == BR_GEMM_F16 ? BR_F16 : compute == BR_GEMM_BF16 ? BR_BF16 : BR_F32;
    if (compute != BR_GEMM_F16 && compute != BR_GEMM_BF16 && compute != BR_GEMM_F32) return BR_ERR_ATTR;
    if (a_dtype != BR_F32 && a_dtype != native) return BR_ERR_TODO;
    if (b_dtype != BR_F32 && b_dtype != native) return BR_ERR_TODO;
    if (c_dtype != BR_F32 && c_dtype != native) return BR_ERR_TODO;

    // A launch of 2^32 or more work items runs without those beyond, and without an error: so many batch entries go in
    // several launches, of as many as any kernel's tiles (of 32 x 32 elements or more, 512 threads or fewer) leave room for.
    const double tiles = (double)((m + 31) / 32) * (double)((n + 31) / 32);
    const int64_t fit = (int64_t)(4294967295.0 / 512.0 / tiles);
    if (batch > 1 && batch > fit && fit >= 1 && !(planned && planned->slices > 1)) {
        for (int64_t i = 0; i < batch; i += fit) {
            auto entry = [&](const void* x, int64_t stride, int dtype) {
                return static_cast<const char*>(x) + i * stride * elem_size(dtype);
            };
            const int rc = gemm_impl(trans_a, trans_b, m, n, k, alpha, entry(a, stride_a, a_dtype), a_dtype, lda, stride_a,
                                     entry(b, stride_b, b_dtype), b_dtype, ldb, stride_b, accumulate,
                                     addend ? entry(addend, stride_c, c_dtype) : nullptr,
                                     const_cast<char*>(entry(c, stride_c, c_dtype)), c_dtype, ldc, stride_c,
                                     bias && extra ? bias + i * extra->bias_stride : bias,
                                     batch - i < fit ? batch - i : fit, compute, stream, planned, padded, nullptr, 0, extra);
            if (rc != BR_OK) return rc;
        }
        return BR_OK;
    }

    GemmArgs g;
    g.a = a; g.b = b; g.c = c; g.bias = bias;
    g.m = m; g.n = n; g.k = k;
    g.lda = lda; g.ldb = ldb; g.ldc = ldc;
    g.sa = stride_a; g.sb = stride_b; g.sc = stride_c;
    g.alpha = alpha;
    g.accumulate = accumulate ? 1 : 0;
    g.addend = accumulate ? addend : nullptr;
    if (extra) g.sbias = extra->bias_stride;
    // taken by the small-tile kernels
    auto sum_beside = [&]() {
        if (!extra || !extra->sum || accumulate || batch != 1) return;
        g.addend = extra->addend;
        g.sum = extra->sum;
        extra->summed = true;
    };
    g.partials = partials;   // room for the partial tiles of a K split inside the kernel
    g.partial_bytes = partials ? partial_bytes : 0;
    g.tiles_m = (int)((m + BM - 1) / BM);
    g.tiles_n = (int)((n + BN - 1) / BN);
    const long long blocks = (long long)g.tiles_m * g.tiles_n * batch;
    if (blocks > 0x7fffffffLL) return BR_ERR_ATTR;
    // 128-bit loads need 16-byte aligned bases, leading dimensions and batch strides
    auto vec_ok = [&](const void* p, int dtype, long long ld, long long stride) {
        const long long es = elem_size(dtype);
        return aligned16(p) && (ld * es) % 16 == 0 && (batch == 1 || (stride * es) % 16 == 0);
    };
    g.vec_a = vec_ok(a, a_dtype, lda, stride_a) ? 1 : 0;
    g.vec_b = vec_ok(b, b_dtype, ldb, stride_b) ? 1 : 0;
    hipStream_t st = as_stream(stream);
    // opA is k-strided in memory when A is stored [k,m]; opB when B is stored [k,n]
    const bool ak = trans_a != 0, bk = trans_b == 0;
    gemm16::Problem p;
    p.a_f32 = a_dtype == BR_F32;
    p.b_f32 = b_dtype == BR_F32;
    p.a_kstr = ak;
    p.b_kstr = bk;
    p.c_dtype = c_dtype;
    p.padded = padded;
    if (compute == BR_GEMM_F32) {
        // the small-tile kernel's per-lane offsets span 64 rows in 32 bits
        const long long lim = 1LL << 31;
        const int kernel = gemm16::fp32_kernel(m, n, k, batch);
        if (kernel != gemm16::kTile128 && 256 * lda < lim && 256 * ldb < lim && m < lim && n < lim && k < lim && k > 0) {
            const bool words = !g.vec_a || !g.vec_b || (k % 4 != 0 && !(ak && bk));
            sum_beside();
            return gemm_fp32(g, p, kernel, words, batch, st);
        }
        if (ak && bk) gemm_mfma32_kernel<true, true><<<(unsigned)blocks, kThreads, 0, st>>>(g);
        else if (ak) gemm_mfma32_kernel<true, false><<<(unsigned)blocks, kThreads, 0, st>>>(g);
        else if (bk) gemm_mfma32_kernel<false, true><<<(unsigned)blocks, kThreads, 0, st>>>(g);
        else gemm_mfma32_kernel<false, false><<<(unsigned)blocks, kThreads, 0, st>>>(g);
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
    if (gemm16::dtl_applies(g, p)) {
        if (planned && planned->slices > 1) {
            // c holds one partial product per slice, `batch` of them
            const long long per = gemm16::slice_length(k, planned->slices);
            if (per * planned->slices == k) {
                // all alike: batch entries whose operands lie `per` k-values apart, on the kernels that check nothing
                // ([64 x 4096] from K = 12288 in slices 53 -> 30 us, [512 x 2048] from K = 8192 44 -> 33)
                g.k = per;
                g.sa = ak ? per * lda : per;
                g.sb = bk ? per * ldb : per;
            } else {
                g.splits = (int)batch;
                g.k_slice = (int)per;
            }
        }
        const gemm16::Plan plan = planned ? *planned : gemm16::gemm_plan(m, n, k, batch, false);
        // On two waves to a tile a second output costs more than a launch that adds, from some K on: K <= 768 0.84 to 0.97 of two
        // launches, 1024 0.93 to 1.03, 1536 to 3072 0.99 to 1.03 ([800 x 2560] from 1536 27.6 us in two, 28.4 in one).
        const bool two_launches = plan.kernel == gemm16::kFlex64Short && k > 1024;
        if (gemm16::is_flex(plan.kernel) && !two_launches && c_dtype == BR_F32) sum_beside();
        return run_plan(g, p, plan, batch, compute, st);
    }
    // the register-staged kernel; its fast form loads 128 bits at a time and never checks k
    const long long va = p.a_f32 ? 4 : 8, vb = p.b_f32 ? 4 : 8;
    p.guarded = !g.vec_a || !g.vec_b || k % 32 != 0 || (ak && m % va != 0) || (bk && n % vb != 0);
    return compute == BR_GEMM_F16 ? gemm16_registers_f16(g, p, batch, st) : gemm16_registers_bf16(g, p, batch, st);
}

}  // namespace

extern "C" int br_hip_gemm(int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha, const void* a,
                           int a_dtype, int64_t lda, int64_t stride_a, const void* b, int b_dtype, int64_t ldb,
                           int64_t stride_b, int accumulate, void* c, int c_dtype, int64_t ldc, int64_t stride_c,
                           const float* bias, int64_t batch, int compute, br_stream_t stream) {
    return gemm_impl(trans_a, trans_b, m, n, k, alpha, a, a_dtype, lda, stride_a, b, b_dtype, ldb, stride_b, accumulate,
                     nullptr, c, c_dtype, ldc, stride_c, bias, batch, compute, stream);
}

extern "C" int br_hip_gemm_kernel(int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, int c_dtype, int64_t batch,
                                  int staged, int* slices) {
    using namespace gemm16;
    // sizes alone decide
    (void)trans_a;
    (void)trans_b;
    (void)c_dtype;
    if (m <= 0 || n <= 0 || k <= 0 || batch <= 0) return BR_ERR_ATTR;
    if (!slices) return BR_ERR_OUTPUT;
    const Plan plan = gemm_plan(m, n, k, batch, staged != 0);
    *slices = plan.pair ? -2 : plan.slices;
    return plan.kernel;
}

extern "C" int br_hip_gemm_fp32_kernel(int64_t m, int64_t n, int64_t k, int64_t batch, int* waves) {
    if (m <= 0 || n <= 0 || k <= 0 || batch <= 0) return BR_ERR_ATTR;
    if (!waves) return BR_ERR_OUTPUT;
    const int kernel = gemm16::fp32_kernel(m, n, k, batch);
    *waves = gemm16::fp32_waves(kernel, m, n, k, batch);
    return kernel;
}

extern "C" int br_hip_linear_gelu(const void* x, const void* w, const float* bias, void* u, void* y, int dtype,
                                  int64_t rows, int64_t out, int64_t in, br_stream_t stream) {
    if (rows < 0 || out <= 0 || in <= 0) return BR_ERR_ATTR;
    if (dtype != BR_F16 && dtype != BR_BF16) return BR_ERR_TODO;
    if (rows == 0) return BR_OK;
    if (!x || !w) return BR_ERR_INPUT;
    if (!u || !y || u == y) return BR_ERR_OUTPUT;
    // the GELU epilogue exists in the direct-to-LDS kernels only
    if (in % 32 != 0 || out % 8 != 0 || !aligned16(x) || !aligned16(w) || !aligned16(u) || !aligned16(y))
        return BR_ERR_TODO;
    GemmArgs g;
    g.a = x; g.b = w; g.c = u; g.c2 = y; g.bias = bias;
    g.m = rows; g.n = out; g.k = in;
    g.lda = in; g.ldb = in; g.ldc = out;
    g.sa = g.sb = g.sc = 0;
    g.alpha = 1.0f;
    g.accumulate = 0;
    g.tiles_m = g.tiles_n = 0;  // set by the launcher for the tile it picks
    g.vec_a = g.vec_b = 1;
    gemm16::Problem p;
    p.a_f32 = p.b_f32 = false;
    p.a_kstr = p.b_kstr = false;
    p.c_dtype = dtype;
    p.guarded = false;
    if (!gemm16::dtl_applies(g, p)) return BR_ERR_TODO;
    return run_plan(g, p, gemm16::gemm_plan(rows, out, in, 1, false), 1, dtype == BR_F16 ? BR_GEMM_F16 : BR_GEMM_BF16,
                    as_stream(stream));
}

// ---- operands staged as dense, aligned 16-bit copies ------------------------
namespace {

// What is copied: dst[b][r][0 .. pitch) = convert(src[b*stride + r*ld + c]) for c < cols, zero from there to the pitch
// (a multiple of 8); fp32 values, or 16-bit ones whose rows do not start on 16-byte boundaries.
struct StageJob {
    const void* src;
    gemm16::u32x4* dst;
    long long ld, stride, total;   // total: 16-byte granules written
    unsigned rows, cols, granules; // granules: of a row
    bool f32, flat;                // flat: rows follow each other without gaps, fp32 and aligned
};
constexpr int kStageJobs = 4;
struct StageJobs {
    unsigned first[kStageJobs];   // the first workgroup of each operand
    int count;
    StageJob job[kStageJobs];
};

__device__ __forceinline__ gemm16::u32x4 pack16(const float (&v)[8], bool bf) {
    using namespace gemm16;
    if (bf)
        return mk4(pack2(Cvt<BR_GEMM_BF16>::from_f32(v[0]), Cvt<BR_GEMM_BF16>::from_f32(v[1])),
                   pack2(Cvt<BR_GEMM_BF16>::from_f32(v[2]), Cvt<BR_GEMM_BF16>::from_f32(v[3])),
                   pack2(Cvt<BR_GEMM_BF16>::from_f32(v[4]), Cvt<BR_GEMM_BF16>::from_f32(v[5])),
                   pack2(Cvt<BR_GEMM_BF16>::from_f32(v[6]), Cvt<BR_GEMM_BF16>::from_f32(v[7])));
    return mk4(pack2(Cvt<BR_GEMM_F16>::from_f32(v[0]), Cvt<BR_GEMM_F16>::from_f32(v[1])),
               pack2(Cvt<BR_GEMM_F16>::from_f32(v[2]), Cvt<BR_GEMM_F16>::from_f32(v[3])),
               pack2(Cvt<BR_GEMM_F16>::from_f32(v[4]), Cvt<BR_GEMM_F16>::from_f32(v[5])),
               pack2(Cvt<BR_GEMM_F16>::from_f32(v[6]), Cvt<BR_GEMM_F16>::from_f32(v[7])));
}

// One 16-byte granule per thread; the operands of a product (or of two) one after the other in one launch.  What it costs
// is bytes on large operands and the launch on small ones: [1024 x 2048] fp32 4-6 us, as does [64 x 256].  The operands
// of attention's backward products over 32 heads x 512 tokens, scores among them, one by one / at once (us):
// dO, P, V 5.3 + 11.2 + 6.2 / 13.5, dS, K, Q 10.5 + 5.2 + 5.4 / 12.
template <bool BF>
__global__ __launch_bounds__(256) void stage_kernel(StageJobs jobs) {
    // every line of the arguments is on its way before the first is looked at
    asm volatile("" ::"s"(jobs.count), "s"(jobs.job[0].src), "s"(jobs.job[1].src), "s"(jobs.job[2].src), "s"(jobs.job[3].src));
    int which = 0;
#pragma unroll
    for (int i = 1; i < kStageJobs; i++)
        if (i < jobs.count && blockIdx.x >= jobs.first[i]) which = i;
    which = __builtin_amdgcn_readfirstlane(which);
    const StageJob& job = jobs.job[which];
    const void* const src = job.src;
    gemm16::u32x4* const dst = job.dst;
    const long long total = job.total;
    const unsigned first = jobs.first[which];
    const bool f32 = job.f32, flat = job.flat;
    const long long i = (long long)(blockIdx.x - first) * 256 + threadIdx.x;
    if (i >= total) return;
    if (flat) {
        const float4 a = static_cast<const float4*>(src)[2 * i], b = static_cast<const float4*>(src)[2 * i + 1];
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        dst[i] = pack16(v, BF);
        return;
    }
    const unsigned rows = job.rows, cols = job.cols, granules = job.granules;
    const long long ld = job.ld, stride = job.stride;
    const unsigned c = (unsigned)(i % granules) * 8;
    const long long row = i / granules;
    const long long at = row / rows * stride + row % rows * ld + c;
    gemm16::u32x4 o;
    if (f32) {
        const float* s = static_cast<const float*>(src) + at;
        float v[8];
        if (c + 8 <= cols) {
            __builtin_memcpy(v, s, sizeof(v));
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = c + e < cols ? s[e] : 0.f;
        }
        o = pack16(v, BF);
    } else {   // bits are moved as they are
        const gemm16::u16* s = static_cast<const gemm16::u16*>(src) + at;
        if (c + 8 <= cols) {
            __builtin_memcpy(&o, s, sizeof(o));
        } else {
            gemm16::u16 h[8];
#pragma unroll
            for (int e = 0; e < 8; e++) h[e] = c + e < cols ? s[e] : (gemm16::u16)0;
            o = gemm16::mk4(gemm16::pack2(h[0], h[1]), gemm16::pack2(h[2], h[3]), gemm16::pack2(h[4], h[5]),
                            gemm16::pack2(h[6], h[7]));
        }
    }
    dst[i] = o;
}

// Row length of a staged copy of `cols` columns.
int64_t staged_pitch(int64_t cols) { return (cols + 7) & ~(int64_t)7; }

// Operands gathered for one launch.
struct Stager {
    StageJobs jobs;
    long long blocks = 0;
    int compute;
    hipStream_t st;
    Stager(int compute_, hipStream_t st_) : compute(compute_), st(st_) { jobs.count = 0; }
    int add(const void* src, bool f32, long long ld, long long stride, long long rows, long long cols, long long batch, void* dst) {
        const bool flat = f32 && ld == cols && cols % 8 == 0 && (batch == 1 || stride == rows * cols) && aligned16(src);
        const long long granules = staged_pitch(cols) / 8, total = batch * rows * granules;
        if (rows > 0xffffffffLL || cols > 0xfffffff0LL) return BR_ERR_ATTR;
        const long long need = (total + 255) / 256;
        // a launch holds less than 2^32 work items: what does not fit into this one starts another
        constexpr long long most = (1 << 24) - 1;
        if (need > most) {
            // so much in one operand goes in pieces of whole batch entries and rows
            const long long piece = most * 256 / granules;
            if (piece < 1) return BR_ERR_ATTR;
            for (long long b = 0; b < batch; b++)
                for (long long r = 0; r < rows; r += piece) {
                    const long long some = rows - r < piece ? rows - r : piece;
                    const char* from = static_cast<const char*>(src) + (b * stride + r * ld) * (f32 ? 4 : 2);
                    const int rc = add(from, f32, ld, some * ld, some, cols, 1, static_cast<char*>(dst) + (b * rows + r) * granules * 16);
                    if (rc != BR_OK) return rc;
                }
            return BR_OK;
        }
        if (jobs.count == kStageJobs || blocks + need > most) {
            const int rc = run();
            if (rc != BR_OK) return rc;
        }
        jobs.first[jobs.count] = (unsigned)blocks;
        jobs.job[jobs.count++] = StageJob{src, static_cast<gemm16::u32x4*>(dst), ld, stride, total, (unsigned)rows, (unsigned)cols,
                                          (unsigned)granules, f32, flat};
        blocks += need;
        return BR_OK;
    }
    int run() {
        if (jobs.count == 0) return BR_OK;
        if (compute == BR_GEMM_BF16) stage_kernel<true><<<(unsigned)blocks, 256, 0, st>>>(jobs);
        else stage_kernel<false><<<(unsigned)blocks, 256, 0, st>>>(jobs);
        jobs.count = 0;
        blocks = 0;
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
};

// ---- split-K ------------------------------------------------------------------
// A product with few output tiles and a long K leaves most CUs idle.  Two forms,
// both deterministic and free of floating-point atomics; gemm_plan chooses:
//  * slices of K as batch entries, each leaving an fp32 partial product in the
//    workspace, followed by a fixed-order sum in a second kernel;
//  * two slices inside the direct-to-LDS kernel, the slice that finishes last
//    adds the other's partial tile and runs the epilogue (gemm_dtl16.hpp).
//    Measured on the same box, this form loses to the first when four or more
//    slices exchange partial tiles (its device-coherent accesses move 1.5-3
//    TB/s, ordinary stores 6-7) and wins with two, where only one of the two
//    slices writes anything.
//
// The sum of the slices.  It reads what the product has just written, mostly from the caches, so what it takes is the
// latency of its loads: with S slices, the numbers that plans come to, all of them are in flight at once beside whatever
// else an element needs (S = 0: any number, four at a time); rows are found by a 32-bit division, and C is written 16 (8)
// bytes at a time where its rows start on such an address (VEC).  One load after the other, a 64-bit division and single
// stores: four slices of [1002 x 2048] 13.3 us with a bias and a residual, 10.2 without; now 9.9 and 8.0.
template <typename T, int S, bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float4* __restrict__ part, int splits, unsigned mn4,
                                                            unsigned n4, float alpha, const float* bias, const T* old, T* c,
                                                            long long ldc, const float* addend, float* sum) {
    using gemm16::c_load;
    using gemm16::c_store;
    using gemm16::c_store4;
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i >= mn4) return;
    const unsigned r = i / n4, col = (i - r * n4) * 4;
    const long long at = (long long)r * ldc + col;
    float4 v[S ? S : 4];
    if (S) {
#pragma unroll
        for (int p = 0; p < S; p++) v[p] = part[(long long)p * mn4 + i];
    }
    float b[4] = {0.f, 0.f, 0.f, 0.f}, was[4], more[4];
    auto read4 = [&](const auto* p, float (&to)[4]) {
        using E = std::remove_cv_t<std::remove_pointer_t<decltype(p)>>;
        if constexpr (VEC && sizeof(E) == 4) {
            const float4 q = *reinterpret_cast<const float4*>(p);
            to[0] = q.x; to[1] = q.y; to[2] = q.z; to[3] = q.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) to[j] = c_load<E>(p + j);
        }
    };
    if (bias) {
#pragma unroll
        for (int j = 0; j < 4; j++) b[j] = bias[col + j];
    }
    if (old) read4(old + at, was);
    if (sizeof(T) == 4 && sum) read4(addend + at, more);
    float4 s;
    if (S) {
        s = v[0];
#pragma unroll
        for (int p = 1; p < S; p++) { s.x += v[p].x; s.y += v[p].y; s.z += v[p].z; s.w += v[p].w; }
    } else {
        s = part[i];
        int p = 1;
        for (; p + 4 <= splits; p += 4) {
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = part[(long long)(p + q) * mn4 + i];
#pragma unroll
            for (int q = 0; q < 4; q++) { s.x += v[q].x; s.y += v[q].y; s.z += v[q].z; s.w += v[q].w; }
        }
        for (; p < splits; p++) {
            const float4 q = part[(long long)p * mn4 + i];
            s.x += q.x; s.y += q.y; s.z += q.z; s.w += q.w;
        }
    }
    float o[4] = {__fmul_rn(alpha, s.x), __fmul_rn(alpha, s.y), __fmul_rn(alpha, s.z), __fmul_rn(alpha, s.w)};
    if (bias) {
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] += b[j];
    }
    float w[4];
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = old ? o[j] + was[j] : o[j];
    if (VEC) {
        c_store4<T>(c + at, w);
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) c_store<T>(c + at + j, w[j]);
    }
    if constexpr (sizeof(T) == 4) {
        if (sum) {   // c plus the addend, beside c
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] += more[j];
            if (VEC) {
                c_store4<float>(sum + at, o);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) sum[at + j] = o[j];
            }
        }
    }
}

template <typename T>
int splitk_reduce(const float* part, int splits, long long m, long long n, float alpha, const float* bias, const void* old, void* c,
                  long long ldc, const float* addend, float* sum, hipStream_t st) {
    const long long mn4 = m * n / 4;
    const unsigned grid = (unsigned)((mn4 + 255) / 256);
    auto lies = [&](const void* p) { return (reinterpret_cast<uintptr_t>(p) & (4 * sizeof(T) - 1)) == 0; };
    const bool vec = ldc % 4 == 0 && lies(c) && lies(old) && (sizeof(T) != 4 || (lies(addend) && lies(sum)));
#define BR_REDUCE(S)                                                                                                             \
    if (vec) splitk_reduce_kernel<T, S, true><<<grid, 256, 0, st>>>(reinterpret_cast<const float4*>(part), splits, (unsigned)mn4,   \
                 (unsigned)(n / 4), alpha, bias, static_cast<const T*>(old), static_cast<T*>(c), ldc, addend, sum);                 \
    else splitk_reduce_kernel<T, S, false><<<grid, 256, 0, st>>>(reinterpret_cast<const float4*>(part), splits, (unsigned)mn4,      \
                 (unsigned)(n / 4), alpha, bias, static_cast<const T*>(old), static_cast<T*>(c), ldc, addend, sum)
    switch (splits) {
        case 2: BR_REDUCE(2); break;
        case 4: BR_REDUCE(4); break;
        case 8: BR_REDUCE(8); break;
        default: BR_REDUCE(0);
    }
#undef BR_REDUCE
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

size_t staged_bytes(int64_t rows, int64_t cols, int64_t batch) {
    const size_t b = (size_t)rows * (size_t)staged_pitch(cols) * (size_t)batch * 2;
    return (b + 255) & ~(size_t)255;
}

// Whether an operand is copied before the product, dense as it is: fp32 operands are converted, 16-bit ones whose rows
// do not start on 16-byte boundaries are moved to rows that do.
bool wants_staging(int dtype, int64_t cols) { return dtype == BR_F32 || cols % 8 != 0; }

// Room for the partial sums of a product whose K is cut.
size_t sums_bytes(int64_t m, int64_t n, int64_t k, int64_t batch) {
    const gemm16::Plan plan = gemm16::gemm_plan(m, n, k, batch, true);
    return (plan.slices > 1 ? (size_t)plan.slices * (size_t)m * (size_t)n * sizeof(float) : 0) + gemm16::pair_bytes(plan, m, n);
}

}  // namespace

extern "C" size_t br_hip_gemm_staged_workspace(int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, int a_dtype,
                                               int b_dtype, int64_t batch) {
    if (m <= 0 || n <= 0 || k <= 0 || batch <= 0) return 0;
    size_t need = 0;
    if (wants_staging(a_dtype, trans_a ? m : k)) need += staged_bytes(trans_a ? k : m, trans_a ? m : k, batch);
    if (wants_staging(b_dtype, trans_b ? k : n)) need += staged_bytes(trans_b ? n : k, trans_b ? k : n, batch);
    return need + sums_bytes(m, n, k, batch);
}

namespace {
// br_hip_gemm_staged with the tensor an accumulating product adds to named separately (null = c itself).  zero_filled: the
// operands are in the products' type already, their rows aligned and zero-filled to whole granules.
int staged_impl(int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha, const void* a, int a_dtype,
                int64_t lda, int64_t stride_a, const void* b, int b_dtype, int64_t ldb, int64_t stride_b, int accumulate,
                const void* addend, void* c, int c_dtype, int64_t ldc, int64_t stride_c, const float* bias,
                int64_t batch, int compute, void* workspace, size_t workspace_bytes, br_stream_t stream,
                bool zero_filled = false, Extra* extra = nullptr) {
    const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
    const bool sixteen = compute == BR_GEMM_F16 || compute == BR_GEMM_BF16;
    const int64_t a_rows = trans_a ? k : m, a_cols = trans_a ? m : k;
    const int64_t b_rows = trans_b ? n : k, b_cols = trans_b ? k : n;
    // Stage (and consider splitting K) only with the workspace that was asked for; every other case is the plain
    // entry point's business.
    const bool stage = sixteen && workspace && aligned16(workspace) && m > 0 && n > 0 && k > 0 && batch > 0 && a && b &&
                       c && lda >= a_cols && ldb >= b_cols && ldc >= n &&
                       (a_dtype == BR_F32 || a_dtype == native) && (b_dtype == BR_F32 || b_dtype == native) &&
                       (c_dtype == BR_F32 || c_dtype == native) &&
                       (zero_filled ? sums_bytes(m, n, k, batch)
                                    : br_hip_gemm_staged_workspace(trans_a, trans_b, m, n, k, a_dtype, b_dtype, batch)) <=
                           workspace_bytes;
    if (!stage)
        return gemm_impl(trans_a, trans_b, m, n, k, alpha, a, a_dtype, lda, stride_a, b, b_dtype, ldb, stride_b,
                         accumulate, addend, c, c_dtype, ldc, stride_c, bias, batch, compute, stream, nullptr, false, nullptr, 0,
                         extra);
    hipStream_t st = as_stream(stream);
    char* ws = static_cast<char*>(workspace);
    // 16-bit rows that start on 16-byte boundaries all the same (their pitch is padded) are taken where they are, unless
    // they run along K and end inside a granule, whose rest would have to be zero
    auto in_place = [&](const void* x, int dtype, bool along_k, int64_t ld, int64_t stride) {
        return dtype != BR_F32 && !along_k && aligned16(x) && ld % 8 == 0 && (batch == 1 || stride % 8 == 0);
    };
    // every row of a staged copy is zero-filled up to its pitch
    Stager stager(compute, st);
    if (wants_staging(a_dtype, a_cols) && !zero_filled && !in_place(a, a_dtype, !trans_a, lda, stride_a)) {
        const int64_t copies = stride_a == 0 ? 1 : batch;   // one A for every batch entry
        const int rc = stager.add(a, a_dtype == BR_F32, lda, stride_a, a_rows, a_cols, copies, ws);
        if (rc != BR_OK) return rc;
        a = ws;
        a_dtype = native;
        lda = staged_pitch(a_cols);
        stride_a = stride_a == 0 ? 0 : a_rows * lda;
        ws += staged_bytes(a_rows, a_cols, copies);
    }
    if (wants_staging(b_dtype, b_cols) && !zero_filled && !in_place(b, b_dtype, trans_b, ldb, stride_b)) {
        const int rc = stager.add(b, b_dtype == BR_F32, ldb, stride_b, b_rows, b_cols, batch, ws);
        if (rc != BR_OK) return rc;
        b = ws;
        b_dtype = native;
        ldb = staged_pitch(b_cols);
        stride_b = b_rows * ldb;
        ws += staged_bytes(b_rows, b_cols, batch);
    }
    const int staged = stager.run();
    if (staged != BR_OK) return staged;
    const gemm16::Plan plan = gemm16::gemm_plan(m, n, k, batch, true);
    // only the direct-to-LDS kernels know slices: the register-staged one would sum all of K once per slice
    const bool sliceable = aligned16(a) && aligned16(b) && lda % 8 == 0 && ldb % 8 == 0 && m * n / 4 <= 0x7fffffffLL &&
                           gemm16::dtl_spans(trans_a != 0, lda, trans_b == 0, ldb, n, m, n, k);
    if (plan.slices > 1 && sliceable) {
        float* part = reinterpret_cast<float*>(ws);
        const int rc = gemm_impl(trans_a, trans_b, m, n, k, 1.0f, a, a_dtype, lda, 0, b, b_dtype, ldb, 0, 0, nullptr,
                                 part, BR_F32, n, m * n, nullptr, plan.slices, compute, stream, &plan, true);
        if (rc != BR_OK) return rc;
        const bool summing = extra && extra->sum && !accumulate && c_dtype == BR_F32;
        const void* const old = accumulate ? (addend ? addend : c) : nullptr;
        const int sum_rc =
            c_dtype == BR_F32 ? splitk_reduce<float>(part, plan.slices, m, n, alpha, bias, old, c, ldc, summing ? extra->addend : nullptr,
                                                     summing ? extra->sum : nullptr, as_stream(stream))
            : c_dtype == BR_F16 ? splitk_reduce<__half>(part, plan.slices, m, n, alpha, bias, old, c, ldc, nullptr, nullptr, as_stream(stream))
                                : splitk_reduce<__hip_bfloat16>(part, plan.slices, m, n, alpha, bias, old, c, ldc, nullptr, nullptr,
                                                                as_stream(stream));
        if (summing) extra->summed = true;
        return sum_rc;
    }
    // two slices inside the kernel: what is left of the workspace holds one partial tile per output tile
    float* partials = plan.pair ? reinterpret_cast<float*>(ws) : nullptr;
    return gemm_impl(trans_a, trans_b, m, n, k, alpha, a, a_dtype, lda, stride_a, b, b_dtype, ldb, stride_b, accumulate,
                     addend, c, c_dtype, ldc, stride_c, bias, batch, compute, stream, plan.slices > 1 ? nullptr : &plan,
                     true, partials, gemm16::pair_bytes(plan, m, n), extra);
}
}  // namespace

extern "C" int br_hip_gemm_staged(int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha, const void* a,
                                  int a_dtype, int64_t lda, int64_t stride_a, const void* b, int b_dtype, int64_t ldb,
                                  int64_t stride_b, int accumulate, void* c, int c_dtype, int64_t ldc,
                                  int64_t stride_c, const float* bias, int64_t batch, int compute, void* workspace,
                                  size_t workspace_bytes, br_stream_t stream) {
    return staged_impl(trans_a, trans_b, m, n, k, alpha, a, a_dtype, lda, stride_a, b, b_dtype, ldb, stride_b,
                       accumulate, nullptr, c, c_dtype, ldc, stride_c, bias, batch, compute, workspace, workspace_bytes,
                       stream);
}

extern "C" int br_hip_linear_residual(const void* x, int x_dtype, const void* w, int w_dtype, const float* bias,
                                      const void* r, void* y, int y_dtype, int64_t rows, int64_t out, int64_t in,
                                      int compute, void* workspace, size_t workspace_bytes, br_stream_t stream) {
    if (rows < 0 || out <= 0 || in <= 0) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!x || !w || !r) return BR_ERR_INPUT;
    if (!y) return BR_ERR_OUTPUT;
    return staged_impl(0, 1, rows, out, in, 1.0f, x, x_dtype, in, 0, w, w_dtype, in, 0, 1, r, y, y_dtype, out, 0, bias, 1,
                       compute, workspace, workspace_bytes, stream);
}

// ---- two products in one launch -------------------------------------------------
namespace {

// A stored operand: rows x cols of a batch entry, rows `ld` apart, entries `stride`.
struct Stored {
    const void* at;
    int dtype;
    int64_t rows, cols, ld, stride, batch;
    bool along_k;   // rows run along K
};
Stored stored_a(const br_product& p) {
    return {p.a, p.a_dtype, p.trans_a ? p.k : p.m, p.trans_a ? p.m : p.k, p.lda, p.stride_a, p.batch, p.trans_a == 0};
}
Stored stored_b(const br_product& p) {
    return {p.b, p.b_dtype, p.trans_b ? p.n : p.k, p.trans_b ? p.k : p.n, p.ldb, p.stride_b, p.batch, p.trans_b != 0};
}
Stored stored_c(const br_product& p) { return {p.c, p.c_dtype, p.m, p.n, p.ldc, p.stride_c, p.batch, false}; }

bool same_memory(const Stored& x, const Stored& y) {
    return x.at == y.at && x.dtype == y.dtype && x.rows == y.rows && x.cols == y.cols && x.ld == y.ld &&
           (x.batch == 1 || x.stride == y.stride) && x.batch == y.batch;
}

bool overlap(const Stored& x, const Stored& y) {
    auto bytes = [](const Stored& s) { return (uintptr_t)((s.batch - 1) * s.stride + (s.rows - 1) * s.ld + s.cols) * elem_size(s.dtype); };
    const uintptr_t x0 = reinterpret_cast<uintptr_t>(x.at), y0 = reinterpret_cast<uintptr_t>(y.at);
    return x0 < y0 + bytes(y) && y0 < x0 + bytes(x);
}

size_t staged_size(const Stored& s) { return wants_staging(s.dtype, s.cols) ? staged_bytes(s.rows, s.cols, s.batch) : 0; }

bool sizes_ok(const br_product& p) {
    return p.m > 0 && p.n > 0 && p.k > 0 && p.batch > 0 && p.a && p.b && p.c && p.lda >= (p.trans_a ? p.m : p.k) &&
           p.ldb >= (p.trans_b ? p.k : p.n) && p.ldc >= p.n && (p.batch == 1 || (p.stride_a >= 0 && p.stride_b >= 0 && p.stride_c >= 0));
}

// What two products read, with the operands that have to be copied first in `copies`: one that both read is copied once.
struct PairOperands {
    Stored before[4], now[4];   // a and b of the first, a and b of the second
    int copy_of[4] = {-1, -1, -1, -1};
    size_t bytes = 0;           // of all copies
    PairOperands(const br_product& first, const br_product& second, int compute, char* ws)
        : before{stored_a(first), stored_b(first), stored_a(second), stored_b(second)}, now{before[0], before[1], before[2], before[3]} {
        if (compute == BR_GEMM_F32) return;
        for (int i = 0; i < 4; i++) {
            const Stored& s = before[i];
            // as in staged_impl
            const bool in_place = s.dtype != BR_F32 && !s.along_k && aligned16(s.at) && s.ld % 8 == 0 && (s.batch == 1 || s.stride % 8 == 0);
            if (!wants_staging(s.dtype, s.cols) || in_place) continue;
            copy_of[i] = i;
            for (int j = 0; j < i; j++)
                if (copy_of[j] == j && same_memory(s, before[j])) copy_of[i] = j;
            if (copy_of[i] == i) {
                now[i].at = ws + bytes;
                bytes += staged_bytes(s.rows, s.cols, s.batch);
            } else {
                now[i].at = now[copy_of[i]].at;
            }
            now[i].dtype = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            now[i].ld = staged_pitch(s.cols);
            now[i].stride = s.rows * now[i].ld;
        }
    }
    int run(int compute, hipStream_t st) const {
        Stager stager(compute, st);
        for (int i = 0; i < 4; i++) {
            if (copy_of[i] != i) continue;
            const Stored& s = before[i];
            const int rc = stager.add(s.at, s.dtype == BR_F32, s.ld, s.stride, s.rows, s.cols, s.batch, const_cast<void*>(now[i].at));
            if (rc != BR_OK) return rc;
        }
        return stager.run();
    }
};

// Both products (and the sums) as one launch.
struct PairLaunch {
    int kernel, w, x;   // w: the product with both operands row-contiguous
    gemm16::GemmArgs g[2];
    gemm16::Problem p[2];
    gemm16::ColumnSums cs;
    gemm16::PartialSums ps;
};
// BR_ERR_TODO where they have to run one after the other.
int plan_pair(const br_product& first, const br_product& second, const PairOperands& ops, const br_column_sums* sums,
              const br_partial_sums* later, int compute, PairLaunch& launch) {
    using namespace gemm16;
    const bool fp32 = compute == BR_GEMM_F32;
    const int native = compute == BR_GEMM_F16 ? BR_F16 : fp32 ? BR_F32 : BR_BF16;
    // the one with both operands row-contiguous
    auto wide = [](const br_product& p) { return p.trans_a && !p.trans_b && p.c_dtype == BR_F32; };
    const int w = wide(first) ? 0 : 1, x = 1 - w;
    if (!wide(w ? second : first) || (w ? first : second).trans_a) return BR_ERR_TODO;
    const br_product* const products[2] = {&first, &second};
    auto sizes = [&](int i) { return PairSizes{products[i]->m, products[i]->n, products[i]->k, products[i]->batch}; };
    const int kernel = pair_kernel(sizes(w), sizes(x), fp32);
    if (kernel < 0) return BR_ERR_TODO;
    const Stored out[2] = {stored_c(first), stored_c(second)};
    if (out[x].dtype != native && out[x].dtype != BR_F32) return BR_ERR_TODO;
    // nothing is written that another part reads or writes (what is copied first is read ahead of all writes)
    if (overlap(out[0], out[1]) || overlap(out[1], ops.now[0]) || overlap(out[1], ops.now[1])) return BR_ERR_TODO;
    ColumnSums& cs = launch.cs;
    if (sums) {
        const Stored sx{sums->x, sums->dtype, sums->rows, sums->cols, sums->cols, 0, 1, false};
        const Stored so{sums->out, BR_F32, 1, sums->cols, sums->cols, 0, 1, false};
        const long long vec = fp32 ? 4 : 8;
        if (!sums->x || !sums->out || sums->dtype != native || sums->rows <= 0 || sums->cols <= 0 || sums->cols % vec != 0 ||
            sums->rows > 0x3fffffffLL || sums->cols > 0x3fffffffLL || !aligned16(sums->x))
            return BR_ERR_TODO;
        for (const Stored& s : ops.before)
            if (overlap(so, s)) return BR_ERR_TODO;
        for (const Stored& s : out)
            if (overlap(so, s) || overlap(sx, s)) return BR_ERR_TODO;
        cs.x = sums->x;
        cs.out = sums->out;
        cs.rows = (int)sums->rows;
        cs.cols = (int)sums->cols;
        cs.scale = sums->scale;
    }
    PartialSums& ps = launch.ps;
    if (later && later->partials) {
        if (later->arrays < 1 || later->arrays > 3 || later->parts <= 0 || later->parts > 0x3fffffffLL || later->cols <= 0 ||
            later->cols % 4 != 0 || later->cols > 0x3fffffffLL || !aligned16(later->partials))
            return BR_ERR_TODO;
        const Stored sp{later->partials, BR_F32, later->arrays * later->parts, later->cols, later->cols, 0, 1, false};
        for (int i = 0; i < later->arrays; i++) {
            if (!later->out[i] || !aligned16(later->out[i])) return BR_ERR_TODO;
            const Stored so{later->out[i], BR_F32, 1, later->cols, later->cols, 0, 1, false};
            if (overlap(so, sp)) return BR_ERR_TODO;
            for (int j = 0; j < i; j++)
                if (overlap(so, Stored{later->out[j], BR_F32, 1, later->cols, later->cols, 0, 1, false})) return BR_ERR_TODO;
            // the column sums come behind these, and read what they have written
            if (sums) {
                const Stored sx{sums->x, sums->dtype, sums->rows, sums->cols, sums->cols, 0, 1, false};
                const Stored ss{sums->out, BR_F32, 1, sums->cols, sums->cols, 0, 1, false};
                if (overlap(so, ss) || overlap(so, sx) || overlap(ss, sp)) return BR_ERR_TODO;
            }
            // so do the products, also what they read by way of a copy made ahead of everything
            for (int j = 0; j < 4; j++)
                if (overlap(so, ops.now[j]) || overlap(so, ops.before[j])) return BR_ERR_TODO;
            for (const Stored& s : out)
                if (overlap(so, s) || overlap(sp, s)) return BR_ERR_TODO;
            ps.out[i] = reinterpret_cast<flex_f32x4*>(later->out[i]);
        }
        ps.partials = reinterpret_cast<const flex_f32x4*>(later->partials);
        ps.arrays = later->arrays;
        ps.parts = (int)later->parts;
        ps.cols4 = (int)(later->cols / 4);
        ps.scale = later->scale;
    }
    GemmArgs(&g)[2] = launch.g;
    Problem(&p)[2] = launch.p;
    for (int i = 0; i < 2; i++) {
        const Stored &a = ops.now[2 * i], &b = ops.now[2 * i + 1];
        const br_product& d = *products[i];
        GemmArgs& q = g[i];
        q.a = a.at; q.b = b.at; q.c = d.c; q.bias = nullptr;
        q.m = d.m; q.n = d.n; q.k = d.k;
        q.lda = a.ld; q.ldb = b.ld; q.ldc = d.ldc;
        q.sa = a.stride; q.sb = b.stride; q.sc = d.stride_c;
        q.alpha = d.alpha;
        q.accumulate = 0;
        q.tiles_m = q.tiles_n = 0;   // set by the launcher
        auto aligned = [&](const Stored& s) {
            const long long es = elem_size(s.dtype);
            return aligned16(s.at) && s.ld * es % 16 == 0 && (s.batch == 1 || s.stride * es % 16 == 0);
        };
        q.vec_a = aligned(a);
        q.vec_b = aligned(b);
        p[i].a_f32 = a.dtype == BR_F32;
        p[i].b_f32 = b.dtype == BR_F32;
        p[i].a_kstr = d.trans_a != 0;
        p[i].b_kstr = d.trans_b == 0;
        p[i].c_dtype = d.c_dtype;
        p[i].guarded = false;
        p[i].padded = true;
        if (fp32) {
            const long long lim = 1LL << 31;
            if (256 * q.lda >= lim || 256 * q.ldb >= lim || q.m >= lim || q.n >= lim || q.k >= lim || !q.vec_a || !q.vec_b ||
                (q.k % 4 != 0 && !(p[i].a_kstr && p[i].b_kstr)))
                return BR_ERR_TODO;
        } else if (!dtl_applies(q, p[i])) {
            return BR_ERR_TODO;
        }
    }
    launch.kernel = kernel;
    launch.w = w;
    launch.x = x;
    return BR_OK;
}

bool pair_types_ok(const br_product& p, int compute) {
    const int native = compute == BR_GEMM_F16 ? BR_F16 : compute == BR_GEMM_BF16 ? BR_BF16 : BR_F32;
    return (p.a_dtype == BR_F32 || p.a_dtype == native) && (p.b_dtype == BR_F32 || p.b_dtype == native) &&
           (p.c_dtype == BR_F32 || p.c_dtype == native);
}
// Whether their operands may be copied ahead of both products: there is room, and the first does not write what the
// second's copies are made of.
bool copies_ahead(const br_product& first, const PairOperands& ops, const void* workspace, size_t workspace_bytes) {
    return (ops.bytes == 0 || (workspace && aligned16(workspace) && ops.bytes <= workspace_bytes)) &&
           !overlap(stored_c(first), ops.before[2]) && !overlap(stored_c(first), ops.before[3]);
}

}  // namespace

extern "C" size_t br_hip_gemm_pair_workspace(const br_product* first, const br_product* second, int compute) {
    if (!first || !second || compute == BR_GEMM_F32) return 0;
    size_t copies = 0, sums = 0, most = 0;
    for (const br_product* p : {first, second}) {
        if (p->m <= 0 || p->n <= 0 || p->k <= 0 || p->batch <= 0) continue;
        copies += staged_size(stored_a(*p)) + staged_size(stored_b(*p));
        const size_t partial = sums_bytes(p->m, p->n, p->k, p->batch);
        const size_t one = br_hip_gemm_staged_workspace(p->trans_a, p->trans_b, p->m, p->n, p->k, p->a_dtype, p->b_dtype, p->batch);
        if (partial > sums) sums = partial;
        if (one > most) most = one;
    }
    return copies + sums > most ? copies + sums : most;
}

extern "C" int br_hip_gemm_pair_kernel(int64_t m1, int64_t n1, int64_t k1, int64_t batch1, int64_t m2, int64_t n2, int64_t k2,
                                       int64_t batch2, int compute) {
    if (m1 <= 0 || n1 <= 0 || k1 <= 0 || batch1 <= 0 || m2 <= 0 || n2 <= 0 || k2 <= 0 || batch2 <= 0) return BR_ERR_ATTR;
    return gemm16::pair_kernel({m1, n1, k1, batch1}, {m2, n2, k2, batch2}, compute == BR_GEMM_F32);
}

extern "C" int br_hip_gemm_pair_joined(const br_product* first, const br_product* second, const br_column_sums* sums,
                                       const br_partial_sums* later, int compute, const void* workspace, size_t workspace_bytes) {
    if (!first || !second) return BR_ERR_INPUT;
    if (compute != BR_GEMM_F16 && compute != BR_GEMM_BF16 && compute != BR_GEMM_F32) return BR_ERR_ATTR;
    if (!sizes_ok(*first) || !sizes_ok(*second) || !pair_types_ok(*first, compute) || !pair_types_ok(*second, compute)) return -1;
    const PairOperands ops(*first, *second, compute, static_cast<char*>(const_cast<void*>(workspace)));
    PairLaunch launch;
    if (!copies_ahead(*first, ops, workspace, workspace_bytes) || plan_pair(*first, *second, ops, sums, later, compute, launch) != BR_OK)
        return -1;
    return launch.kernel;
}

extern "C" int br_hip_gemm_pair(const br_product* first, const br_product* second, const br_column_sums* sums,
                                const br_partial_sums* later, int compute, void* workspace, size_t workspace_bytes,
                                br_stream_t stream) {
    if (!first || !second) return BR_ERR_INPUT;
    if (compute != BR_GEMM_F16 && compute != BR_GEMM_BF16 && compute != BR_GEMM_F32) return BR_ERR_ATTR;
    hipStream_t st = as_stream(stream);
    auto before_them = [&]() {
        const int rl = later ? br_hip_finish_sums(later, stream) : (int)BR_OK;
        if (!sums || rl != BR_OK) return rl;
        return br_hip_colsum(sums->x, sums->dtype, sums->out, sums->rows, sums->cols, sums->scale, sums->workspace,
                             sums->workspace_bytes, stream);
    };
    if (sizes_ok(*first) && sizes_ok(*second) && pair_types_ok(*first, compute) && pair_types_ok(*second, compute)) {
        char* ws = static_cast<char*>(workspace);
        const PairOperands ops(*first, *second, compute, ws);
        if (copies_ahead(*first, ops, workspace, workspace_bytes)) {
            PairLaunch l;
            int rc = plan_pair(*first, *second, ops, sums, later, compute, l);
            if (rc == BR_OK) rc = ops.run(compute, st);
            if (rc == BR_OK) {
                auto* const launch = compute == BR_GEMM_F32 ? gemm_pair_f32 : compute == BR_GEMM_F16 ? gemm_pair_f16 : gemm_pair_bf16;
                const br_product* const products[2] = {first, second};
                rc = launch(l.g[l.w], l.p[l.w], products[l.w]->batch, l.g[l.x], l.p[l.x], products[l.x]->batch, l.kernel, l.cs, l.ps, st);
            }
            if (rc != BR_ERR_TODO) return rc;
            if (ops.bytes > 0 && workspace_bytes >= ops.bytes) {
                // one after the other, on copies made in one launch
                const int rs = before_them();
                if (rs != BR_OK) return rs;
                const int rt = ops.run(compute, st);
                if (rt != BR_OK) return rt;
                const size_t left = workspace_bytes - ops.bytes;
                for (int i = 0; i < 2; i++) {
                    const br_product& p = i ? *second : *first;
                    const Stored &a = ops.now[2 * i], &b = ops.now[2 * i + 1];
                    const int rp = staged_impl(p.trans_a, p.trans_b, p.m, p.n, p.k, p.alpha, a.at, a.dtype, a.ld, a.stride, b.at,
                                               b.dtype, b.ld, b.stride, 0, nullptr, p.c, p.c_dtype, p.ldc, p.stride_c, nullptr,
                                               p.batch, compute, ws + ops.bytes, left, stream, true);
                    if (rp != BR_OK) return rp;
                }
                return BR_OK;
            }
        }
    }
    const int rs = before_them();
    if (rs != BR_OK) return rs;
    for (const br_product* p : {first, second}) {
        const int rp = compute == BR_GEMM_F32
            ? gemm_impl(p->trans_a, p->trans_b, p->m, p->n, p->k, p->alpha, p->a, p->a_dtype, p->lda, p->stride_a, p->b, p->b_dtype,
                        p->ldb, p->stride_b, 0, nullptr, p->c, p->c_dtype, p->ldc, p->stride_c, nullptr, p->batch, compute, stream)
            : staged_impl(p->trans_a, p->trans_b, p->m, p->n, p->k, p->alpha, p->a, p->a_dtype, p->lda, p->stride_a, p->b, p->b_dtype,
                          p->ldb, p->stride_b, 0, nullptr, p->c, p->c_dtype, p->ldc, p->stride_c, nullptr, p->batch, compute,
                          workspace, workspace_bytes, stream);
        if (rp != BR_OK) return rp;
    }
    return BR_OK;
}

// ---- linear layers of the operator stream ----------------------------------------
extern "C" size_t br_hip_linear_group_workspace(int count, int64_t rows, int64_t out, int64_t in, int x_dtype, int w_dtype) {
    if (count <= 0 || rows <= 0 || out <= 0 || in <= 0) return 0;
    return br_hip_gemm_staged_workspace(0, 1, rows, out, in, x_dtype, w_dtype, count);
}

extern "C" int br_hip_linear_group(const void* x, int x_dtype, const void* w, int w_dtype, const float* bias, void* y, int y_dtype,
                                   int count, int64_t rows, int64_t out, int64_t in, int compute, void* workspace,
                                   size_t workspace_bytes, br_stream_t stream) {
    if (count < 0 || rows < 0 || out <= 0 || in <= 0) return BR_ERR_ATTR;
    if (rows == 0 || count == 0) return BR_OK;
    if (!x || !w) return BR_ERR_INPUT;
    if (!y) return BR_ERR_OUTPUT;
    Extra extra;
    extra.bias_stride = out;
    return staged_impl(0, 1, rows, out, in, 1.0f, x, x_dtype, in, 0, w, w_dtype, in, out * in, 0, nullptr, y, y_dtype, out, rows * out, bias,
                       count, compute, workspace, workspace_bytes, stream, false, &extra);
}

extern "C" int br_hip_linear_sum(const void* x, int x_dtype, const void* w, int w_dtype, const float* bias, const float* r,
                                 float* y, float* sum, int64_t rows, int64_t out, int64_t in, int compute, void* workspace,
                                 size_t workspace_bytes, br_stream_t stream) {
    if (rows < 0 || out <= 0 || in <= 0) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!x || !w || !r) return BR_ERR_INPUT;
    if (!y || !sum || y == sum || y == r) return BR_ERR_OUTPUT;
    Extra extra;
    extra.addend = r;
    extra.sum = sum;
    const int rc = staged_impl(0, 1, rows, out, in, 1.0f, x, x_dtype, in, 0, w, w_dtype, in, 0, 0, nullptr, y, BR_F32, out, 0,
                               bias, 1, compute, workspace, workspace_bytes, stream, false, &extra);
    if (rc != BR_OK || extra.summed) return rc;
    const int64_t shape[4] = {1, rows, 1, out};
    return br_hip_add_bcast(y, r, sum, BR_F32, shape, shape, stream);
}
