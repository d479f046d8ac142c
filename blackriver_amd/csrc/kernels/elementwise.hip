// Memory-bound elementwise kernels for gfx950: fill, cast, broadcast add,
// (bias-)GELU forward / backward, transpose 0213, column sums and the
// data-preparation tables.  All of them move 128 bits per lane per access and
// are launched as grid-stride loops over a few thousand workgroups.
#include "common.hpp"

#include <type_traits>

#include <float.h>
#include <hip/hip_bf16.h>

using namespace brk;

namespace {

constexpr int kBlock = 256;

// ------------------------------------------------------------------ fill
template <typename T>
__global__ __launch_bounds__(kBlock) void fill_kernel(T* dst, T value, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) dst[i] = value;
}

// ------------------------------------------------------------------ cast
template <typename T>
__device__ __forceinline__ float to_f32(T v);
template <>
__device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ float to_f32<__half>(__half v) { return __half2float(v); }
template <>
__device__ __forceinline__ float to_f32<__hip_bfloat16>(__hip_bfloat16 v) { return __bfloat162float(v); }

template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ __half from_f32<__half>(float v) { return __float2half_rn(v); }
template <>
__device__ __forceinline__ __hip_bfloat16 from_f32<__hip_bfloat16>(float v) { return __float2bfloat16(v); }

template <typename S, typename D>
__global__ __launch_bounds__(kBlock) void cast_kernel(const S* src, D* dst, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * kBlock * 4;
    for (int64_t i = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4; i < n; i += stride) {
        if (i + 3 < n) {
            S s[4];
#pragma unroll
            for (int j = 0; j < 4; j++) s[j] = src[i + j];
#pragma unroll
            for (int j = 0; j < 4; j++) dst[i + j] = from_f32<D>(to_f32<S>(s[j]));
        } else {
            for (int64_t j = i; j < n; j++) dst[j] = from_f32<D>(to_f32<S>(src[j]));
        }
    }
}

// 8 elements per thread through 128-bit accesses (n % 8 == 0, 16-byte aligned).
template <typename S, typename D>
__global__ __launch_bounds__(kBlock) void cast_x8_kernel(const S* __restrict__ src, D* __restrict__ dst, int64_t n8) {
    struct alignas(16) SV { S v[8]; };
    struct alignas(16) DV { D v[8]; };
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += stride) {
        float f[8];
        if constexpr (sizeof(S) == 4) {
            const float4 a = load_stream(reinterpret_cast<const float4*>(src) + 2 * i),
                         b = load_stream(reinterpret_cast<const float4*>(src) + 2 * i + 1);
            f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
        } else {
            const uint4 raw = load_stream(reinterpret_cast<const uint4*>(src) + i);
            const unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const unsigned short lo = (unsigned short)(w[j] & 0xffffu), hi = (unsigned short)(w[j] >> 16);
                f[2 * j] = to_f32<S>(__builtin_bit_cast(S, lo));
                f[2 * j + 1] = to_f32<S>(__builtin_bit_cast(S, hi));
            }
        }
        if constexpr (sizeof(D) == 4) {
            reinterpret_cast<float4*>(dst)[2 * i] = make_float4(f[0], f[1], f[2], f[3]);
            reinterpret_cast<float4*>(dst)[2 * i + 1] = make_float4(f[4], f[5], f[6], f[7]);
        } else {
            unsigned w[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const unsigned lo = __builtin_bit_cast(unsigned short, from_f32<D>(f[2 * j]));
                const unsigned hi = __builtin_bit_cast(unsigned short, from_f32<D>(f[2 * j + 1]));
                w[j] = lo | (hi << 16);
            }
            reinterpret_cast<uint4*>(dst)[i] = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

// Same type on both sides: a copy, one 16-byte granule per thread (the form that measured fastest: 5.3-5.6 TB/s at
// 2 x 34 MB, 6.0-6.5 TB/s from 2 x 134 MB up; two granules per thread as in cast_x8_kernel: 4.6 / 5.1-5.5).
__global__ __launch_bounds__(kBlock) void copy_x16_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, int64_t n16) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n16; i += stride)
        store_stream(dst + i, load_stream(src + i));
}

template <typename S, typename D>
void cast_launch(const void* src, void* dst, int64_t n, hipStream_t st) {
    if (std::is_same<S, D>::value && (n * (int64_t)sizeof(S)) % 16 == 0 && aligned16(src) && aligned16(dst)) {
        const int64_t n16 = n * (int64_t)sizeof(S) / 16;
        copy_x16_kernel<<<grid_for(n16, kBlock), kBlock, 0, st>>>((const uint4*)src, (uint4*)dst, n16);
        return;
    }
    if (n % 8 == 0 && aligned16(src) && aligned16(dst))
        cast_x8_kernel<S, D><<<grid_for(n / 8, kBlock), kBlock, 0, st>>>((const S*)src, (D*)dst, n / 8);
    else
        cast_kernel<S, D><<<grid_for((n + 3) / 4, kBlock), kBlock, 0, st>>>((const S*)src, (D*)dst, n);
}

template <typename S>
int cast_from(const void* src, void* dst, int dst_dtype, int64_t n, hipStream_t st) {
    switch (dst_dtype) {
        case BR_F32: cast_launch<S, float>(src, dst, n, st); break;
        case BR_F16: cast_launch<S, __half>(src, dst, n, st); break;
        case BR_BF16: cast_launch<S, __hip_bfloat16>(src, dst, n, st); break;
        default: return BR_ERR_TODO;
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// --------------------------------------------------------- broadcast add
// Same-shape fast path: 128-bit loads, no index arithmetic.
__global__ __launch_bounds__(kBlock) void add_same_f32x4(const float4* a, const float4* b, float4* c,
                                                          int64_t n4) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n4; i += stride) {
        float4 x = a[i], y = b[i];
        c[i] = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
    }
}

__global__ __launch_bounds__(kBlock) void add_same_f16x8(const half8* a, const half8* b, half8* c,
                                                          int64_t n8) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += stride) {
        half8 x = a[i], y = b[i], z;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            // add in fp32 and round once, like a + b on fp16 values
            float2 fx = __half22float2(x.v[j]), fy = __half22float2(y.v[j]);
            z.v[j] = __floats2half2_rn(fx.x + fy.x, fx.y + fy.y);
        }
        c[i] = z;
    }
}

struct BcastDims {
    unsigned s1, s2, s3v;      // a's dims 1,2 and dim 3 in vectors
    long long bst0, bst1, bst2;  // b's element strides (0 where broadcast)
    int bst3;                    // 0 when b's last dim is broadcast, else 1
};

// General path over vectors of 4 fp32 along the last dimension.
__global__ __launch_bounds__(kBlock) void add_bcast_f32x4(const float* a, const float* b, float* c,
                                                           long long nvec, BcastDims d) {
    const long long stride = (long long)gridDim.x * kBlock;
    for (long long v = (long long)blockIdx.x * kBlock + threadIdx.x; v < nvec; v += stride) {
        unsigned long long r = (unsigned long long)v;
        const unsigned i3v = (unsigned)(r % d.s3v);
        r /= d.s3v;
        const unsigned i2 = (unsigned)(r % d.s2);
        r /= d.s2;
        const unsigned i1 = (unsigned)(r % d.s1);
        const unsigned long long i0 = r / d.s1;
        const float4 x = reinterpret_cast<const float4*>(a)[v];
        const float* bp = b + i0 * d.bst0 + i1 * d.bst1 + i2 * d.bst2;
        float4 y;
        if (d.bst3) {
            y = *reinterpret_cast<const float4*>(bp + (long long)i3v * 4);
        } else {
            const float s = bp[0];
            y = make_float4(s, s, s, s);
        }
        reinterpret_cast<float4*>(c)[v] = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
    }
}

// Fallback for shapes / pointers that do not allow 128-bit accesses.
template <typename T>
__global__ __launch_bounds__(kBlock) void add_bcast_scalar(const T* a, const T* b, T* c, long long n,
                                                            unsigned s1, unsigned s2, unsigned s3,
                                                            long long bst0, long long bst1,
                                                            long long bst2, int bst3) {
    const long long stride = (long long)gridDim.x * kBlock;
    for (long long v = (long long)blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
        unsigned long long r = (unsigned long long)v;
        const unsigned i3 = (unsigned)(r % s3);
        r /= s3;
        const unsigned i2 = (unsigned)(r % s2);
        r /= s2;
        const unsigned i1 = (unsigned)(r % s1);
        const unsigned long long i0 = r / s1;
        const T y = b[i0 * bst0 + i1 * bst1 + i2 * bst2 + (long long)i3 * bst3];
        c[v] = from_f32<T>(to_f32<T>(a[v]) + to_f32<T>(y));
    }
}

// ------------------------------------------------------------------ GELU
// d/dv gelu(v) = s + 2 v s (1 - s) u',  s = sigmoid(2u),
//   u = 0.79788456 v (1 + 0.044715 v^2),  u' = 0.79788456 + 0.1070322243 v^2
// evaluated from e = exp(-2|u|) = 2^(-|w|), w = 2*log2(e)*u, in (0,1] so that s
// and s(1-s) keep full relative accuracy for large |v|.
__device__ __forceinline__ float gelu_grad_one(float v) {
    const float v2 = v * v;
    const float w = v * (kLog2e2 * 0.79788456f + (kLog2e2 * 0.79788456f * 0.044715f) * v2);
    const float e = __builtin_amdgcn_exp2f(-fabsf(w));
    const float inv = __builtin_amdgcn_rcpf(1.0f + e);
    const float ei = e * inv;
    const float s = w >= 0.f ? inv : ei;
    return s + v * (ei * inv) * (2.0f * 0.79788456f + (2.0f * 0.1070322243f) * v2);
}

__global__ __launch_bounds__(kBlock) void gelu_fwd_f32(const float* x, float* y, int64_t n4) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n4; i += stride) {
        const float4 v = reinterpret_cast<const float4*>(x)[i];
        reinterpret_cast<float4*>(y)[i] =
            make_float4(gelu_one(v.x), gelu_one(v.y), gelu_one(v.z), gelu_one(v.w));
    }
}

__global__ __launch_bounds__(kBlock) void gelu_fwd_f16(const half8* x, half8* y, int64_t n8) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += stride) {
        float f[8];
        unpack8(x[i], f);
#pragma unroll
        for (int j = 0; j < 8; j++) f[j] = gelu_one(f[j]);
        y[i] = pack8(f);
    }
}

// fp32 in, 16-bit out: the output of the 4h activation when it only feeds the
// next product (rounded once, exactly as that product would round an fp32 copy);
// y32: written as fp32 too ([1024 x 8192] 11 us, and 8.6 for the product's own
// copy of it otherwise)
template <typename D>
__global__ __launch_bounds__(kBlock) void gelu_fwd_f32_to_16(const float4* x, uint4* y, int64_t n8, float4* y32 = nullptr) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += stride) {
        const float4 a = x[2 * i], b = x[2 * i + 1];
        float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        unsigned w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float lo = gelu_one(f[2 * j]), hi = gelu_one(f[2 * j + 1]);
            // the fp32 results are rounded to fp32 first, then to the 16-bit type
            asm volatile("" : "+v"(lo), "+v"(hi));
            w[j] = (unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(lo)) |
                   ((unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(hi)) << 16);
            f[2 * j] = lo;
            f[2 * j + 1] = hi;
        }
        if (y32) {
            y32[2 * i] = make_float4(f[0], f[1], f[2], f[3]);
            y32[2 * i + 1] = make_float4(f[4], f[5], f[6], f[7]);
        }
        y[i] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

__global__ __launch_bounds__(kBlock) void gelu_bwd_f32(const float* dy, const float* x, float* dx,
                                                        int64_t n4) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n4; i += stride) {
        const float4 v = reinterpret_cast<const float4*>(x)[i];
        const float4 g = reinterpret_cast<const float4*>(dy)[i];
        reinterpret_cast<float4*>(dx)[i] =
            make_float4(g.x * gelu_grad_one(v.x), g.y * gelu_grad_one(v.y),
                        g.z * gelu_grad_one(v.z), g.w * gelu_grad_one(v.w));
    }
}

__global__ __launch_bounds__(kBlock) void gelu_bwd_f16(const half8* dy, const half8* x, half8* dx,
                                                        int64_t n8) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n8; i += stride) {
        float v[8], g[8];
        unpack8(x[i], v);
        unpack8(dy[i], g);
#pragma unroll
        for (int j = 0; j < 8; j++) g[j] *= gelu_grad_one(v[j]);
        dx[i] = pack8(g);
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void gelu_scalar(const T* dy, const T* x, const float* bias, T* out,
                                                       int64_t n, int64_t cols, bool backward) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        float v = to_f32<T>(x[i]);
        if (bias) v += bias[i % cols];
        out[i] = from_f32<T>(backward ? to_f32<T>(dy[i]) * gelu_grad_one(v) : gelu_one(v));
    }
}

// Bias-GELU backward over a strip of rows.  A workgroup owns kBlock*VEC
// columns and `rows_per_block` rows; each thread keeps VEC running column
// sums of dx in registers and writes them to partial[blockIdx.y][col].
template <typename T, int VEC>
struct VecIO;
template <>
struct VecIO<float, 4> {
    static __device__ __forceinline__ void load(const float* p, float (&f)[4]) {
        const float4 v = load_stream(reinterpret_cast<const float4*>(p));
        f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w;
    }
    static __device__ __forceinline__ void store(float* p, const float (&f)[4]) {
        store_stream(reinterpret_cast<float4*>(p), make_float4(f[0], f[1], f[2], f[3]));
    }
    // store, and leave in f exactly the values that were stored
    static __device__ __forceinline__ void store_rounded(float* p, float (&f)[4]) { store(p, f); }
};
template <>
struct VecIO<__half, 8> {
    static __device__ __forceinline__ void load(const __half* p, float (&f)[8]) {
        unpack8(load_stream(reinterpret_cast<const half8*>(p)), f);
    }
    static __device__ __forceinline__ void store(__half* p, const float (&f)[8]) {
        store_stream(reinterpret_cast<half8*>(p), pack8(f));
    }
    // The compiler is free to fuse the producing multiply into the fp16
    // conversion (v_fma_mixlo_f16: one rounding) for one use and not for
    // another (v_mul_f32 + v_cvt: two roundings), which differ on rare inputs.
    // The empty asm makes the packed registers opaque, so the store and the
    // read-back see the very same bits.
    static __device__ __forceinline__ void store_rounded(__half* p, float (&f)[8]) {
        uint4 u = __builtin_bit_cast(uint4, pack8(f));
        asm volatile("" : "+v"(u.x), "+v"(u.y), "+v"(u.z), "+v"(u.w));
        const half8 h = __builtin_bit_cast(half8, u);
        store_stream(reinterpret_cast<half8*>(p), h);
        unpack8(h, f);
    }
};

template <>
struct VecIO<__hip_bfloat16, 8> {
    static __device__ __forceinline__ void load(const __hip_bfloat16* p, float (&f)[8]) {
        unpack(load_stream(reinterpret_cast<const uint4*>(p)), f);
    }
    static __device__ __forceinline__ void unpack(const uint4& u, float (&f)[8]) {
        const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            f[2 * i] = __builtin_bit_cast(float, w[i] << 16);
            f[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ uint4 pack(const float (&f)[8]) {
        unsigned w[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            w[i] = (unsigned)__builtin_bit_cast(unsigned short, __float2bfloat16(f[2 * i])) |
                   ((unsigned)__builtin_bit_cast(unsigned short, __float2bfloat16(f[2 * i + 1])) << 16);
        return make_uint4(w[0], w[1], w[2], w[3]);
    }
    static __device__ __forceinline__ void store(__hip_bfloat16* p, const float (&f)[8]) {
        store_stream(reinterpret_cast<uint4*>(p), pack(f));
    }
    static __device__ __forceinline__ void store_rounded(__hip_bfloat16* p, float (&f)[8]) {
        uint4 u = pack(f);
        asm volatile("" : "+v"(u.x), "+v"(u.y), "+v"(u.z), "+v"(u.w));
        store_stream(reinterpret_cast<uint4*>(p), u);
        unpack(u, f);
    }
};

// The rows of one strip of a strip kernel (grid y = strips).  Strip s takes rows s, s + S, s + 2S, ... (S strips): all
// workgroups of the launch then read one window of S consecutive rows at a time and the launch sweeps memory front
// to back (see grid_for), instead of S windows a strip apart (bias-GELU backward at [2048,16384]: 43.0 -> 41.6 us).
// A strip's rows are summed in this order, whatever the kernel.
#ifndef BR_STRIPS_INTERLEAVED
#define BR_STRIPS_INTERLEAVED 1
#endif
struct StripWalk {
    int64_t first, end, step;
};
__device__ __forceinline__ StripWalk strip_walk(int64_t rows, int rows_per_block) {
    if (BR_STRIPS_INTERLEAVED) return StripWalk{(int64_t)blockIdx.y, rows, (int64_t)gridDim.y};
    const int64_t r0 = (int64_t)blockIdx.y * rows_per_block;
    return StripWalk{r0, r0 + rows_per_block < rows ? r0 + rows_per_block : rows, 1};
}

// Bias-GELU forward with the same tiling: the VEC bias values of a thread's
// columns stay in registers while it walks down its strip of rows.
template <typename T, int VEC>
__global__ __launch_bounds__(kBlock) void bias_gelu_fwd_kernel(const T* x, const float* bias, T* y,
                                                                int64_t rows, int64_t cols,
                                                                int rows_per_block) {
    const int64_t col = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * VEC;
    if (col >= cols) return;
    float b[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) b[j] = bias[col + j];
    const int64_t r0 = (int64_t)blockIdx.y * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < rows ? r0 + rows_per_block : rows;
    // four rows of loads in flight per thread
    int64_t r = r0;
    for (; r + 4 <= r1; r += 4) {
        float v[4][VEC];
#pragma unroll
        for (int u = 0; u < 4; u++) VecIO<T, VEC>::load(x + (r + u) * cols + col, v[u]);
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int j = 0; j < VEC; j++) v[u][j] = gelu_one(v[u][j] + b[j]);
            VecIO<T, VEC>::store(y + (r + u) * cols + col, v[u]);
        }
    }
    for (; r < r1; r++) {
        float v[VEC];
        VecIO<T, VEC>::load(x + r * cols + col, v);
#pragma unroll
        for (int j = 0; j < VEC; j++) v[j] = gelu_one(v[j] + b[j]);
        VecIO<T, VEC>::store(y + r * cols + col, v);
    }
}

template <typename T, int VEC>
__global__ __launch_bounds__(kBlock) void bias_gelu_bwd_kernel(const T* dy, const T* x, const float* bias,
                                                                T* dx, float* partial, int64_t rows,
                                                                int64_t cols, int rows_per_block) {
    const int64_t col = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * VEC;
    if (col >= cols) return;
    float b[VEC], acc[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) {
        b[j] = bias ? bias[col + j] : 0.f;
        acc[j] = 0.f;
    }
    const StripWalk w = strip_walk(rows, rows_per_block);
    const int64_t step = w.step, r1 = w.end;
    // four rows (eight loads) in flight per thread; a strip's rows are still summed in order
    int64_t r = w.first;
    for (; r + 3 * step < r1; r += 4 * step) {
        float v[4][VEC], g[4][VEC];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            VecIO<T, VEC>::load(x + (r + u * step) * cols + col, v[u]);
            VecIO<T, VEC>::load(dy + (r + u * step) * cols + col, g[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int j = 0; j < VEC; j++) g[u][j] *= gelu_grad_one(v[u][j] + b[j]);
            // sum what was stored, i.e. after rounding to the storage type
            VecIO<T, VEC>::store_rounded(dx + (r + u * step) * cols + col, g[u]);
#pragma unroll
            for (int j = 0; j < VEC; j++) acc[j] += g[u][j];
        }
    }
    for (; r < r1; r += step) {
        float v[VEC], g[VEC];
        VecIO<T, VEC>::load(x + r * cols + col, v);
        VecIO<T, VEC>::load(dy + r * cols + col, g);
#pragma unroll
        for (int j = 0; j < VEC; j++) g[j] *= gelu_grad_one(v[j] + b[j]);
        VecIO<T, VEC>::store_rounded(dx + r * cols + col, g);
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[j] += g[j];
    }
    if (partial) {
#pragma unroll
        for (int j = 0; j < VEC; j++) partial[(int64_t)blockIdx.y * cols + col + j] = acc[j];
    }
}

// --------------------------------------------------------------- colsum
// Stage 1: partial[g][c] = sum over the g-th strip of rows of x[r,c].
template <typename T>
__global__ __launch_bounds__(kBlock) void colsum_partial(const T* x, float* partial, int64_t rows,
                                                          int64_t cols, int rows_per_block) {
    const int64_t col = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (col >= cols) return;
    const int64_t r0 = (int64_t)blockIdx.y * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < rows ? r0 + rows_per_block : rows;
    float acc = 0.f;
    for (int64_t r = r0; r < r1; r++) acc += to_f32<T>(x[r * cols + col]);
    partial[(int64_t)blockIdx.y * cols + col] = acc;
}

// Stage 2: out[c] = sum_g partial[g][c]  (fixed order: deterministic).
__global__ __launch_bounds__(kBlock) void colsum_final(const float* partial, float* out, int groups,
                                                        int64_t cols, float scale) {
    const int64_t col = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (col >= cols) return;
    float acc = 0.f;
    for (int g = 0; g < groups; g++) acc += partial[(int64_t)g * cols + col];
    out[col] = acc * scale;
}

// Vector forms of the two stages (cols % VEC == 0, 16-byte aligned rows).
// Stage 1: a thread owns VEC adjacent columns and sums a strip of rows, four
// rows of loads in flight at a time.
template <typename T, int VEC>
__global__ __launch_bounds__(kBlock) void colsum_partial_vec(const T* __restrict__ x, float* __restrict__ partial,
                                                              int64_t rows, int64_t cols, int rows_per_block) {
    const int64_t col = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * VEC;
    if (col >= cols) return;
    const StripWalk w = strip_walk(rows, rows_per_block);
    const int64_t step = w.step, r1 = w.end;
    float acc[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) acc[j] = 0.f;
    int64_t r = w.first;
    for (; r + 3 * step < r1; r += 4 * step) {
        float v[4][VEC];
#pragma unroll
        for (int u = 0; u < 4; u++) VecIO<T, VEC>::load(x + (r + u * step) * cols + col, v[u]);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int j = 0; j < VEC; j++) acc[j] += v[u][j];
    }
    for (; r < r1; r += step) {
        float v[VEC];
        VecIO<T, VEC>::load(x + r * cols + col, v);
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[j] += v[j];
    }
#pragma unroll
    for (int j = 0; j < VEC; j++) partial[(int64_t)blockIdx.y * cols + col + j] = acc[j];
}

// Stage 1 for fp32 x that is also wanted as a 16-bit copy (the gradient of a
// linear layer: its column sums are the bias gradient, its 16-bit copy is the
// operand of the two products that follow): one pass over x does both.
template <typename D>
__global__ __launch_bounds__(kBlock) void colsum_cast_partial(const float* __restrict__ x, float* __restrict__ partial,
                                                               D* __restrict__ x16, int64_t rows, int64_t cols,
                                                               int rows_per_block) {
    const int64_t col = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4;
    if (col >= cols) return;
    const StripWalk w = strip_walk(rows, rows_per_block);
    const int64_t step = w.step, r1 = w.end;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    auto emit = [&](int64_t r, const float (&v)[4]) {
        const unsigned lo = (unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[0])) |
                            ((unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[1])) << 16);
        const unsigned hi = (unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[2])) |
                            ((unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[3])) << 16);
        *reinterpret_cast<uint2*>(x16 + r * cols + col) = make_uint2(lo, hi);
    };
    int64_t r = w.first;
    for (; r + 3 * step < r1; r += 4 * step) {
        float v[4][4];
#pragma unroll
        for (int u = 0; u < 4; u++) VecIO<float, 4>::load(x + (r + u * step) * cols + col, v[u]);
#pragma unroll
        for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] += v[u][j];
            emit(r + u * step, v[u]);
        }
    }
    for (; r < r1; r += step) {
        float v[4];
        VecIO<float, 4>::load(x + r * cols + col, v);
#pragma unroll
        for (int j = 0; j < 4; j++) acc[j] += v[j];
        emit(r, v);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) partial[(int64_t)blockIdx.y * cols + col + j] = acc[j];
}

// The same pass with x produced on the fly: x = dy * gelu'(u), the GELU
// backward whose result is the gradient of the linear layer below it.  Writes
// the fp32 gradient (dx may be u's or dy's own buffer), its 16-bit copy and
// the column-sum partials; dx is rounded to fp32 before it is summed and
// converted, so all three equal what the separate kernels produce.
template <typename D>
__global__ __launch_bounds__(kBlock) void gelu_bwd_colsum_cast_partial(const float* dy, const float* u, float* dx,
                                                                        float* __restrict__ partial,
                                                                        D* __restrict__ dx16, int64_t rows,
                                                                        int64_t cols, int rows_per_block) {
    const int64_t col = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4;
    if (col >= cols) return;
    const StripWalk w = strip_walk(rows, rows_per_block);
    const int64_t step = w.step, r1 = w.end;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    auto emit = [&](int64_t r, const float (&g)[4], const float (&x)[4]) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v[j] = g[j] * gelu_grad_one(x[j]);
            asm volatile("" : "+v"(v[j]));
            acc[j] += v[j];
        }
        VecIO<float, 4>::store(dx + r * cols + col, v);
        const unsigned lo = (unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[0])) |
                            ((unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[1])) << 16);
        const unsigned hi = (unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[2])) |
                            ((unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[3])) << 16);
        *reinterpret_cast<uint2*>(dx16 + r * cols + col) = make_uint2(lo, hi);
    };
    int64_t r = w.first;
    for (; r + step < r1; r += 2 * step) {
        float g[2][4], x[2][4];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            VecIO<float, 4>::load(dy + (r + k * step) * cols + col, g[k]);
            VecIO<float, 4>::load(u + (r + k * step) * cols + col, x[k]);
        }
#pragma unroll
        for (int k = 0; k < 2; k++) emit(r + k * step, g[k], x[k]);
    }
    for (; r < r1; r += step) {
        float g[4], x[4];
        VecIO<float, 4>::load(dy + r * cols + col, g);
        VecIO<float, 4>::load(u + r * cols + col, x);
        emit(r, g, x);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) partial[(int64_t)blockIdx.y * cols + col + j] = acc[j];
}

// Stage 2 for cols % 4 == 0: 1024 threads = 16 column quads x 64 slices of
// groups, every load of a workgroup in flight at once; slices are combined in
// LDS in a fixed order.
__global__ __launch_bounds__(1024) void colsum_final_x4(const float4* __restrict__ partial, float4* __restrict__ out,
                                                        int groups, int cols4, float scale) {
    __shared__ float4 l[64][16];
    const int q = threadIdx.x & 15, sl = threadIdx.x >> 4;
    const int c4 = blockIdx.x * 16 + q;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (c4 < cols4) {
#pragma unroll 4
        for (int g = sl; g < groups; g += 64) {
            const float4 a = partial[(int64_t)g * cols4 + c4];
            s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
        }
    }
    l[sl][q] = s;
    __syncthreads();
    if (sl < 8) {
        for (int k = sl + 8; k < 64; k += 8) {
            const float4 a = l[k][q];
            s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
        }
        l[sl][q] = s;
    }
    __syncthreads();
    if (sl == 0 && c4 < cols4) {
        for (int k = 1; k < 8; k++) {
            const float4 a = l[k][q];
            s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
        }
        out[c4] = make_float4(s.x * scale, s.y * scale, s.z * scale, s.w * scale);
    }
}

// Launches stage 2 in its vector form when the shapes allow.
int colsum_finish(const float* partial, float* out, int groups, int64_t cols, float scale, hipStream_t st) {
    if (cols % 4 == 0 && aligned16(partial) && aligned16(out))
        colsum_final_x4<<<(unsigned)((cols / 4 + 15) / 16), 1024, 0, st>>>(reinterpret_cast<const float4*>(partial),
                                                                            reinterpret_cast<float4*>(out), groups,
                                                                            (int)(cols / 4), scale);
    else
        colsum_final<<<(unsigned)((cols + kBlock - 1) / kBlock), kBlock, 0, st>>>(partial, out, groups, cols, scale);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// Row strips of the vector column sum: about 1024 workgroups in all, at most
// 256 strips.
constexpr int kMaxColsumGroups = 256;
int colsum_vec_rows_per_block(int64_t rows, int64_t blocks_x) {
    int64_t groups = 1024 / (blocks_x < 1 ? 1 : blocks_x);
    if (groups < 1) groups = 1;
    if (groups > kMaxColsumGroups) groups = kMaxColsumGroups;
    int64_t rpb = (rows + groups - 1) / groups;
    if (rpb < 4) rpb = 4;
    return (int)rpb;
}

// ------------------------------------------------ column sums in one launch
// A workgroup of 1024 threads owns LPR * VEC columns (LPR = 8: 128 bytes of a row) and walks ALL rows: LPR lanes per
// row, 1024 / LPR rows per pass, UNROLL passes in flight.  No partial sums leave the workgroup and there is no second
// launch; the row slots of a wave are combined by lane exchanges, the waves in LDS, in a fixed order, so the result
// depends on the shape alone.  What bounds it on few rows is latency -- launch, one pass of loads, the combination --
// and on wide ones the CU's load rate; fewer lanes per row make more, shorter workgroups (owner_lanes has the
// measurements).  What is summed, and what else is written on the way, is the Source's business:
//   load(at, in)      the loads of one row position (all of a pass's loads are issued before any is used)
//   finish(at, in)    leaves the values to be summed in in[0]; may store
template <typename T, int V>
struct OwnPlain {
    const T* x;
    static constexpr int VEC = V, NIN = 1;
    __device__ __forceinline__ void init(int64_t) {}
    __device__ __forceinline__ void load(int64_t at, float (&in)[NIN][VEC]) const { VecIO<T, V>::load(x + at, in[0]); }
    __device__ __forceinline__ void finish(int64_t, float (&)[NIN][VEC]) const {}
};
template <typename D>
__device__ __forceinline__ void store4_as16(D* p, const float (&v)[4]) {
    const unsigned lo = (unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[0])) |
                        ((unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[1])) << 16);
    const unsigned hi = (unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[2])) |
                        ((unsigned)__builtin_bit_cast(unsigned short, from_f32<D>(v[3])) << 16);
    *reinterpret_cast<uint2*>(p) = make_uint2(lo, hi);
}
// fp32 x, summed as it is, with its 16-bit copy written (colsum_cast_partial)
template <typename D>
struct OwnCast {
    const float* x;
    D* x16;
    static constexpr int VEC = 4, NIN = 1;
    __device__ __forceinline__ void init(int64_t) {}
    __device__ __forceinline__ void load(int64_t at, float (&in)[NIN][VEC]) const { VecIO<float, 4>::load(x + at, in[0]); }
    __device__ __forceinline__ void finish(int64_t at, float (&in)[NIN][VEC]) const { store4_as16<D>(x16 + at, in[0]); }
};
// dx = dy * gelu'(u) in fp32, written as fp32 and as a 16-bit copy, summed (gelu_bwd_colsum_cast_partial)
template <typename D>
struct OwnGeluBwdCast {
    const float* dy;
    const float* u;
    float* dx;
    D* dx16;
    static constexpr int VEC = 4, NIN = 2;
    __device__ __forceinline__ void init(int64_t) {}
    __device__ __forceinline__ void load(int64_t at, float (&in)[NIN][VEC]) const {
        VecIO<float, 4>::load(dy + at, in[0]);
        VecIO<float, 4>::load(u + at, in[1]);
    }
    __device__ __forceinline__ void finish(int64_t at, float (&in)[NIN][VEC]) const {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            in[0][j] = in[0][j] * gelu_grad_one(in[1][j]);
            asm volatile("" : "+v"(in[0][j]));   // one fp32 value for the store, the copy and the sum
        }
        VecIO<float, 4>::store(dx + at, in[0]);
        store4_as16<D>(dx16 + at, in[0]);
    }
};
// dx = dy * gelu'(x + bias) in the storage type; what was stored is what is summed (bias_gelu_bwd_kernel)
template <typename T, int V>
struct OwnBiasGeluBwd {
    const T* dy;
    const T* x;
    const float* bias;
    T* dx;
    T* dy_copy;   // null: none
    float b[V];
    static constexpr int VEC = V, NIN = 2;
    __device__ __forceinline__ void init(int64_t col) {
#pragma unroll
        for (int j = 0; j < V; j++) b[j] = bias ? bias[col + j] : 0.f;
    }
    __device__ __forceinline__ void load(int64_t at, float (&in)[NIN][VEC]) const {
        VecIO<T, V>::load(dy + at, in[0]);
        VecIO<T, V>::load(x + at, in[1]);
    }
    __device__ __forceinline__ void finish(int64_t at, float (&in)[NIN][VEC]) const {
        if (dy_copy) VecIO<T, V>::store_rounded(dy_copy + at, in[0]);   // exact: the values are of this type
#pragma unroll
        for (int j = 0; j < V; j++) in[0][j] *= gelu_grad_one(in[1][j] + b[j]);
        VecIO<T, V>::store_rounded(dx + at, in[0]);
    }
};

constexpr int kOwnThreads = 1024;

// Workgroup ids are dealt to the 8 XCDs in turn: the b-th of n takes a position such that an XCD's workgroups are
// neighbours (strips narrower than a cache line share their lines in one L2).
__device__ __forceinline__ unsigned xcd_contiguous(unsigned b, unsigned n) {
    const unsigned per = n / 8, rem = n % 8, x = b % 8;
    return x * per + (x < rem ? x : rem) + b / 8;
}

template <int LPR, int UNROLL, typename Src>
__global__ __launch_bounds__(kOwnThreads) void colsum_owner_kernel(Src src_arg, float* __restrict__ out, int64_t rows,
                                                                   int64_t cols, float scale) {
    constexpr int VEC = Src::VEC, NIN = Src::NIN, RPP = kOwnThreads / LPR, CW = LPR * VEC, WAVES = kOwnThreads / 64;
    __shared__ float slots[WAVES][CW];
    Src src = src_arg;
    const int lr = threadIdx.x % LPR, rr = threadIdx.x / LPR;
    const int64_t strip = xcd_contiguous(blockIdx.x, gridDim.x);
    const int64_t col = strip * CW + lr * VEC;
    float acc[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) acc[j] = 0.f;
    if (col < cols) {
        src.init(col);
        // One pass over rows that are all there: nothing conditional, so that the arithmetic of all positions overlaps
        // ([512 x 8192] fp16 5.4 -> 4.8 us).  Several passes keep the test of every position: each position then waits for
        // its own loads alone ([4096 x 16384] fp16 25.9 us, 28.8 without).
        const bool whole = UNROLL > 1 && rows <= UNROLL * RPP && rr + (UNROLL - 1) * RPP < rows;
        if (whole) {
            float in[UNROLL][NIN][VEC];
#pragma unroll
            for (int u = 0; u < UNROLL; u++) src.load((int64_t)(rr + u * RPP) * cols + col, in[u]);
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                src.finish((int64_t)(rr + u * RPP) * cols + col, in[u]);
#pragma unroll
                for (int j = 0; j < VEC; j++) acc[j] += in[u][0][j];
            }
        } else {
            for (int64_t r = rr; r < rows; r += UNROLL * RPP) {
                float in[UNROLL][NIN][VEC];
                // positions past the last row read that row (every load of a pass leaves before the first is used)
#pragma unroll
                for (int u = 0; u < UNROLL; u++) {
                    const int64_t at = r + u * RPP;
                    src.load((at < rows ? at : rows - 1) * cols + col, in[u]);
                }
#pragma unroll
                for (int u = 0; u < UNROLL; u++) {
                    if (r + u * RPP < rows) {
                        src.finish((r + u * RPP) * cols + col, in[u]);
#pragma unroll
                        for (int j = 0; j < VEC; j++) acc[j] += in[u][0][j];
                    }
                }
            }
        }
    }
    // the 64 / LPR row slots of a wave meet by lane exchanges, the waves through LDS
#pragma unroll
    for (int d = LPR; d < 64; d *= 2)
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[j] += __shfl_xor(acc[j], d);
    if ((threadIdx.x & 63) < LPR) {
#pragma unroll
        for (int j = 0; j < VEC; j++) slots[threadIdx.x >> 6][lr * VEC + j] = acc[j];
    }
    __syncthreads();
    if (threadIdx.x < CW) {
        float z = 0.f;
#pragma unroll
        for (int k = 0; k < WAVES; k++) z += slots[k][threadIdx.x];
        const int64_t oc = strip * CW + threadIdx.x;
        if (oc < cols) out[oc] = z * scale;
    }
}

// Lanes per row of the one-launch column sum, or 0 where two launches are faster: on many rows, where a workgroup's walk
// takes longer than the second launch.  Depends on the shape, the element size and the kind of source alone, so entries
// that promise each other's bits (br_hip_colsum / br_hip_colsum_cast / br_hip_gelu_bwd_colsum_cast on fp32) always
// agree on the path -- the rule for fp32 is therefore one that suits all three.  Measured, us, two launches / one with 2,
// 4, 8 lanes:
//   16-bit sums         [64,1024] 4.8 / 3.7 3.4 3.1   [256,4096] 5.5 / 3.9 4.2 4.3   [512,2048] 5.8 / 4.6 5.0 4.5
//                       [1000,1024] 6.7 / 6.0 6.1 6.6   [1024,8192] 12.0 / 9.8 7.0 7.0   [2048,1024] 6.6 / 8.7 9.1 10.2
//                       [2048,4096] 9.6 / 9.4 9.8 10.8   [2048,6144] 11.7 / 16.5 10.4 11.3   [4096,512] 7.3 / 14 15 17
//                       [4096,6144] 14.8 / 30 18 20   [4096,16384] 29.7 / 54 37 25.9   [65536,512] 44 / - 204 -
//   fp32 sum and copy   [64,1024] 4.8 / 3.0 2.9 2.9   [256,1024] 4.9 / 3.2 3.2 3.4   [512,1024] 5.7 / 4.1 4.6 5.0
//                       [512,8192] 10.3 / 12 9.0 7.3   [1000,1024] 7.5 / 6.9 7.0 7.8   [1000,4096] 11.2 / 12 8.6 9.2
//                       [1000,8192] 14.7 / 23 15 11.7
//   with GELU backward  [64,1024] 5.8 / 3.1 3.0 3.1   [256,1024] 6.4 / 4.2 4.5 5.1   [512,1024] 7.0 / 6.8 7.8 8.8
//   in front            [768,1024] 8.0 / 9.9 11 12   [1000,2048] 11.7 / 15 16 17   [1000,4096] 16.8 / 30 18.1 19.1
//                       [1000,8192] 26.1 / 65 38 25.4
//   bias-GELU backward  [64,4096] 8.2 / 4.5 4.3 4.2   [256,2048] 8.2 / 6.3 5.6 5.8   [512,4096] 9.3 / 8.7 8.6 9.3
//   (fp16)              [1000,1024] 12.3 / 11.0 12.4 14   [1000,4096] 13.7 / 14.4 14.1 15   [1000,8192] 15.7 / 27 16.5 17.2
//                       [1000,16384] 24.4 / 55 32 21.9;  (fp32) [512,2048] 8.2 / 7.6 8.1 8.6   [768,1024] 8.7 / 9.2 10 11
enum OwnerKind { kOwnSum, kOwnBiasGelu };
int owner_lanes(int64_t rows, int64_t cols, int elem_bytes, OwnerKind kind) {
    const bool narrow_type = elem_bytes != 4;   // 16-bit elements
    if (cols % (narrow_type ? 8 : 4) != 0) return 0;
    if (rows <= 128) return 8;   // one row position a thread
    if (rows <= 512) {
        if (cols > 4096) return 8;
        if (narrow_type) return kind == kOwnSum ? 2 : 4;
        return cols <= 2048 ? 2 : 4;
    }
    if (kind == kOwnSum && narrow_type) {
        if (rows <= 1024) return cols <= 8192 ? 4 : 8;
        if (rows <= 2048 && cols >= 6144) return cols <= 8192 ? 4 : 8;
        return cols >= 12288 ? 8 : 0;
    }
    if (rows > 1024) return 0;
    if (kind == kOwnBiasGelu) return narrow_type ? (cols <= 2048 ? 2 : cols < 12288 ? 0 : 8) : (cols < 6144 ? 0 : 8);
    // Fewer than four times as many columns as rows: a block's sums over its hidden size, one launch fewer in a chain of
    // short ones (a step over 1000 tokens at hidden 1024 450 us, 457 with two launches).  The GELU backward, which comes
    // at four times the hidden size in a block, pays for it where a caller has it on fewer columns.
    if (cols < 3072) return cols < 4 * rows ? 2 : 0;
    return cols <= 4096 ? 4 : 8;
}

template <int LPR, int UNROLL, typename Src>
void colsum_owner_launch_lanes(const Src& src, float* out, int64_t rows, int64_t cols, float scale, hipStream_t st) {
    const int64_t cw = LPR * Src::VEC;
    const unsigned grid = (unsigned)((cols + cw - 1) / cw);
    // rows of a single pass: no loads beside those of that pass (with two or four passes in flight their surplus costs
    // 0.4 us, half as much again with the GELU gradient)
    if (rows <= kOwnThreads / LPR) colsum_owner_kernel<LPR, 1, Src><<<grid, kOwnThreads, 0, st>>>(src, out, rows, cols, scale);
    else colsum_owner_kernel<LPR, UNROLL, Src><<<grid, kOwnThreads, 0, st>>>(src, out, rows, cols, scale);
}
template <int UNROLL, typename Src>
int colsum_owner_launch(int lanes, const Src& src, float* out, int64_t rows, int64_t cols, float scale, hipStream_t st) {
    if (lanes == 8) colsum_owner_launch_lanes<8, UNROLL>(src, out, rows, cols, scale, st);
    else if (lanes == 4) colsum_owner_launch_lanes<4, UNROLL>(src, out, rows, cols, scale, st);
    else colsum_owner_launch_lanes<2, UNROLL>(src, out, rows, cols, scale, st);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// Several fp32 matrices packed side by side, columns summed on the way: blockIdx.y is the matrix, a workgroup owns a
// strip of LPR quads of its columns as in colsum_owner_kernel.
constexpr int kPacked = 4;
struct PackSet {
    const float* x[kPacked];
};
template <int LPR, typename D>
__global__ __launch_bounds__(kOwnThreads) void pack_colsum_kernel(PackSet set, float* __restrict__ out, D* __restrict__ packed,
                                                                  int64_t rows, int64_t cols, int64_t pitch, float scale) {
    constexpr int VEC = 4, UNROLL = 4, RPP = kOwnThreads / LPR, CW = LPR * VEC, WAVES = kOwnThreads / 64;
    __shared__ float slots[WAVES][CW];
    const float* x = set.x[0];
#pragma unroll
    for (int i = 1; i < kPacked; i++)
        if (blockIdx.y == (unsigned)i) x = set.x[i];
    out += blockIdx.y * cols;
    packed += blockIdx.y * cols;
    const int lr = threadIdx.x % LPR, rr = threadIdx.x / LPR;
    const int64_t strip = xcd_contiguous(blockIdx.x, gridDim.x);
    const int64_t col = strip * CW + lr * VEC;
    float acc[VEC] = {0.f, 0.f, 0.f, 0.f};
    if (col < cols) {
        for (int64_t r = rr; r < rows; r += UNROLL * RPP) {
            float in[UNROLL][VEC];
            // positions past the last row read that row (every load of a pass leaves before the first is used)
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int64_t at = r + u * RPP;
                VecIO<float, VEC>::load(x + (at < rows ? at : rows - 1) * cols + col, in[u]);
            }
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                if (r + u * RPP >= rows) break;
                D* const to = packed + (r + u * RPP) * pitch + col;
                if constexpr (sizeof(D) == 4) VecIO<float, VEC>::store(to, in[u]);
                else store4_as16<D>(to, in[u]);
#pragma unroll
                for (int j = 0; j < VEC; j++) acc[j] += in[u][j];
            }
        }
    }
#pragma unroll
    for (int d = LPR; d < 64; d *= 2)
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[j] += __shfl_xor(acc[j], d);
    if ((threadIdx.x & 63) < LPR) {
#pragma unroll
        for (int j = 0; j < VEC; j++) slots[threadIdx.x >> 6][lr * VEC + j] = acc[j];
    }
    __syncthreads();
    // The waves' sums meet in pairs: one after the other, sixteen of them are most of a result's error ([1024] from 300 rows against
    // 64 bits 9.9e-8, so 7.9e-8; [2048] from 1024 1.06e-7, 9.1e-8).
    if (threadIdx.x < CW) {
        float z[WAVES];
#pragma unroll
        for (int k = 0; k < WAVES; k++) z[k] = slots[k][threadIdx.x];
#pragma unroll
        for (int half = WAVES / 2; half > 0; half /= 2)
#pragma unroll
            for (int k = 0; k < half; k++) z[k] += z[k + half];
        const int64_t oc = strip * CW + threadIdx.x;
        if (oc < cols) out[oc] = z[0] * scale;
    }
}
template <typename D>
int pack_colsum(const PackSet& set, int count, float* out, void* packed, int64_t rows, int64_t cols, float scale, hipStream_t st) {
    // The widest strips that make 128 workgroups: with narrower ones a line of x is asked for by several.  Strips of 2 / 4 / 8
    // quads, three matrices to fp16, us: [1000 x 512] 6.0 / 6.5 / 7.4, [1000 x 1024] 11.7 / 8.1 / 8.6, [1024 x 2048] 17.4 / 14.2 / 10.3,
    // [500 x 1024] 6.3 / 4.8 / 5.2, [512 x 2048] 10.0 / 8.1 / 6.2, [300 x 1024] 4.1 / 3.7 / 3.8.
    const int lanes = rows <= 128 || count * cols / 32 >= 128 ? 8 : count * cols / 16 >= 128 ? 4 : 2;
    const dim3 grid((unsigned)((cols + lanes * 4 - 1) / (lanes * 4)), (unsigned)count);
    D* const p = (D*)packed;
    if (lanes == 2) pack_colsum_kernel<2, D><<<grid, kOwnThreads, 0, st>>>(set, out, p, rows, cols, count * cols, scale);
    else if (lanes == 4) pack_colsum_kernel<4, D><<<grid, kOwnThreads, 0, st>>>(set, out, p, rows, cols, count * cols, scale);
    else pack_colsum_kernel<8, D><<<grid, kOwnThreads, 0, st>>>(set, out, p, rows, cols, count * cols, scale);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// ------------------------------------------------------- transpose 0213
// One 16-byte granule per thread, indexed by OUTPUT position so stores are
// fully coalesced; loads are contiguous runs of s3 elements.
//
// blockIdx.y picks one of several tensors of the same shape: the heads of q, k and v change places in one launch (a
// launch of 2.5-5 us each, of which a block of a thousand tokens has two times three).
constexpr int kTransposes = 4;
struct TransposeSet {
    const uint4* x[kTransposes];
    uint4* y[kTransposes];
};
__global__ __launch_bounds__(kBlock) void transpose_0213_x16(TransposeSet set, long long n16,
                                                              unsigned s1, unsigned s2, unsigned s3g) {
    const uint4* x = set.x[0];
    uint4* y = set.y[0];
#pragma unroll
    for (int i = 1; i < kTransposes; i++)
        if (blockIdx.y == (unsigned)i) x = set.x[i], y = set.y[i];
    const long long stride = (long long)gridDim.x * kBlock;
    for (long long o = (long long)blockIdx.x * kBlock + threadIdx.x; o < n16; o += stride) {
        unsigned long long r = (unsigned long long)o;
        const unsigned i3 = (unsigned)(r % s3g);
        r /= s3g;
        const unsigned i1 = (unsigned)(r % s1);  // output dim 2 is input dim 1
        r /= s1;
        const unsigned i2 = (unsigned)(r % s2);
        const unsigned long long i0 = r / s2;
        y[o] = x[((i0 * s1 + i1) * s2 + i2) * s3g + i3];
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void transpose_0213_scalar(const T* x, T* y, long long n, unsigned s1,
                                                                 unsigned s2, unsigned s3) {
    const long long stride = (long long)gridDim.x * kBlock;
    for (long long o = (long long)blockIdx.x * kBlock + threadIdx.x; o < n; o += stride) {
        unsigned long long r = (unsigned long long)o;
        const unsigned i3 = (unsigned)(r % s3);
        r /= s3;
        const unsigned i1 = (unsigned)(r % s1);
        r /= s1;
        const unsigned i2 = (unsigned)(r % s2);
        const unsigned long long i0 = r / s2;
        y[o] = x[((i0 * s1 + i1) * s2 + i2) * s3 + i3];
    }
}

// ------------------------------------------------------ data preparation
// One workgroup per output row; rows whose id is out of range are zeroed.
__global__ __launch_bounds__(kBlock) void gather_rows_x16(const uint4* table, const int32_t* ids, uint4* out,
                                                           int64_t row16, int64_t vocab) {
    const int64_t row = blockIdx.x;
    const int64_t id = ids[row];
    const bool ok = id >= 0 && id < vocab;
    for (int64_t i = threadIdx.x; i < row16; i += kBlock)
        out[row * row16 + i] = ok ? table[id * row16 + i] : make_uint4(0, 0, 0, 0);
}

__global__ __launch_bounds__(kBlock) void gather_rows_bytes(const unsigned char* table, const int32_t* ids,
                                                             unsigned char* out, int64_t row_bytes,
                                                             int64_t vocab) {
    const int64_t row = blockIdx.x;
    const int64_t id = ids[row];
    const bool ok = id >= 0 && id < vocab;
    for (int64_t i = threadIdx.x; i < row_bytes; i += kBlock)
        out[row * row_bytes + i] = ok ? table[id * row_bytes + i] : (unsigned char)0;
}

// The same with 16-bit rows converted to fp32 on the way; one launch and one pass over the rows fewer than gathering and
// then converting them.
template <typename T>
__global__ __launch_bounds__(kBlock) void gather_rows_f32(const T* table, const int32_t* ids, float* out, int64_t hidden, int64_t vocab) {
    const int64_t row = blockIdx.x;
    const int64_t id = ids[row];
    const bool ok = id >= 0 && id < vocab;
    for (int64_t i = threadIdx.x; i < hidden; i += kBlock) out[row * hidden + i] = ok ? (float)table[id * hidden + i] : 0.f;
}

// Rows picked by the host, named in the kernel's arguments: row i of out is x[at[i], :] as type D.  Grid (rows, pieces
// of a row), VEC columns a thread.
//
// A dozen kilobytes a row: what it costs is the launch.  Eight rows of 4096 copied one by one and then converted to
// fp16 took nine dependent launches of 2-5 us each; here they are one (scores of 8 sequences over 250880 words 361 ->
// 346 us, 5.95 TB/s over the head's weights).
constexpr int kPickedRows = 256;
struct PickedRows {
    int64_t at[kPickedRows];
};
template <typename D, int VEC>
__global__ __launch_bounds__(kBlock) void pick_rows_kernel(const float* x, PickedRows rows, D* out, int64_t cols) {
    const float* src = x + rows.at[blockIdx.x] * cols;
    D* dst = out + blockIdx.x * cols;
    const int64_t stride = (int64_t)gridDim.y * kBlock * VEC;
    for (int64_t c = ((int64_t)blockIdx.y * kBlock + threadIdx.x) * VEC; c < cols; c += stride) {
        if (VEC == 4) {
            const float4 v = *reinterpret_cast<const float4*>(src + c);
            dst[c] = from_f32<D>(v.x);
            dst[c + 1] = from_f32<D>(v.y);
            dst[c + 2] = from_f32<D>(v.z);
            dst[c + 3] = from_f32<D>(v.w);
        } else {
            dst[c] = from_f32<D>(src[c]);
        }
    }
}

template <typename D>
int pick_rows(const float* x, const int64_t* rows, void* out_, int64_t n, int64_t cols, hipStream_t st) {
    D* out = static_cast<D*>(out_);
    const bool vec = cols % 4 == 0 && aligned16(x);
    const int64_t per_block = vec ? 4 * kBlock : kBlock, pieces = (cols + per_block - 1) / per_block;
    for (int64_t first = 0; first < n; first += kPickedRows) {
        PickedRows r{};
        const int64_t count = n - first < kPickedRows ? n - first : kPickedRows;
        for (int64_t i = 0; i < count; i++) r.at[i] = rows[first + i];
        const dim3 grid((unsigned)count, (unsigned)(pieces < 1024 ? pieces : 1024));
        if (vec)
            pick_rows_kernel<D, 4><<<grid, kBlock, 0, st>>>(x, r, out + first * cols, cols);
        else
            pick_rows_kernel<D, 1><<<grid, kBlock, 0, st>>>(x, r, out + first * cols, cols);
        BR_HIP_LAUNCH_CHECK();
    }
    return BR_OK;
}

constexpr int kSlopeChunk = 128;
struct SlopeChunk {
    double v[kSlopeChunk];
};

__global__ __launch_bounds__(kBlock) void alibi_table_kernel(float* alibi, SlopeChunk slopes, int head0,
                                                              int nheads, int64_t tokens) {
    const int64_t n = (int64_t)nheads * tokens;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        const int h = (int)(i / tokens);
        const int64_t k = i % tokens;
        // fp64 product rounded once to fp32, as the host code it replaces does
        alibi[(int64_t)head0 * tokens + i] = (float)((double)k * 1.0 * slopes.v[h]);
    }
}

// One workgroup per (batch, query row).  valid = index of the first zero in
// mask[b,:] (tokens when there is none) is found by a min-reduction.
__global__ __launch_bounds__(kBlock) void xmask_table_kernel(const int32_t* mask, float* xmask,
                                                              int64_t tokens) {
    __shared__ int s_valid[kBlock / kWave];
    const int64_t b = blockIdx.y;
    const int64_t q = blockIdx.x;
    const int32_t* m = mask + b * tokens;
    int first_zero = (int)tokens;
    // keys beyond q are masked by causality anyway, so scanning [0, q] suffices
    for (int64_t k = threadIdx.x; k <= q; k += kBlock)
        if (m[k] == 0 && (int)k < first_zero) first_zero = (int)k;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(first_zero, off, kWave);
        first_zero = o < first_zero ? o : first_zero;
    }
    if ((threadIdx.x & 63) == 0) s_valid[threadIdx.x >> 6] = first_zero;
    __syncthreads();
    int valid = s_valid[0];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; w++) valid = s_valid[w] < valid ? s_valid[w] : valid;
    float* row = xmask + (b * tokens + q) * tokens;
    for (int64_t k = threadIdx.x; k < tokens; k += kBlock)
        row[k] = (k <= q && k < valid) ? 0.0f : -FLT_MAX;
}

bool fits_u32(int64_t v) { return v > 0 && v <= 0xffffffffLL; }

// ---------------------------------------------------------- normal fill
// dst[i] = mean + std * z_i with z_i a standard normal that depends only on
// (seed, i): SplitMix64 of the pair gives two 24-bit uniforms, Box-Muller one
// normal.  The same (seed, i) gives the same value on any launch geometry.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
template <typename T>
__global__ __launch_bounds__(kBlock) void normal_kernel(T* dst, float mean, float std, unsigned long long seed,
                                                         int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        const unsigned long long h = splitmix64(splitmix64(seed) ^ (unsigned long long)i);
        const float u1 = ((float)(unsigned)(h >> 40) + 1.0f) * (1.0f / 16777216.0f);  // (0, 1]
        const float u2 = (float)(unsigned)((h >> 8) & 0xffffffu) * (1.0f / 16777216.0f);
        const float z = sqrtf(-2.0f * __logf(u1)) * __cosf(6.28318530718f * u2);
        float value = mean + std * z;
        // keep the fp32 rounding: without the barrier the multiply-add is fused into
        // the 16-bit conversion and a 16-bit tensor would not be the rounded fp32 one
        asm volatile("" : "+v"(value));
        dst[i] = from_f32<T>(value);
    }
}

// Backward of the row gather: grad[ids[i], :] += dx[i, :] for i = 0 .. n-1, in
// that order, so that the result does not depend on scheduling when an id
// occurs several times.  Workgroup (i, s) owns column blocks s, s + gridDim.y, .. (of kBlock * VEC columns) of the
// row of id = ids[i] if i is that id's first position; it collects the later positions
// of the same id, a block of positions at a time, into an ascending list in LDS
// and folds their rows in, four loads in flight, starting from the row's current
// value.  What bounds it is the longest run of one id (text repeats a few ids
// often).  Reading ids[] one position at a time instead, as each column block
// did, cost 109 us for 512 positions of 4096 columns with ids as frequent as
// words are; this takes 9.
template <int VEC>
__global__ __launch_bounds__(kBlock) void scatter_add_rows(const float* __restrict__ dx,
                                                            const int32_t* __restrict__ ids, float* grad, int n,
                                                            int64_t hidden, int64_t vocab, float scale) {
    __shared__ int list[kBlock];
    __shared__ int found[kBlock / kWave];
    const int i = blockIdx.x, t = threadIdx.x;
    const int32_t id = ids[i];
    if (id < 0 || (int64_t)id >= vocab) return;
    int seen = 0;
    for (int j = t; j < i; j += kBlock) seen |= ids[j] == id;
    if (__syncthreads_or(seen)) return;
    auto read = [](const float* p, float (&f)[VEC]) {
        if constexpr (VEC == 4) VecIO<float, 4>::load(p, f);
        else f[0] = *p;
    };
    for (int64_t first = (int64_t)blockIdx.y * kBlock * VEC; first < hidden; first += (int64_t)gridDim.y * kBlock * VEC) {
        const int64_t c = first + t * VEC;
        const bool mine = c < hidden;
        float* row = grad + (int64_t)id * hidden + c;
        float acc[VEC];
        if (mine) read(row, acc);
        for (int base = i; base < n; base += kBlock) {
            const int j = base + t;
            const bool hit = j < n && ids[j] == id;
            const unsigned long long hits = __ballot(hit);
            if ((t & 63) == 0) found[t >> 6] = __popcll(hits);
            __syncthreads();
            int at = __popcll(hits & ((1ull << (t & 63)) - 1)), count = 0;
#pragma unroll
            for (int w = 0; w < kBlock / kWave; w++) {
                at += w < (t >> 6) ? found[w] : 0;
                count += found[w];
            }
            if (hit) list[at] = j;
            __syncthreads();
            if (mine) {
                int p = 0;
                for (; p + 4 <= count; p += 4) {
                    float d[4][VEC];
#pragma unroll
                    for (int u = 0; u < 4; u++) read(dx + (int64_t)list[p + u] * hidden + c, d[u]);
#pragma unroll
                    for (int u = 0; u < 4; u++)
#pragma unroll
                        for (int e = 0; e < VEC; e++) acc[e] += d[u][e] * scale;
                }
                for (; p < count; p++) {
                    float d[VEC];
                    read(dx + (int64_t)list[p] * hidden + c, d);
#pragma unroll
                    for (int e = 0; e < VEC; e++) acc[e] += d[e] * scale;
                }
            }
            __syncthreads();   // the list is used up
        }
        if (mine) {
            if constexpr (VEC == 4) VecIO<float, 4>::store(row, acc);
            else *row = acc[0];
        }
    }
}

}  // namespace

extern "C" {

int br_hip_fill(void* dst, int dtype, float value, int64_t n, br_stream_t stream) {
    if (n < 0) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!dst) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    const int grid = grid_for(n, kBlock);
    switch (dtype) {
        case BR_F32: fill_kernel<float><<<grid, kBlock, 0, st>>>((float*)dst, value, n); break;
        case BR_F16: fill_kernel<__half><<<grid, kBlock, 0, st>>>((__half*)dst, __float2half_rn(value), n); break;
        case BR_BF16:
            fill_kernel<__hip_bfloat16><<<grid, kBlock, 0, st>>>((__hip_bfloat16*)dst, __float2bfloat16(value), n);
            break;
        case BR_I32: fill_kernel<int32_t><<<grid, kBlock, 0, st>>>((int32_t*)dst, (int32_t)value, n); break;
        default: return BR_ERR_TODO;
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_normal(void* dst, int dtype, float mean, float std, uint64_t seed, int64_t n, br_stream_t stream) {
    if (n < 0) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!dst) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    const int grid = grid_for(n, kBlock);
    switch (dtype) {
        case BR_F32: normal_kernel<float><<<grid, kBlock, 0, st>>>((float*)dst, mean, std, seed, n); break;
        case BR_F16: normal_kernel<__half><<<grid, kBlock, 0, st>>>((__half*)dst, mean, std, seed, n); break;
        case BR_BF16:
            normal_kernel<__hip_bfloat16><<<grid, kBlock, 0, st>>>((__hip_bfloat16*)dst, mean, std, seed, n);
            break;
        default: return BR_ERR_TODO;
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_cast(const void* src, int src_dtype, void* dst, int dst_dtype, int64_t n, br_stream_t stream) {
    if (n < 0) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!src) return BR_ERR_INPUT;
    if (!dst) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    switch (src_dtype) {
        case BR_F32: return cast_from<float>(src, dst, dst_dtype, n, st);
        case BR_F16: return cast_from<__half>(src, dst, dst_dtype, n, st);
        case BR_BF16: return cast_from<__hip_bfloat16>(src, dst, dst_dtype, n, st);
        default: return BR_ERR_TODO;
    }
}

int br_hip_add_bcast(const void* a, const void* b, void* c, int dtype, const int64_t as[4],
                     const int64_t bs[4], br_stream_t stream) {
    if (!a || !b || !as || !bs) return BR_ERR_INPUT;
    if (!c) return BR_ERR_OUTPUT;
    if (dtype != BR_F32 && dtype != BR_F16) return BR_ERR_TODO;
    bool same = true;
    for (int i = 0; i < 4; i++) {
        if (as[i] <= 0 || bs[i] <= 0) return BR_ERR_ATTR;
        if (bs[i] != as[i] && bs[i] != 1) return BR_ERR_INPUT;
        same = same && bs[i] == as[i];
    }
    const int64_t n = as[0] * as[1] * as[2] * as[3];
    hipStream_t st = as_stream(stream);
    const bool al = aligned16(a) && aligned16(b) && aligned16(c);
    if (same && al && dtype == BR_F32 && n % 4 == 0) {
        add_same_f32x4<<<grid_for(n / 4, kBlock), kBlock, 0, st>>>((const float4*)a, (const float4*)b,
                                                                   (float4*)c, n / 4);
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
    if (same && al && dtype == BR_F16 && n % 8 == 0) {
        add_same_f16x8<<<grid_for(n / 8, kBlock), kBlock, 0, st>>>((const half8*)a, (const half8*)b,
                                                                   (half8*)c, n / 8);
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
    if (!fits_u32(as[1]) || !fits_u32(as[2]) || !fits_u32(as[3])) return BR_ERR_ATTR;
    const long long bst3 = bs[3] == 1 ? 0 : 1;
    const long long bst2 = bs[2] == 1 ? 0 : bs[3];
    const long long bst1 = bs[1] == 1 ? 0 : bs[2] * bs[3];
    const long long bst0 = bs[0] == 1 ? 0 : bs[1] * bs[2] * bs[3];
    // 128-bit path: needs every row start of a, b and c to stay 16-byte aligned
    const bool vec_ok = dtype == BR_F32 && al && as[3] % 4 == 0 && (bst3 == 0 || bs[3] % 4 == 0);
    if (vec_ok) {
        BcastDims d;
        d.s1 = (unsigned)as[1];
        d.s2 = (unsigned)as[2];
        d.s3v = (unsigned)(as[3] / 4);
        d.bst0 = bst0; d.bst1 = bst1; d.bst2 = bst2; d.bst3 = (int)bst3;
        add_bcast_f32x4<<<grid_for(n / 4, kBlock), kBlock, 0, st>>>((const float*)a, (const float*)b,
                                                                    (float*)c, n / 4, d);
    } else if (dtype == BR_F32) {
        add_bcast_scalar<float><<<grid_for(n, kBlock), kBlock, 0, st>>>(
            (const float*)a, (const float*)b, (float*)c, n, (unsigned)as[1], (unsigned)as[2],
            (unsigned)as[3], bst0, bst1, bst2, (int)bst3);
    } else {
        add_bcast_scalar<__half><<<grid_for(n, kBlock), kBlock, 0, st>>>(
            (const __half*)a, (const __half*)b, (__half*)c, n, (unsigned)as[1], (unsigned)as[2],
            (unsigned)as[3], bst0, bst1, bst2, (int)bst3);
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

static int strip_rows(int64_t rows) {
    // strips of rows per workgroup: about 64 strips, at least 8 rows each
    int64_t rpb = (rows + 63) / 64;
    if (rpb < 8) rpb = 8;
    return (int)rpb;
}

int br_hip_gelu_fwd_f32_to_16(const float* x, void* y, int y_dtype, int64_t n, br_stream_t stream) {
    if (n < 0) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!x) return BR_ERR_INPUT;
    if (!y) return BR_ERR_OUTPUT;
    if (y_dtype != BR_F16 && y_dtype != BR_BF16) return BR_ERR_TODO;
    if (n % 8 != 0 || !aligned16(x) || !aligned16(y)) return BR_ERR_TODO;
    const int grid = grid_for(n / 8, kBlock);
    if (y_dtype == BR_F16)
        gelu_fwd_f32_to_16<__half><<<grid, kBlock, 0, as_stream(stream)>>>((const float4*)x, (uint4*)y, n / 8);
    else
        gelu_fwd_f32_to_16<__hip_bfloat16><<<grid, kBlock, 0, as_stream(stream)>>>((const float4*)x, (uint4*)y, n / 8);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_gelu_fwd_copy16(const float* x, float* y, void* y16, int y16_dtype, int64_t n, br_stream_t stream) {
    if (n < 0) return BR_ERR_ATTR;
    if (y16_dtype != BR_F16 && y16_dtype != BR_BF16) return BR_ERR_TODO;
    if (n == 0) return BR_OK;
    if (!x) return BR_ERR_INPUT;
    if (!y || !y16) return BR_ERR_OUTPUT;
    if (n % 8 != 0 || !aligned16(x) || !aligned16(y) || !aligned16(y16)) return BR_ERR_TODO;
    const unsigned grid = (unsigned)grid_for(n / 8, kBlock);
    if (y16_dtype == BR_F16)
        gelu_fwd_f32_to_16<__half><<<grid, kBlock, 0, as_stream(stream)>>>((const float4*)x, (uint4*)y16, n / 8, (float4*)y);
    else
        gelu_fwd_f32_to_16<__hip_bfloat16><<<grid, kBlock, 0, as_stream(stream)>>>((const float4*)x, (uint4*)y16, n / 8, (float4*)y);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_gelu_fwd(const void* x, void* y, int dtype, int64_t n, br_stream_t stream) {
    if (n < 0) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!x) return BR_ERR_INPUT;
    if (!y) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    const bool al = aligned16(x) && aligned16(y);
    if (dtype == BR_F32 && al && n % 4 == 0) {
        gelu_fwd_f32<<<grid_for(n / 4, kBlock), kBlock, 0, st>>>((const float*)x, (float*)y, n / 4);
    } else if (dtype == BR_F16 && al && n % 8 == 0) {
        gelu_fwd_f16<<<grid_for(n / 8, kBlock), kBlock, 0, st>>>((const half8*)x, (half8*)y, n / 8);
    } else if (dtype == BR_F32) {
        gelu_scalar<float><<<grid_for(n, kBlock), kBlock, 0, st>>>(nullptr, (const float*)x, nullptr, (float*)y,
                                                                  n, 1, false);
    } else if (dtype == BR_F16) {
        gelu_scalar<__half><<<grid_for(n, kBlock), kBlock, 0, st>>>(nullptr, (const __half*)x, nullptr,
                                                                   (__half*)y, n, 1, false);
    } else {
        return BR_ERR_TODO;
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_bias_gelu_fwd(const void* x, const float* bias, void* y, int dtype, int64_t rows, int64_t cols,
                         br_stream_t stream) {
    if (rows < 0 || cols <= 0) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!x || !bias) return BR_ERR_INPUT;
    if (!y) return BR_ERR_OUTPUT;
    if (dtype != BR_F32 && dtype != BR_F16) return BR_ERR_TODO;
    hipStream_t st = as_stream(stream);
#ifndef BR_GELU_FWD_FLAT
#define BR_GELU_FWD_FLAT 1
#endif
    // one row per workgroup row of the grid (workgroups in memory order, see grid_for) while the grid allows
    const int rpb = BR_GELU_FWD_FLAT && rows <= 65535 ? 1 : strip_rows(rows);
    const unsigned groups = (unsigned)((rows + rpb - 1) / rpb);
    const bool al = aligned16(x) && aligned16(y);
    if (dtype == BR_F32 && al && cols % 4 == 0) {
        dim3 grid((unsigned)((cols / 4 + kBlock - 1) / kBlock), groups);
        bias_gelu_fwd_kernel<float, 4><<<grid, kBlock, 0, st>>>((const float*)x, bias, (float*)y, rows, cols, rpb);
    } else if (dtype == BR_F16 && al && cols % 8 == 0) {
        dim3 grid((unsigned)((cols / 8 + kBlock - 1) / kBlock), groups);
        bias_gelu_fwd_kernel<__half, 8><<<grid, kBlock, 0, st>>>((const __half*)x, bias, (__half*)y, rows, cols,
                                                                  rpb);
    } else {
        const int64_t n = rows * cols;
        if (dtype == BR_F32)
            gelu_scalar<float><<<grid_for(n, kBlock), kBlock, 0, st>>>(nullptr, (const float*)x, bias, (float*)y,
                                                                      n, cols, false);
        else
            gelu_scalar<__half><<<grid_for(n, kBlock), kBlock, 0, st>>>(nullptr, (const __half*)x, bias,
                                                                       (__half*)y, n, cols, false);
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_gelu_bwd(const void* dy, const void* x, void* dx, int dtype, int64_t n, br_stream_t stream) {
    if (n < 0) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!dy || !x) return BR_ERR_INPUT;
    if (!dx) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    const bool al = aligned16(dy) && aligned16(x) && aligned16(dx);
    if (dtype == BR_F32 && al && n % 4 == 0) {
        gelu_bwd_f32<<<grid_for(n / 4, kBlock), kBlock, 0, st>>>((const float*)dy, (const float*)x, (float*)dx,
                                                                n / 4);
    } else if (dtype == BR_F16 && al && n % 8 == 0) {
        gelu_bwd_f16<<<grid_for(n / 8, kBlock), kBlock, 0, st>>>((const half8*)dy, (const half8*)x, (half8*)dx,
                                                                n / 8);
    } else if (dtype == BR_F32) {
        gelu_scalar<float><<<grid_for(n, kBlock), kBlock, 0, st>>>((const float*)dy, (const float*)x, nullptr,
                                                                  (float*)dx, n, 1, true);
    } else if (dtype == BR_F16) {
        gelu_scalar<__half><<<grid_for(n, kBlock), kBlock, 0, st>>>((const __half*)dy, (const __half*)x, nullptr,
                                                                   (__half*)dx, n, 1, true);
    } else {
        return BR_ERR_TODO;
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

size_t br_hip_bias_gelu_bwd_workspace(int64_t rows, int64_t cols) { return br_hip_colsum_workspace(rows, cols); }

// Rows and columns that a single launch owns with its sums (owner_lanes): the copy is one more store there, in the two
// launches of larger sizes, where the products around fill the chip one at a time, nothing asks for it.
int br_hip_bias_gelu_bwd_copies(int64_t rows, int64_t cols) {
    return rows > 0 && cols > 0 && owner_lanes(rows, cols, 2, kOwnBiasGelu) != 0;
}

int br_hip_bias_gelu_bwd_copy(const void* dy, const void* x, const float* bias, void* dx, float* dbias, void* dy_copy, int dtype,
                              int64_t rows, int64_t cols, float dbias_scale, br_stream_t stream) {
    if (rows < 0 || cols <= 0) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!dy || !x) return BR_ERR_INPUT;
    if (!dx || !dbias || !dy_copy || dy_copy == dy || dy_copy == dx || dy_copy == x) return BR_ERR_OUTPUT;
    if ((dtype != BR_F16 && dtype != BR_BF16) || !br_hip_bias_gelu_bwd_copies(rows, cols) || !aligned16(dy) || !aligned16(x) ||
        !aligned16(dx) || !aligned16(dy_copy))
        return BR_ERR_TODO;
    const int lanes = owner_lanes(rows, cols, 2, kOwnBiasGelu);
    hipStream_t st = as_stream(stream);
    if (dtype == BR_F16)
        return colsum_owner_launch<2>(lanes, OwnBiasGeluBwd<__half, 8>{(const __half*)dy, (const __half*)x, bias, (__half*)dx,
                                                                       (__half*)dy_copy}, dbias, rows, cols, dbias_scale, st);
    return colsum_owner_launch<2>(lanes, OwnBiasGeluBwd<__hip_bfloat16, 8>{(const __hip_bfloat16*)dy, (const __hip_bfloat16*)x, bias,
                                                                           (__hip_bfloat16*)dx, (__hip_bfloat16*)dy_copy},
                                  dbias, rows, cols, dbias_scale, st);
}

int br_hip_bias_gelu_bwd(const void* dy, const void* x, const float* bias, void* dx, float* dbias, int dtype,
                         int64_t rows, int64_t cols, float dbias_scale, void* workspace, size_t workspace_bytes,
                         br_stream_t stream) {
    if (rows < 0 || cols <= 0) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!dy || !x) return BR_ERR_INPUT;
    if (!dx) return BR_ERR_OUTPUT;
    if (dtype != BR_F32 && dtype != BR_F16 && dtype != BR_BF16) return BR_ERR_TODO;
    hipStream_t st = as_stream(stream);
    const int rpb = strip_rows(rows);
    const int groups = (int)((rows + rpb - 1) / rpb);
    float* partial = nullptr;
    if (dbias) {
        if (!workspace || workspace_bytes < br_hip_bias_gelu_bwd_workspace(rows, cols)) return BR_ERR_ATTR;
        partial = (float*)workspace;
    }
    const bool al = aligned16(dy) && aligned16(x) && aligned16(dx);
    if (const int lanes = dbias && al ? owner_lanes(rows, cols, dtype == BR_F32 ? 4 : 2, kOwnBiasGelu) : 0) {
        // gradient and bias gradient from one launch
        if (dtype == BR_F32)
            return colsum_owner_launch<2>(lanes, OwnBiasGeluBwd<float, 4>{(const float*)dy, (const float*)x, bias, (float*)dx, nullptr},
                                          dbias, rows, cols, dbias_scale, st);
        if (dtype == BR_F16)
            return colsum_owner_launch<2>(lanes, OwnBiasGeluBwd<__half, 8>{(const __half*)dy, (const __half*)x, bias, (__half*)dx, nullptr},
                                          dbias, rows, cols, dbias_scale, st);
        return colsum_owner_launch<2>(lanes, OwnBiasGeluBwd<__hip_bfloat16, 8>{(const __hip_bfloat16*)dy, (const __hip_bfloat16*)x,
                                                                        bias, (__hip_bfloat16*)dx, nullptr},
                                      dbias, rows, cols, dbias_scale, st);
    }
    if (dtype == BR_F32 && al && cols % 4 == 0) {
        dim3 grid((unsigned)((cols / 4 + kBlock - 1) / kBlock), (unsigned)groups);
        bias_gelu_bwd_kernel<float, 4><<<grid, kBlock, 0, st>>>((const float*)dy, (const float*)x, bias,
                                                                 (float*)dx, partial, rows, cols, rpb);
    } else if (dtype == BR_F16 && al && cols % 8 == 0) {
        dim3 grid((unsigned)((cols / 8 + kBlock - 1) / kBlock), (unsigned)groups);
        bias_gelu_bwd_kernel<__half, 8><<<grid, kBlock, 0, st>>>((const __half*)dy, (const __half*)x, bias,
                                                                  (__half*)dx, partial, rows, cols, rpb);
    } else if (dtype == BR_BF16 && al && cols % 8 == 0) {
        dim3 grid((unsigned)((cols / 8 + kBlock - 1) / kBlock), (unsigned)groups);
        bias_gelu_bwd_kernel<__hip_bfloat16, 8><<<grid, kBlock, 0, st>>>((const __hip_bfloat16*)dy,
                                                                         (const __hip_bfloat16*)x, bias,
                                                                         (__hip_bfloat16*)dx, partial, rows, cols, rpb);
    } else if (dtype == BR_BF16) {
        return BR_ERR_TODO;
    } else {
        // unaligned shapes: elementwise pass, then a separate column sum of dx
        const int64_t n = rows * cols;
        if (dtype == BR_F32)
            gelu_scalar<float><<<grid_for(n, kBlock), kBlock, 0, st>>>((const float*)dy, (const float*)x, bias,
                                                                      (float*)dx, n, cols, true);
        else
            gelu_scalar<__half><<<grid_for(n, kBlock), kBlock, 0, st>>>((const __half*)dy, (const __half*)x,
                                                                       bias, (__half*)dx, n, cols, true);
        BR_HIP_LAUNCH_CHECK();
        if (dbias) return br_hip_colsum(dx, dtype, dbias, rows, cols, dbias_scale, workspace, workspace_bytes, stream);
        return BR_OK;
    }
    BR_HIP_LAUNCH_CHECK();
    if (dbias) return colsum_finish(partial, dbias, groups, cols, dbias_scale, st);
    return BR_OK;
}

size_t br_hip_colsum_workspace(int64_t rows, int64_t cols) {
    if (rows <= 0 || cols <= 0) return 0;
    const int rpb = strip_rows(rows);
    const size_t strips = (size_t)((rows + rpb - 1) / rpb) * (size_t)cols * sizeof(float);
    const size_t vec = (size_t)kMaxColsumGroups * (size_t)cols * sizeof(float);
    return strips > vec ? strips : vec;
}

int br_hip_colsum(const void* x, int dtype, float* out, int64_t rows, int64_t cols, float out_scale, void* workspace,
                  size_t workspace_bytes, br_stream_t stream) {
    if (rows < 0 || cols <= 0) return BR_ERR_ATTR;
    if (!out) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    if (rows == 0) return br_hip_fill(out, BR_F32, 0.f, cols, stream);
    if (!x) return BR_ERR_INPUT;
    if (!workspace || workspace_bytes < br_hip_colsum_workspace(rows, cols)) return BR_ERR_ATTR;
    if (dtype != BR_F32 && dtype != BR_F16 && dtype != BR_BF16) return BR_ERR_TODO;
    float* partial = (float*)workspace;
    const int vec = dtype == BR_F32 ? 4 : 8;
    if (cols % vec == 0 && aligned16(x) && (cols * (dtype == BR_F32 ? 4 : 2)) % 16 == 0) {
        if (const int lanes = owner_lanes(rows, cols, dtype == BR_F32 ? 4 : 2, kOwnSum)) {
            if (dtype == BR_F32) return colsum_owner_launch<4>(lanes, OwnPlain<float, 4>{(const float*)x}, out, rows, cols, out_scale, st);
            if (dtype == BR_F16) return colsum_owner_launch<4>(lanes, OwnPlain<__half, 8>{(const __half*)x}, out, rows, cols, out_scale, st);
            return colsum_owner_launch<4>(lanes, OwnPlain<__hip_bfloat16, 8>{(const __hip_bfloat16*)x}, out, rows, cols, out_scale, st);
        }
        const int64_t blocks_x = (cols / vec + kBlock - 1) / kBlock;
        const int rpb = colsum_vec_rows_per_block(rows, blocks_x);
        const int groups = (int)((rows + rpb - 1) / rpb);
        const dim3 grid((unsigned)blocks_x, (unsigned)groups);
        if (dtype == BR_F32)
            colsum_partial_vec<float, 4><<<grid, kBlock, 0, st>>>((const float*)x, partial, rows, cols, rpb);
        else if (dtype == BR_F16)
            colsum_partial_vec<__half, 8><<<grid, kBlock, 0, st>>>((const __half*)x, partial, rows, cols, rpb);
        else
            colsum_partial_vec<__hip_bfloat16, 8><<<grid, kBlock, 0, st>>>((const __hip_bfloat16*)x, partial, rows, cols, rpb);
        BR_HIP_LAUNCH_CHECK();
        return colsum_finish(partial, out, groups, cols, out_scale, st);
    }
    const int rpb = strip_rows(rows);
    const int groups = (int)((rows + rpb - 1) / rpb);
    dim3 grid((unsigned)((cols + kBlock - 1) / kBlock), (unsigned)groups);
    if (dtype == BR_F32)
        colsum_partial<float><<<grid, kBlock, 0, st>>>((const float*)x, partial, rows, cols, rpb);
    else if (dtype == BR_F16)
        colsum_partial<__half><<<grid, kBlock, 0, st>>>((const __half*)x, partial, rows, cols, rpb);
    else
        colsum_partial<__hip_bfloat16><<<grid, kBlock, 0, st>>>((const __hip_bfloat16*)x, partial, rows, cols, rpb);
    BR_HIP_LAUNCH_CHECK();
    return colsum_finish(partial, out, groups, cols, out_scale, st);
}

int br_hip_colsum_cast(const float* x, float* out, void* x16, int x16_dtype, int64_t rows, int64_t cols,
                       float out_scale, void* workspace, size_t workspace_bytes, br_stream_t stream) {
    if (rows <= 0 || cols <= 0) return BR_ERR_ATTR;
    if (!x) return BR_ERR_INPUT;
    if (!out || !x16) return BR_ERR_OUTPUT;
    if (x16_dtype != BR_F16 && x16_dtype != BR_BF16) return BR_ERR_TODO;
    if (cols % 4 != 0 || !aligned16(x) || (reinterpret_cast<uintptr_t>(x16) & 7u) != 0) return BR_ERR_TODO;
    if (!workspace || workspace_bytes < br_hip_colsum_workspace(rows, cols)) return BR_ERR_ATTR;
    hipStream_t st = as_stream(stream);
    if (const int lanes = owner_lanes(rows, cols, 4, kOwnSum)) {
        if (x16_dtype == BR_F16) return colsum_owner_launch<4>(lanes, OwnCast<__half>{x, (__half*)x16}, out, rows, cols, out_scale, st);
        return colsum_owner_launch<4>(lanes, OwnCast<__hip_bfloat16>{x, (__hip_bfloat16*)x16}, out, rows, cols, out_scale, st);
    }
    float* partial = (float*)workspace;
    const int64_t blocks_x = (cols / 4 + kBlock - 1) / kBlock;
    const int rpb = colsum_vec_rows_per_block(rows, blocks_x);
    const int groups = (int)((rows + rpb - 1) / rpb);
    dim3 grid((unsigned)blocks_x, (unsigned)groups);
    if (x16_dtype == BR_F16)
        colsum_cast_partial<__half><<<grid, kBlock, 0, st>>>(x, partial, (__half*)x16, rows, cols, rpb);
    else
        colsum_cast_partial<__hip_bfloat16><<<grid, kBlock, 0, st>>>(x, partial, (__hip_bfloat16*)x16, rows, cols, rpb);
    BR_HIP_LAUNCH_CHECK();
    return colsum_finish(partial, out, groups, cols, out_scale, st);
}

int br_hip_pack_colsum(const float* const* x, int count, float* out, void* packed, int packed_dtype, int64_t rows,
                       int64_t cols, float out_scale, br_stream_t stream) {
    if (rows <= 0 || cols <= 0 || count <= 0) return BR_ERR_ATTR;
    if (!x) return BR_ERR_INPUT;
    if (!out || !packed) return BR_ERR_OUTPUT;
    if (count > kPacked || cols % 8 != 0 || !aligned16(packed) || cols > (1 << 24)) return BR_ERR_TODO;
    PackSet set = {};
    for (int i = 0; i < count; i++) {
        if (!x[i]) return BR_ERR_INPUT;
        if (!aligned16(x[i])) return BR_ERR_TODO;
        set.x[i] = x[i];
    }
    hipStream_t st = as_stream(stream);
    if (packed_dtype == BR_F32) return pack_colsum<float>(set, count, out, packed, rows, cols, out_scale, st);
    if (packed_dtype == BR_F16) return pack_colsum<__half>(set, count, out, packed, rows, cols, out_scale, st);
    if (packed_dtype == BR_BF16) return pack_colsum<__hip_bfloat16>(set, count, out, packed, rows, cols, out_scale, st);
    return BR_ERR_TODO;
}

namespace {
// The gradient and its copy with partial column sums of strips in `partial`; returns the number of strips.
int gelu_bwd_strips(const float* dy, const float* x, float* dx, float* partial, void* dx16, int dx16_dtype, int64_t rows, int64_t cols,
                    hipStream_t st) {
    // same strips as br_hip_colsum_cast, hence the same summation order
    const int64_t blocks_x = (cols / 4 + kBlock - 1) / kBlock;
    const int rpb = colsum_vec_rows_per_block(rows, blocks_x);
    const int groups = (int)((rows + rpb - 1) / rpb);
    dim3 grid((unsigned)blocks_x, (unsigned)groups);
    if (dx16_dtype == BR_F16)
        gelu_bwd_colsum_cast_partial<__half><<<grid, kBlock, 0, st>>>(dy, x, dx, partial, (__half*)dx16, rows, cols, rpb);
    else
        gelu_bwd_colsum_cast_partial<__hip_bfloat16><<<grid, kBlock, 0, st>>>(dy, x, dx, partial, (__hip_bfloat16*)dx16, rows, cols, rpb);
    return groups;
}
int gelu_bwd_cast_checks(const float* dy, const float* x, float* dx, float* out, void* dx16, int dx16_dtype, int64_t rows, int64_t cols,
                         void* workspace, size_t workspace_bytes) {
    if (rows <= 0 || cols <= 0) return BR_ERR_ATTR;
    if (!dy || !x) return BR_ERR_INPUT;
    if (!dx || !out || !dx16) return BR_ERR_OUTPUT;
    if (dx16_dtype != BR_F16 && dx16_dtype != BR_BF16) return BR_ERR_TODO;
    if (cols % 4 != 0 || !aligned16(dy) || !aligned16(x) || !aligned16(dx) || (reinterpret_cast<uintptr_t>(dx16) & 7u) != 0)
        return BR_ERR_TODO;
    if (!workspace || workspace_bytes < br_hip_colsum_workspace(rows, cols)) return BR_ERR_ATTR;
    return BR_OK;
}
}  // namespace

int br_hip_gelu_bwd_colsum_cast(const float* dy, const float* x, float* dx, float* out, void* dx16, int dx16_dtype,
                                int64_t rows, int64_t cols, float out_scale, void* workspace, size_t workspace_bytes,
                                br_stream_t stream) {
    const int rc = gelu_bwd_cast_checks(dy, x, dx, out, dx16, dx16_dtype, rows, cols, workspace, workspace_bytes);
    if (rc != BR_OK) return rc;
    hipStream_t st = as_stream(stream);
    if (const int lanes = owner_lanes(rows, cols, 4, kOwnSum)) {
        if (dx16_dtype == BR_F16)
            return colsum_owner_launch<2>(lanes, OwnGeluBwdCast<__half>{dy, x, dx, (__half*)dx16}, out, rows, cols, out_scale, st);
        return colsum_owner_launch<2>(lanes, OwnGeluBwdCast<__hip_bfloat16>{dy, x, dx, (__hip_bfloat16*)dx16}, out, rows, cols,
                                      out_scale, st);
    }
    float* partial = (float*)workspace;
    const int groups = gelu_bwd_strips(dy, x, dx, partial, dx16, dx16_dtype, rows, cols, st);
    BR_HIP_LAUNCH_CHECK();
    return colsum_finish(partial, out, groups, cols, out_scale, st);
}

int br_hip_gelu_bwd_cast_sums(const float* dy, const float* x, float* dx, float* out, void* dx16, int dx16_dtype, int64_t rows,
                              int64_t cols, float out_scale, br_partial_sums* later, void* workspace, size_t workspace_bytes,
                              br_stream_t stream) {
    if (!later) return BR_ERR_OUTPUT;
    const int rc = gelu_bwd_cast_checks(dy, x, dx, out, dx16, dx16_dtype, rows, cols, workspace, workspace_bytes);
    if (rc != BR_OK) return rc;
    if (!aligned16(out) || !aligned16(workspace)) return BR_ERR_TODO;
    *later = br_partial_sums{};
    const int groups = gelu_bwd_strips(dy, x, dx, (float*)workspace, dx16, dx16_dtype, rows, cols, as_stream(stream));
    BR_HIP_LAUNCH_CHECK();
    later->partials = (const float*)workspace;
    later->arrays = 1;
    later->parts = groups;
    later->cols = cols;
    later->out[0] = out;
    later->scale = out_scale;
    return BR_OK;
}

int br_hip_transpose_0213_group(const void* const* x, void* const* y, int count, int elem_bytes, int64_t s0, int64_t s1,
                                int64_t s2, int64_t s3, br_stream_t stream) {
    if (count < 0) return BR_ERR_ATTR;
    if (count == 0) return BR_OK;
    if (!x) return BR_ERR_INPUT;
    if (!y) return BR_ERR_OUTPUT;
    bool together = count > 1 && count <= kTransposes && (elem_bytes == 2 || elem_bytes == 4) && s0 > 0 && s1 > 0 && s2 > 0 &&
                    s3 > 0 && fits_u32(s1) && fits_u32(s2) && fits_u32(s3) && s3 % (16 / elem_bytes) == 0;
    const uintptr_t bytes = together ? (uintptr_t)(s0 * s1 * s2 * s3) * (uintptr_t)elem_bytes : 0;
    const int64_t n16 = (int64_t)(bytes / 16);
    together = together && n16 <= (int64_t)1 << 28;   // each within a grid of its own size
    for (int i = 0; together && i < count; i++) {
        together = x[i] && y[i] && aligned16(x[i]) && aligned16(y[i]);
        // no tensor written is one that another of them reads or writes
        for (int j = 0; together && j < count; j++) {
            auto apart = [&](const void* a, const void* b) {
                const uintptr_t p = reinterpret_cast<uintptr_t>(a), q = reinterpret_cast<uintptr_t>(b);
                return p + bytes <= q || q + bytes <= p;
            };
            together = apart(y[i], x[j]) && (i == j || apart(y[i], y[j]));
        }
    }
    if (together) {
        TransposeSet set = {};
        for (int i = 0; i < count; i++) set.x[i] = (const uint4*)x[i], set.y[i] = (uint4*)y[i];
        transpose_0213_x16<<<dim3((unsigned)grid_for(n16, kBlock), (unsigned)count), kBlock, 0, as_stream(stream)>>>(
            set, n16, (unsigned)s1, (unsigned)s2, (unsigned)(s3 / (16 / elem_bytes)));
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
    for (int i = 0; i < count; i++) {
        const int rc = br_hip_transpose_0213(x[i], y[i], elem_bytes, s0, s1, s2, s3, stream);
        if (rc != BR_OK) return rc;
    }
    return BR_OK;
}

int br_hip_transpose_0213(const void* x, void* y, int elem_bytes, int64_t s0, int64_t s1, int64_t s2,
                          int64_t s3, br_stream_t stream) {
    if (s0 < 0 || s1 <= 0 || s2 <= 0 || s3 <= 0) return BR_ERR_ATTR;
    if (elem_bytes != 2 && elem_bytes != 4) return BR_ERR_ATTR;
    if (s0 == 0) return BR_OK;
    if (!x) return BR_ERR_INPUT;
    if (!y || x == y) return BR_ERR_OUTPUT;
    if (!fits_u32(s1) || !fits_u32(s2) || !fits_u32(s3)) return BR_ERR_ATTR;
    hipStream_t st = as_stream(stream);
    const int64_t n = s0 * s1 * s2 * s3;
    const int per16 = 16 / elem_bytes;
    if (s3 % per16 == 0 && aligned16(x) && aligned16(y)) {
        const int64_t n16 = n / per16;
        TransposeSet one = {};
        one.x[0] = (const uint4*)x;
        one.y[0] = (uint4*)y;
        transpose_0213_x16<<<grid_for(n16, kBlock), kBlock, 0, st>>>(one, n16, (unsigned)s1, (unsigned)s2,
                                                                    (unsigned)(s3 / per16));
    } else if (elem_bytes == 4) {
        transpose_0213_scalar<uint32_t><<<grid_for(n, kBlock), kBlock, 0, st>>>(
            (const uint32_t*)x, (uint32_t*)y, n, (unsigned)s1, (unsigned)s2, (unsigned)s3);
    } else {
        transpose_0213_scalar<uint16_t><<<grid_for(n, kBlock), kBlock, 0, st>>>(
            (const uint16_t*)x, (uint16_t*)y, n, (unsigned)s1, (unsigned)s2, (unsigned)s3);
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_embedding_gather(const void* table, const int32_t* ids, void* out, int elem_bytes, int64_t n,
                            int64_t hidden, int64_t vocab, br_stream_t stream) {
    if (n < 0 || hidden <= 0 || vocab <= 0 || (elem_bytes != 2 && elem_bytes != 4)) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!table || !ids) return BR_ERR_INPUT;
    if (!out) return BR_ERR_OUTPUT;
    if (n > 0x7fffffff) return BR_ERR_ATTR;
    hipStream_t st = as_stream(stream);
    const int64_t row_bytes = hidden * elem_bytes;
    if (row_bytes % 16 == 0 && aligned16(table) && aligned16(out))
        gather_rows_x16<<<(unsigned)n, kBlock, 0, st>>>((const uint4*)table, ids, (uint4*)out, row_bytes / 16,
                                                        vocab);
    else
        gather_rows_bytes<<<(unsigned)n, kBlock, 0, st>>>((const unsigned char*)table, ids, (unsigned char*)out,
                                                          row_bytes, vocab);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_embedding_gather_f32(const void* table, int table_dtype, const int32_t* ids, float* out, int64_t n,
                                int64_t hidden, int64_t vocab, br_stream_t stream) {
    if (n < 0 || hidden <= 0 || vocab <= 0) return BR_ERR_ATTR;
    if (table_dtype != BR_F16 && table_dtype != BR_BF16) return BR_ERR_TODO;
    if (n == 0) return BR_OK;
    if (!table || !ids) return BR_ERR_INPUT;
    if (!out) return BR_ERR_OUTPUT;
    if (n > 0xffffff) return BR_ERR_ATTR;
    hipStream_t st = as_stream(stream);
    if (table_dtype == BR_F16)
        gather_rows_f32<__half><<<(unsigned)n, kBlock, 0, st>>>((const __half*)table, ids, out, hidden, vocab);
    else
        gather_rows_f32<__hip_bfloat16><<<(unsigned)n, kBlock, 0, st>>>((const __hip_bfloat16*)table, ids, out, hidden, vocab);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_pick_rows(const float* x, const int64_t* rows, void* out, int out_dtype, int64_t n, int64_t cols,
                     br_stream_t stream) {
    if (n < 0 || cols < 0) return BR_ERR_ATTR;
    if (n == 0 || cols == 0) return BR_OK;
    if (!x || !rows) return BR_ERR_INPUT;
    if (!out) return BR_ERR_OUTPUT;
    for (int64_t i = 0; i < n; i++)
        if (rows[i] < 0) return BR_ERR_INPUT;
    hipStream_t st = as_stream(stream);
    if (out_dtype == BR_F32) return pick_rows<float>(x, rows, out, n, cols, st);
    if (out_dtype == BR_F16) return pick_rows<__half>(x, rows, out, n, cols, st);
    if (out_dtype == BR_BF16) return pick_rows<__hip_bfloat16>(x, rows, out, n, cols, st);
    return BR_ERR_TODO;
}

int br_hip_embedding_scatter_add(const float* dx, const int32_t* ids, float* grad, int64_t n, int64_t hidden,
                                 int64_t vocab, float dx_scale, br_stream_t stream) {
    if (n < 0 || hidden <= 0 || vocab <= 0 || n > 0x7fffffff) return BR_ERR_ATTR;
    if (n == 0) return BR_OK;
    if (!dx || !ids) return BR_ERR_INPUT;
    if (!grad || (const float*)grad == dx) return BR_ERR_OUTPUT;
    const int vec = hidden % 4 == 0 && aligned16(dx) && aligned16(grad) ? 4 : 1;
    const int64_t blocks = (hidden + (int64_t)kBlock * vec - 1) / ((int64_t)kBlock * vec);
    const dim3 grid((unsigned)n, (unsigned)(blocks < 65535 ? blocks : 65535));
    if (vec == 4)
        scatter_add_rows<4><<<grid, kBlock, 0, as_stream(stream)>>>(dx, ids, grad, (int)n, hidden, vocab, dx_scale);
    else
        scatter_add_rows<1><<<grid, kBlock, 0, as_stream(stream)>>>(dx, ids, grad, (int)n, hidden, vocab, dx_scale);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_alibi_table(float* alibi, int64_t heads, int64_t tokens, br_stream_t stream) {
    if (heads <= 0 || tokens <= 0 || heads > 65536) return BR_ERR_ATTR;
    if (!alibi) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    double* slopes = new double[heads];
    br_hip_alibi_slopes(slopes, heads);
    int rc = BR_OK;
    for (int64_t h0 = 0; h0 < heads && rc == BR_OK; h0 += kSlopeChunk) {
        SlopeChunk c;
        const int nh = (int)(heads - h0 < kSlopeChunk ? heads - h0 : kSlopeChunk);
        for (int i = 0; i < kSlopeChunk; i++) c.v[i] = i < nh ? slopes[h0 + i] : 0.0;
        alibi_table_kernel<<<grid_for((int64_t)nh * tokens, kBlock), kBlock, 0, st>>>(alibi, c, (int)h0, nh,
                                                                                      tokens);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = (int)e;
    }
    delete[] slopes;
    return rc;
}

int br_hip_xmask_table(const int32_t* mask, float* xmask, int64_t batch, int64_t tokens, br_stream_t stream) {
    if (batch < 0 || tokens <= 0 || tokens > 0x7fffffff || batch > 65535) return BR_ERR_ATTR;
    if (batch == 0) return BR_OK;
    if (!mask) return BR_ERR_INPUT;
    if (!xmask) return BR_ERR_OUTPUT;
    dim3 grid((unsigned)tokens, (unsigned)batch);
    xmask_table_kernel<<<grid, kBlock, 0, as_stream(stream)>>>(mask, xmask, tokens);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

}  // extern "C"
