// Softmax family for gfx950.
//
// Attention softmax (rows of a few hundred to a few thousand scores): one
// wave64 per row, the row held in registers, so HBM sees one read and one
// write; the ALiBi bias and the additive causal / padding mask are folded in
// either from their tables or analytically.
//
// Vocabulary log-softmax + NLL (rows of 250 880 logits, 1 MB each): one
// 1024-thread workgroup per row, a single online (max, sum) sweep with
// 128-bit loads; the backward re-reads the row and writes the gradient.
#include "common.hpp"

#include <float.h>

#include <initializer_list>

using namespace brk;

namespace {

constexpr int kBlock = 256;
constexpr int kRowsPerBlock = kBlock / kWave;  // one wave per row

enum MaskMode { kPlain = 0, kTables = 1, kAnalytic = 2 };

struct RowBias {
    const float* alibi;   // [heads, tk]            (kTables)
    const float* xmask;   // [batch, tq, tk]        (kTables)
    const double* slopes; // [heads]                (kAnalytic)
    const int32_t* valid; // [batch]                (kAnalytic)
    int heads, tq;
};

// Scores, probabilities and their gradients are read once and written once: streaming (non-temporal) accesses,
// measured at [4,32,512,512] fp32 on one box: forward 55.4 us plain, 54.5 with streaming loads, 51.0 with streaming
// stores too; backward 71 / 66.6 / 62.4.
// Rows are held in granules of G floats: four where rows are 16-byte aligned, two or one where an odd number of
// tokens leaves them on 8- or 4-byte boundaries (three sweeps over such a row by a workgroup took 30 us forward and
// 18 backward for the scores of 4 x 16 heads of 250 tokens; a row in one wave's registers takes 7 and 8).
template <int G>
struct Granule;
template <>
struct Granule<4> {
    static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
        const float4 t = load_stream(reinterpret_cast<const float4*>(p));
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    }
    static __device__ __forceinline__ void load_cached(const float* p, float (&v)[4]) {
        const float4 t = *reinterpret_cast<const float4*>(p);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    }
    static __device__ __forceinline__ void store(float* p, const float (&v)[4]) {
        store_stream(reinterpret_cast<float4*>(p), make_float4(v[0], v[1], v[2], v[3]));
    }
    static __device__ __forceinline__ float sum(const float (&v)[4]) { return (v[0] + v[1]) + (v[2] + v[3]); }
    static __device__ __forceinline__ float max(const float (&v)[4]) { return fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])); }
    // also pins v to the values that are stored (see store4_as16)
    static __device__ __forceinline__ void store16(const Copy16& c, int64_t at, float (&v)[4]) {
        float4 t = make_float4(v[0], v[1], v[2], v[3]);
        store4_as16(c, at / 4, t);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    }
};
template <>
struct Granule<2> {
    static __device__ __forceinline__ void load(const float* p, float (&v)[2]) {
        const float2 t = *reinterpret_cast<const float2*>(p);
        v[0] = t.x; v[1] = t.y;
    }
    static __device__ __forceinline__ void load_cached(const float* p, float (&v)[2]) { load(p, v); }
    static __device__ __forceinline__ void store(float* p, const float (&v)[2]) {
        *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
    }
    static __device__ __forceinline__ float sum(const float (&v)[2]) { return v[0] + v[1]; }
    static __device__ __forceinline__ float max(const float (&v)[2]) { return fmaxf(v[0], v[1]); }
    static __device__ __forceinline__ void store16(const Copy16& c, int64_t at, float (&v)[2]) {
        asm volatile("" : "+v"(v[0]), "+v"(v[1]));
        if (!c.base) return;
        auto bits = [&](float f) {
            return (unsigned)(c.bf16 ? __builtin_bit_cast(unsigned short, __float2bfloat16(f))
                                     : __builtin_bit_cast(unsigned short, __float2half_rn(f)));
        };
        static_cast<unsigned*>(c.base)[at / 2] = bits(v[0]) | (bits(v[1]) << 16);
    }
};
template <>
struct Granule<1> {
    static __device__ __forceinline__ void load(const float* p, float (&v)[1]) { v[0] = *p; }
    static __device__ __forceinline__ void load_cached(const float* p, float (&v)[1]) { v[0] = *p; }
    static __device__ __forceinline__ void store(float* p, const float (&v)[1]) { *p = v[0]; }
    static __device__ __forceinline__ float sum(const float (&v)[1]) { return v[0]; }
    static __device__ __forceinline__ float max(const float (&v)[1]) { return v[0]; }
    static __device__ __forceinline__ void store16(const Copy16&, int64_t, float (&)[1]) {}   // not offered at odd widths
};

// exp(x - m) for x <= m, via the hardware exp2
__device__ __forceinline__ float exp_sub(float x, float m) { return __expf(x - m); }

// VPL granules of G floats per lane; cols = G * granules <= 64 * G * VPL.
template <int VPL, int MODE, int G>
__global__ __launch_bounds__(kBlock) void softmax_fwd_wave(const float* __restrict__ x, float* __restrict__ y,
                                                            int64_t rows, int granules, RowBias rb, Copy16 y16) {
    using Gr = Granule<G>;
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    if (row >= rows) return;
    const float* xr = x + row * granules * G;
    float v[VPL][G];
#pragma unroll
    for (int i = 0; i < VPL; i++) {
        const int idx = lane + i * kWave;
        if (idx < granules) {
            Gr::load(xr + idx * G, v[i]);
        } else {
#pragma unroll
            for (int j = 0; j < G; j++) v[i][j] = -INFINITY;
        }
    }
    if (MODE != kPlain) {
        // row = (b * heads + h) * tq + q
        const int q = (int)(row % rb.tq);
        const int64_t bh = row / rb.tq;
        const int h = (int)(bh % rb.heads);
        const int64_t b = bh / rb.heads;
        if (MODE == kTables) {
            const float* ar = rb.alibi ? rb.alibi + (int64_t)h * granules * G : nullptr;
            const float* mr = rb.xmask ? rb.xmask + (b * rb.tq + q) * granules * G : nullptr;
#pragma unroll
            for (int i = 0; i < VPL; i++) {
                const int idx = lane + i * kWave;
                if (idx < granules) {
                    float t[G];
                    if (ar) {
                        Gr::load_cached(ar + idx * G, t);
#pragma unroll
                        for (int j = 0; j < G; j++) v[i][j] += t[j];
                    }
                    if (mr) {
                        Gr::load_cached(mr + idx * G, t);
#pragma unroll
                        for (int j = 0; j < G; j++) v[i][j] += t[j];
                    }
                }
            }
        } else {
            const double slope = rb.slopes[h];
            const int valid = rb.valid[b];
#pragma unroll
            for (int i = 0; i < VPL; i++) {
                const int idx = lane + i * kWave;
                if (idx < granules) {
#pragma unroll
                    for (int j = 0; j < G; j++) {
                        const int k = idx * G + j;
                        // same two additions, in the same order, as the table form
                        v[i][j] += (float)((double)k * 1.0 * slope);
                        v[i][j] += (k <= q && k < valid) ? 0.0f : -FLT_MAX;
                    }
                }
            }
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < VPL; i++) m = fmaxf(m, Gr::max(v[i]));
    m = wave_max(m);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; i++) {
#pragma unroll
        for (int j = 0; j < G; j++) v[i][j] = exp_sub(v[i][j], m);
        s += Gr::sum(v[i]);
    }
    s = wave_sum(s);
    const float inv = 1.0f / s;
    float* yr = y + row * granules * G;
#pragma unroll
    for (int i = 0; i < VPL; i++) {
        const int idx = lane + i * kWave;
        if (idx < granules) {
#pragma unroll
            for (int j = 0; j < G; j++) v[i][j] *= inv;
            Gr::store16(y16, (row * granules + idx) * G, v[i]);
            Gr::store(yr + idx * G, v[i]);
        }
    }
}

template <int VPL, int G>
__global__ __launch_bounds__(kBlock) void softmax_bwd_wave(const float* __restrict__ dy, const float* __restrict__ y,
                                                            float* __restrict__ dx, int64_t rows, int granules,
                                                            Copy16 dx16) {
    using Gr = Granule<G>;
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    if (row >= rows) return;
    const float* gr = dy + row * granules * G;
    const float* yr = y + row * granules * G;
    float g[VPL][G], p[VPL][G];
    float dot = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; i++) {
        const int idx = lane + i * kWave;
        float t[G];
        if (idx < granules) {
            Gr::load(gr + idx * G, g[i]);
            Gr::load(yr + idx * G, p[i]);
        } else {
#pragma unroll
            for (int j = 0; j < G; j++) g[i][j] = p[i][j] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < G; j++) t[j] = g[i][j] * p[i][j];
        dot += Gr::sum(t);
    }
    dot = wave_sum(dot);
#pragma unroll
    for (int i = 0; i < VPL; i++) {
        const int idx = lane + i * kWave;
        if (idx < granules) {
            float o[G];
#pragma unroll
            for (int j = 0; j < G; j++) o[j] = p[i][j] * (g[i][j] - dot);
            Gr::store16(dx16, (row * granules + idx) * G, o);
            if (dx) Gr::store(dx + (row * granules + idx) * G, o);  // dx == nullptr: only the 16-bit gradient is wanted
        }
    }
}

// Any width / alignment: one workgroup per row, three sweeps from global.
template <int MODE>
__global__ __launch_bounds__(kBlock) void softmax_fwd_generic(const float* x, float* y, int64_t cols, RowBias rb) {
    __shared__ float lds[2][kBlock / kWave];
    const int64_t row = blockIdx.x;
    const float* xr = x + row * cols;
    float* yr = y + row * cols;
    const int q = MODE != kPlain ? (int)(row % rb.tq) : 0;
    const int64_t bh = MODE != kPlain ? row / rb.tq : 0;
    const int h = MODE != kPlain ? (int)(bh % rb.heads) : 0;
    const int64_t b = MODE != kPlain ? bh / rb.heads : 0;
    auto value = [&](int64_t c) -> float {
        float v = xr[c];
        if (MODE == kTables) {
            if (rb.alibi) v += rb.alibi[(int64_t)h * cols + c];
            if (rb.xmask) v += rb.xmask[(b * rb.tq + q) * cols + c];
        } else if (MODE == kAnalytic) {
            v += (float)((double)c * 1.0 * rb.slopes[h]);
            v += (c <= q && c < rb.valid[b]) ? 0.0f : -FLT_MAX;
        }
        return v;
    };
    float m = -INFINITY;
    for (int64_t c = threadIdx.x; c < cols; c += kBlock) m = fmaxf(m, value(c));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) lds[0][threadIdx.x >> 6] = m;
    __syncthreads();
    m = lds[0][0];
    for (int w = 1; w < kBlock / kWave; w++) m = fmaxf(m, lds[0][w]);
    float s[1] = {0.f};
    for (int64_t c = threadIdx.x; c < cols; c += kBlock) s[0] += exp_sub(value(c), m);
    block_sum<1>(s, lds[1]);
    const float inv = 1.0f / s[0];
    // y may alias x: every element is read (by value()) only by the thread that overwrites it
    for (int64_t c = threadIdx.x; c < cols; c += kBlock) yr[c] = exp_sub(value(c), m) * inv;
}

__global__ __launch_bounds__(kBlock) void softmax_bwd_generic(const float* dy, const float* y, float* dx,
                                                               int64_t cols) {
    __shared__ float lds[kBlock / kWave];
    const int64_t row = blockIdx.x;
    float s[1] = {0.f};
    for (int64_t c = threadIdx.x; c < cols; c += kBlock) s[0] += dy[row * cols + c] * y[row * cols + c];
    block_sum<1>(s, lds);
    for (int64_t c = threadIdx.x; c < cols; c += kBlock)
        dx[row * cols + c] = y[row * cols + c] * (dy[row * cols + c] - s[0]);
}

// Floats per granule for rows of `cols` floats at these addresses (null ones do not count).  Never less than one: an
// address that is no multiple of four bytes is read float by float, as the workgroup-per-row kernel reads it.
int granule_of(int64_t cols, std::initializer_list<const void*> at) {
    int g = cols % 4 == 0 ? 4 : cols % 2 == 0 ? 2 : 1;
    for (const void* p : at)
        while (g > 1 && reinterpret_cast<uintptr_t>(p) % (4 * g) != 0) g /= 2;
    return g;
}
constexpr int64_t kMaxRegisterRow = 2048;   // floats of a row in granules of fewer than four (32 registers of a lane)

template <int MODE, int G>
void launch_softmax_fwd_wave(const float* x, float* y, int64_t rows, int64_t cols, const RowBias& rb, hipStream_t st,
                             Copy16 y16) {
    const int granules = (int)(cols / G);
    const unsigned grid = (unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
    const int vpl = (granules + kWave - 1) / kWave;
    if (vpl <= 1) softmax_fwd_wave<1, MODE, G><<<grid, kBlock, 0, st>>>(x, y, rows, granules, rb, y16);
    else if (vpl <= 2) softmax_fwd_wave<2, MODE, G><<<grid, kBlock, 0, st>>>(x, y, rows, granules, rb, y16);
    else if (vpl <= 4) softmax_fwd_wave<4, MODE, G><<<grid, kBlock, 0, st>>>(x, y, rows, granules, rb, y16);
    else if (vpl <= 8) softmax_fwd_wave<8, MODE, G><<<grid, kBlock, 0, st>>>(x, y, rows, granules, rb, y16);
    else if (vpl <= 16) softmax_fwd_wave<16, MODE, G><<<grid, kBlock, 0, st>>>(x, y, rows, granules, rb, y16);
    else if constexpr (G == 1) softmax_fwd_wave<32, MODE, G><<<grid, kBlock, 0, st>>>(x, y, rows, granules, rb, y16);
}

template <int MODE>
int launch_softmax_fwd(const float* x, float* y, int64_t rows, int64_t cols, const RowBias& rb, hipStream_t st,
                       Copy16 y16 = Copy16{nullptr, 0}) {
    const int g = MODE == kTables ? granule_of(cols, {x, y, rb.alibi, rb.xmask}) : granule_of(cols, {x, y});
    if (g == 4 && cols <= 256 * 16) {
        launch_softmax_fwd_wave<MODE, 4>(x, y, rows, cols, rb, st, y16);
    } else if (g == 2 && cols <= kMaxRegisterRow) {
        launch_softmax_fwd_wave<MODE, 2>(x, y, rows, cols, rb, st, y16);
    } else {
        if (y16.base) return BR_ERR_TODO;  // the copy is written two or four values at a time
        if (cols <= kMaxRegisterRow) launch_softmax_fwd_wave<MODE, 1>(x, y, rows, cols, rb, st, y16);
        else softmax_fwd_generic<MODE><<<(unsigned)rows, kBlock, 0, st>>>(x, y, cols, rb);
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// Granule of the one-wave-per-row backward, 0 where rows do not fit it.
int softmax_bwd_granule(int64_t cols, const void* dy, const void* y, const void* dx) {
    const int g = granule_of(cols, {dy, y, dx});
    return cols <= kMaxRegisterRow ? g : 0;
}

template <int G>
void launch_softmax_bwd_granules(const float* dy, const float* y, float* dx, Copy16 dx16, int64_t rows, int64_t cols,
                                 hipStream_t st) {
    const int granules = (int)(cols / G);
    const unsigned grid = (unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
    const int vpl = (granules + kWave - 1) / kWave;
    if (vpl <= 1) softmax_bwd_wave<1, G><<<grid, kBlock, 0, st>>>(dy, y, dx, rows, granules, dx16);
    else if (vpl <= 2) softmax_bwd_wave<2, G><<<grid, kBlock, 0, st>>>(dy, y, dx, rows, granules, dx16);
    else if (vpl <= 4) softmax_bwd_wave<4, G><<<grid, kBlock, 0, st>>>(dy, y, dx, rows, granules, dx16);
    else if (vpl <= 8) softmax_bwd_wave<8, G><<<grid, kBlock, 0, st>>>(dy, y, dx, rows, granules, dx16);
    else if constexpr (G <= 2) {
        if (vpl <= 16) softmax_bwd_wave<16, G><<<grid, kBlock, 0, st>>>(dy, y, dx, rows, granules, dx16);
        else if constexpr (G == 1) softmax_bwd_wave<32, G><<<grid, kBlock, 0, st>>>(dy, y, dx, rows, granules, dx16);
    }
}
int launch_softmax_bwd_wave(int g, const float* dy, const float* y, float* dx, Copy16 dx16, int64_t rows, int64_t cols,
                            hipStream_t st) {
    if (g == 4) launch_softmax_bwd_granules<4>(dy, y, dx, dx16, rows, cols, st);
    else if (g == 2) launch_softmax_bwd_granules<2>(dy, y, dx, dx16, rows, cols, st);
    else launch_softmax_bwd_granules<1>(dy, y, dx, dx16, rows, cols, st);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// ------------------------------------------------- vocabulary log-softmax
constexpr int kVBlock = 1024;
constexpr int kVWaves = kVBlock / kWave;

struct MaxSum {
    float m, s;
};

__device__ __forceinline__ MaxSum combine(MaxSum a, MaxSum b) {
    const float m = fmaxf(a.m, b.m);
    MaxSum r;
    r.m = m;
    r.s = a.s * __expf(a.m - m) + b.s * __expf(b.m - m);
    return r;
}

// Online (max, sum) over one row; every thread returns the row's logsumexp.  Quads from the row's first 16-byte boundary on, up to
// three values before and after them one by one: rows of an odd vocabulary start anywhere ([200 x 32001] 13.8 -> 8.4 us).  AHEAD
// quads of a thread are on their way at a time: four where a CU has one row, one where others fill the time.
template <int AHEAD>
__device__ __forceinline__ float row_logsumexp(const float* __restrict__ lr, int64_t vocab, MaxSum* lds) {
    // The lowest number rather than minus infinity: what is masked with the latter then adds nothing, also where a thread has met
    // nothing else yet, and no difference is one of infinities.
    MaxSum t;
    t.m = -FLT_MAX;
    t.s = 0.f;
    auto quad = [&](const float4& v) {
        const float m4 = fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w));
        if (m4 > t.m) {
            t.s *= __expf(t.m - m4);
            t.m = m4;
        }
        t.s += (__expf(v.x - t.m) + __expf(v.y - t.m)) + (__expf(v.z - t.m) + __expf(v.w - t.m));
    };
    int64_t head = (int64_t)(-(reinterpret_cast<uintptr_t>(lr) >> 2) & 3);
    if (head > vocab) head = vocab;
    const float4* l4 = reinterpret_cast<const float4*>(lr + head);
    const int64_t n4 = (vocab - head) / 4;
    int64_t i = threadIdx.x;
    if constexpr (AHEAD > 1) {
        for (; i + (AHEAD - 1) * kVBlock < n4; i += AHEAD * kVBlock) {
            float4 v[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; u++) v[u] = load_stream(l4 + i + u * kVBlock);
#pragma unroll
            for (int u = 0; u < AHEAD; u++) quad(v[u]);
        }
    }
    for (; i < n4; i += kVBlock) quad(load_stream(l4 + i));
    if (threadIdx.x < vocab - 4 * n4) {
        const float v = lr[threadIdx.x < head ? threadIdx.x : threadIdx.x + 4 * n4];
        if (v > t.m) {
            t.s *= __expf(t.m - v);
            t.m = v;
        }
        t.s += __expf(v - t.m);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        MaxSum o;
        o.m = __shfl_xor(t.m, off, kWave);
        o.s = __shfl_xor(t.s, off, kWave);
        t = combine(t, o);
    }
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = t;
    __syncthreads();
    MaxSum r = lds[0];
    for (int w = 1; w < kVWaves; w++) r = combine(r, lds[w]);
    return r.m + __logf(r.s);
}

template <int AHEAD>
__global__ __launch_bounds__(kVBlock) void nll_fwd_kernel(const float* __restrict__ logits,
                                                           const int32_t* __restrict__ target,
                                                           const int32_t* __restrict__ keep,
                                                           float* __restrict__ lse, float* __restrict__ row_logp,
                                                           int64_t vocab) {
    __shared__ MaxSum lds[kVWaves];
    const int64_t row = blockIdx.x;
    const float* lr = logits + row * vocab;
    const int32_t t = target[row];
    const bool valid = keep[row] != 0 && t >= 0 && (int64_t)t < vocab;
    const float of_target = valid ? lr[t] : 0.f;
    const float l = row_logsumexp<AHEAD>(lr, vocab, lds);
    if (threadIdx.x == 0) {
        lse[row] = l;
        row_logp[row] = valid ? of_target - l : 0.f;
    }
}

// result[0] = sum(row_logp) / count, result[1] = count; one workgroup,
// fixed summation order.
__global__ __launch_bounds__(kVBlock) void nll_reduce_kernel(const float* __restrict__ row_logp,
                                                              const int32_t* __restrict__ keep,
                                                              float* __restrict__ result, int64_t rows) {
    __shared__ float lds[2 * kVWaves];
    float v[2] = {0.f, 0.f};
    for (int64_t r = threadIdx.x; r < rows; r += kVBlock) {
        v[0] += row_logp[r];
        v[1] += keep[r] != 0 ? 1.f : 0.f;
    }
    block_sum<2>(v, lds);
    if (threadIdx.x == 0) {
        result[0] = v[1] > 0.f ? v[0] / v[1] : 0.f;
        result[1] = v[1];
    }
}

template <typename OUT>
__device__ __forceinline__ void store4(OUT* p, float a, float b, float c, float d);
template <>
__device__ __forceinline__ void store4<float>(float* p, float a, float b, float c, float d) {
    store_stream(reinterpret_cast<float4*>(p), make_float4(a, b, c, d));
}
template <>
__device__ __forceinline__ void store4<__half>(__half* p, float a, float b, float c, float d) {
    half4 h;
    h.v[0] = __floats2half2_rn(a, b);
    h.v[1] = __floats2half2_rn(c, d);
    *reinterpret_cast<half4*>(p) = h;
}
template <typename OUT>
__device__ __forceinline__ OUT cvt_out(float v);
template <>
__device__ __forceinline__ float cvt_out<float>(float v) { return v; }
template <>
__device__ __forceinline__ __half cvt_out<__half>(float v) { return __float2half_rn(v); }
template <>
__device__ __forceinline__ void store4<__hip_bfloat16>(__hip_bfloat16* p, float a, float b, float c, float d) {
    auto bits = [](float v) { return (unsigned)__builtin_bit_cast(unsigned short, __float2bfloat16(v)); };
    *reinterpret_cast<uint2*>(p) = make_uint2(bits(a) | (bits(b) << 16), bits(c) | (bits(d) << 16));
}
template <>
__device__ __forceinline__ __hip_bfloat16 cvt_out<__hip_bfloat16>(float v) { return __float2bfloat16(v); }

template <typename OUT>
__global__ __launch_bounds__(kVBlock) void nll_bwd_kernel(const float* logits, const int32_t* __restrict__ target,
                                                           const int32_t* __restrict__ keep,
                                                           const float* __restrict__ lse, OUT* dlogits, float scale,
                                                           int64_t vocab, bool vec_ok) {
    const int64_t row = blockIdx.x;
    const float* lr = logits + row * vocab;
    OUT* dr = dlogits + row * vocab;
    const int32_t t = target[row];
    const bool on = keep[row] != 0 && t >= 0 && (int64_t)t < vocab;
    if (!on) {
        // rows without a label get an all-zero gradient and are never read
        if (vec_ok) {
            for (int64_t i = threadIdx.x; i < vocab / 4; i += kVBlock) store4<OUT>(dr + i * 4, 0.f, 0.f, 0.f, 0.f);
        } else {
            for (int64_t i = threadIdx.x; i < vocab; i += kVBlock) dr[i] = cvt_out<OUT>(0.f);
        }
        return;
    }
    const float l = lse[row];
    if (vec_ok) {
        const float4* l4 = reinterpret_cast<const float4*>(lr);
        const int64_t t4 = t >> 2;
        for (int64_t i = threadIdx.x; i < vocab / 4; i += kVBlock) {
            const float4 v = load_stream(l4 + i);
            float e[4] = {__expf(v.x - l), __expf(v.y - l), __expf(v.z - l), __expf(v.w - l)};
            if (i == t4) e[t & 3] -= 1.0f;
            store4<OUT>(dr + i * 4, e[0] * scale, e[1] * scale, e[2] * scale, e[3] * scale);
        }
    } else {
        for (int64_t i = threadIdx.x; i < vocab; i += kVBlock) {
            float e = __expf(lr[i] - l);
            if (i == t) e -= 1.0f;
            dr[i] = cvt_out<OUT>(e * scale);
        }
    }
}

// The same gradient with one quad per thread and the workgroups in memory order (blockIdx.x along a row, blockIdx.y
// over the rows): given lse the gradient is element-wise, and a launch that sweeps logits and gradient front to back
// as one stream moves 6.4 TB/s where a workgroup per 1 MB row moves 5.3 (see grid_for).  Same arithmetic, same bits.
// Rows of an odd vocabulary start off 16-byte boundaries, of the logits and of the gradient by as many elements: a row's quads
// begin at its first boundary, and the threads behind them take the up to six values around them one by one ([200 x 32001] to
// fp16 13.7 -> 10.0 us).  WHOLE: a multiple of four, where there are none.
#ifndef BR_NLL_BWD_FLAT
#define BR_NLL_BWD_FLAT 1
#endif
constexpr int kFlatBlock = 256;
template <typename OUT, bool WHOLE>
__global__ __launch_bounds__(kFlatBlock) void nll_bwd_flat_kernel(const float* logits, const int32_t* __restrict__ target,
                                                                  const int32_t* __restrict__ keep,
                                                                  const float* __restrict__ lse, OUT* dlogits,
                                                                  float scale, int64_t vocab) {
    const int64_t row = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * kFlatBlock + threadIdx.x;   // quad of the row
    int64_t head = WHOLE ? 0 : -(row * vocab) & 3;
    if (!WHOLE && head > vocab) head = vocab;
    const int64_t n4 = (vocab - head) / 4, apart = i - n4;   // what is not in quads comes behind them
    if (apart >= (WHOLE ? 0 : vocab - 4 * n4)) return;
    const int32_t t = target[row];
    const bool on = keep[row] != 0 && t >= 0 && (int64_t)t < vocab;
    const float l = lse[row];
    if (!WHOLE && apart >= 0) {
        const int64_t c = apart < head ? apart : apart + 4 * n4;
        float e = on ? __expf(logits[row * vocab + c] - l) : 0.f;
        if (on && c == t) e -= 1.0f;
        dlogits[row * vocab + c] = cvt_out<OUT>(on ? e * scale : 0.f);
        return;
    }
    const int64_t c = head + 4 * i;
    OUT* dr = dlogits + row * vocab + c;
    if (!on) {
        store4<OUT>(dr, 0.f, 0.f, 0.f, 0.f);   // rows without a label are not read
        return;
    }
    const float4 v = load_stream(reinterpret_cast<const float4*>(logits + row * vocab + c));
    float e[4] = {__expf(v.x - l), __expf(v.y - l), __expf(v.z - l), __expf(v.w - l)};
    if (WHOLE ? i == (t >> 2) : (uint64_t)(t - c) < 4) e[WHOLE ? t & 3 : t - c] -= 1.0f;
    store4<OUT>(dr, e[0] * scale, e[1] * scale, e[2] * scale, e[3] * scale);
}

template <typename OUT>
void launch_nll_bwd(const float* logits, const int32_t* target, const int32_t* keep, const float* lse, OUT* dlogits,
                    float scale, int64_t rows, int64_t vocab, bool aligned, hipStream_t st) {
    const bool vec_ok = aligned && vocab % 4 == 0;
    const int64_t blocks_x = (vocab / 4 + (vocab % 4 ? 6 : 0) + kFlatBlock - 1) / kFlatBlock;
    // Rows of an odd vocabulary that the caches hold (256 MB of them) stay a workgroup each, two to a CU, where they fill three
    // quarters of such rounds: memory's order does not matter there, and starting a workgroup for every 4 KB does.  Flat / a
    // workgroup a row, us: [512 x 32001] to fp16 21.2 / 17.1, [1024 x 16001] to fp32 22.6 / 21.1, in place [512 x 8001] 7.3 / 6.0,
    // [2048 x 24001] 63.7 / 57.5; but [1024 x 50257] to fp32, 412 MB, 67 / 97, [300 x 32001], 0.59 of a round, 14.4 / 15.7, [2048 x
    // 3001] to fp16 8.1 / 9.3.  (432 sizes of 3001 to 120001 words: 10028 flat, 9689 by this rule, 9672 by the best of each.)
    const int64_t round = 512, rounds = (rows + round - 1) / round;
    const int64_t touched = rows * vocab * (int64_t)(sizeof(float) + ((const void*)logits == (const void*)dlogits ? 0 : sizeof(OUT)));
    const bool a_row_each = vocab % 4 != 0 && vocab >= 4096 && touched <= 1LL << 28 && 4 * rows >= 3 * rounds * round;
    // (a launch of 2^32 or more work items runs without those beyond, and without an error)
    if (BR_NLL_BWD_FLAT && aligned && !a_row_each && rows <= 65535 && blocks_x <= 0xffffffffLL / kFlatBlock / rows) {
        const dim3 grid((unsigned)blocks_x, (unsigned)rows);
        if (vocab % 4 == 0) nll_bwd_flat_kernel<OUT, true><<<grid, kFlatBlock, 0, st>>>(logits, target, keep, lse, dlogits, scale, vocab);
        else nll_bwd_flat_kernel<OUT, false><<<grid, kFlatBlock, 0, st>>>(logits, target, keep, lse, dlogits, scale, vocab);
    } else {
        nll_bwd_kernel<OUT><<<(unsigned)rows, kVBlock, 0, st>>>(logits, target, keep, lse, dlogits, scale, vocab, vec_ok);
    }
}

}  // namespace

extern "C" {

int br_hip_softmax_fwd(const float* x, float* y, int64_t rows, int64_t cols, br_stream_t stream) {
    if (rows < 0 || cols <= 0 || rows > 0x7fffffff) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!x) return BR_ERR_INPUT;
    if (!y) return BR_ERR_OUTPUT;
    RowBias rb = {nullptr, nullptr, nullptr, nullptr, 1, 1};
    return launch_softmax_fwd<kPlain>(x, y, rows, cols, rb, as_stream(stream));
}

int br_hip_softmax_bwd(const float* dy, const float* y, float* dx, int64_t rows, int64_t cols,
                       br_stream_t stream) {
    if (rows < 0 || cols <= 0 || rows > 0x7fffffff) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!dy || !y) return BR_ERR_INPUT;
    if (!dx) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    const int g = softmax_bwd_granule(cols, dy, y, dx);
    if (g > 0) return launch_softmax_bwd_wave(g, dy, y, dx, Copy16{nullptr, 0}, rows, cols, st);
    softmax_bwd_generic<<<(unsigned)rows, kBlock, 0, st>>>(dy, y, dx, cols);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_softmax_bwd_to16(const float* dy, const float* y, void* dx16, int dx16_dtype, int64_t rows, int64_t cols,
                            br_stream_t stream) {
    if (rows < 0 || cols <= 0 || rows > 0x7fffffff) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!dy || !y) return BR_ERR_INPUT;
    if (!dx16 || dx16 == (const void*)dy || dx16 == (const void*)y) return BR_ERR_OUTPUT;
    const int g = softmax_bwd_granule(cols, dy, y, dy);
    if (!copy16_ok(dx16, dx16_dtype) || g < 2) return BR_ERR_TODO;
    return launch_softmax_bwd_wave(g, dy, y, nullptr, Copy16{dx16, dx16_dtype == BR_BF16}, rows, cols, as_stream(stream));
}

int br_hip_alibi_masked_softmax_fwd(const float* s, const float* alibi, const float* xmask, float* p,
                                    int64_t batch, int64_t heads, int64_t tq, int64_t tk, br_stream_t stream) {
    if (batch < 0 || heads <= 0 || tq <= 0 || tk <= 0 || heads > 0x7fffffff || tq > 0x7fffffff)
        return BR_ERR_ATTR;
    const int64_t rows = batch * heads * tq;
    if (rows > 0x7fffffff) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!s) return BR_ERR_INPUT;
    if (!p) return BR_ERR_OUTPUT;
    RowBias rb = {alibi, xmask, nullptr, nullptr, (int)heads, (int)tq};
    return launch_softmax_fwd<kTables>(s, p, rows, tk, rb, as_stream(stream));
}

int br_hip_alibi_masked_softmax_fwd_copy16(const float* s, const float* alibi, const float* xmask, float* p, void* p16,
                                           int p16_dtype, int64_t batch, int64_t heads, int64_t tq, int64_t tk,
                                           br_stream_t stream) {
    if (batch < 0 || heads <= 0 || tq <= 0 || tk <= 0 || heads > 0x7fffffff || tq > 0x7fffffff)
        return BR_ERR_ATTR;
    const int64_t rows = batch * heads * tq;
    if (rows > 0x7fffffff) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!s) return BR_ERR_INPUT;
    if (!p || !p16) return BR_ERR_OUTPUT;
    if (!copy16_ok(p16, p16_dtype)) return BR_ERR_TODO;
    RowBias rb = {alibi, xmask, nullptr, nullptr, (int)heads, (int)tq};
    return launch_softmax_fwd<kTables>(s, p, rows, tk, rb, as_stream(stream), Copy16{p16, p16_dtype == BR_BF16});
}

int br_hip_alibi_causal_softmax_fwd(const float* s, const double* slopes, const int32_t* valid, float* p,
                                    int64_t batch, int64_t heads, int64_t tq, int64_t tk, br_stream_t stream) {
    if (batch < 0 || heads <= 0 || tq <= 0 || tk <= 0 || heads > 0x7fffffff || tq > 0x7fffffff)
        return BR_ERR_ATTR;
    const int64_t rows = batch * heads * tq;
    if (rows > 0x7fffffff) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!s || !slopes || !valid) return BR_ERR_INPUT;
    if (!p) return BR_ERR_OUTPUT;
    RowBias rb = {nullptr, nullptr, slopes, valid, (int)heads, (int)tq};
    return launch_softmax_fwd<kAnalytic>(s, p, rows, tk, rb, as_stream(stream));
}

int br_hip_logsoftmax_nll_fwd(const float* logits, const int32_t* target, const int32_t* keep, float* lse,
                              float* row_logp, float* result, int64_t rows, int64_t vocab, br_stream_t stream) {
    if (rows < 0 || vocab <= 0 || rows > 0x7fffffff) return BR_ERR_ATTR;
    if (!result) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    if (rows > 0) {
        if (!logits || !target || !keep) return BR_ERR_INPUT;
        if (!lse || !row_logp) return BR_ERR_OUTPUT;
        if (rows <= 256) nll_fwd_kernel<4><<<(unsigned)rows, kVBlock, 0, st>>>(logits, target, keep, lse, row_logp, vocab);
        else nll_fwd_kernel<1><<<(unsigned)rows, kVBlock, 0, st>>>(logits, target, keep, lse, row_logp, vocab);
        BR_HIP_LAUNCH_CHECK();
    }
    nll_reduce_kernel<<<1, kVBlock, 0, st>>>(row_logp, keep, result, rows);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

int br_hip_logsoftmax_nll_bwd(const float* logits, const int32_t* target, const int32_t* keep, const float* lse,
                              void* dlogits, int dlogits_dtype, float scale, int64_t rows, int64_t vocab,
                              br_stream_t stream) {
    if (rows < 0 || vocab <= 0 || rows > 0x7fffffff) return BR_ERR_ATTR;
    if (rows == 0) return BR_OK;
    if (!logits || !target || !keep || !lse) return BR_ERR_INPUT;
    if (!dlogits) return BR_ERR_OUTPUT;
    hipStream_t st = as_stream(stream);
    if (dlogits_dtype == BR_F32) {
        const bool aligned = aligned16(logits) && aligned16(dlogits);
        launch_nll_bwd<float>(logits, target, keep, lse, (float*)dlogits, scale, rows, vocab, aligned, st);
    } else if (dlogits_dtype == BR_F16) {
        if ((const void*)logits == dlogits) return BR_ERR_OUTPUT;
        const bool aligned = aligned16(logits) && aligned8(dlogits);
        launch_nll_bwd<__half>(logits, target, keep, lse, (__half*)dlogits, scale, rows, vocab, aligned, st);
    } else if (dlogits_dtype == BR_BF16) {
        if ((const void*)logits == dlogits) return BR_ERR_OUTPUT;
        const bool aligned = aligned16(logits) && aligned8(dlogits);
        launch_nll_bwd<__hip_bfloat16>(logits, target, keep, lse, (__hip_bfloat16*)dlogits, scale, rows, vocab, aligned, st);
    } else {
        return BR_ERR_TODO;
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

}  // extern "C"
