// AdamW parameter update for gfx950: one pass over (param, grad, m, v), all
// arithmetic in fp32.  HBM-bound: 16 B read + 12 B written per fp32 parameter;
// a 16-bit parameter with an fp32 master copy reads 16 B and writes 14 B.
//
// Any number of tensors of one parameter group share a launch.  Of a block's
// twelve tensors eight are vectors of a few thousand values: a launch each
// costs 4.6 us for a few blocks of work, and every matrix launched by itself
// drains the chip before the next one fills it again.  166 M parameters in 29
// tensors (two blocks at hidden 2048, 32000 words): 1046 us a step with a
// launch per tensor, 924 in three (5.4 TB/s).
#include "common.hpp"

using namespace brk;

namespace {

constexpr int kBlock = 256;

struct AdamW {
    float lr, beta1, beta2, eps, decay;  // decay = 1 - lr * weight_decay
    float step_size;                     // lr / (1 - beta1^t)
    float sqrt_bc2;                      // sqrt(1 - beta2^t)
};

// The update of torch.optim.AdamW (decoupled weight decay), operation for
// operation: decay the parameter, update both moments, then
// p -= step_size * (m / (sqrt(v) / sqrt(1 - beta2^t) + eps)).
__device__ __forceinline__ float adamw_one(float p, float g, float& m, float& v, const AdamW& a) {
    p = p * a.decay;
    m = m + (g - m) * (1.0f - a.beta1);                  // lerp, as torch does it
    v = v * a.beta2 + ((1.0f - a.beta2) * g) * g;
    const float denom = sqrtf(v) / a.sqrt_bc2 + a.eps;
    return p - a.step_size * (m / denom);
}

template <typename T>
__device__ __forceinline__ float to_f32(T x);
template <>
__device__ __forceinline__ float to_f32<float>(float x) { return x; }
template <>
__device__ __forceinline__ float to_f32<__half>(__half x) { return __half2float(x); }
template <>
__device__ __forceinline__ float to_f32<__hip_bfloat16>(__hip_bfloat16 x) { return __bfloat162float(x); }
template <typename T>
__device__ __forceinline__ T from_f32(float x);
template <>
__device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <>
__device__ __forceinline__ __half from_f32<__half>(float x) { return __float2half_rn(x); }
template <>
__device__ __forceinline__ __hip_bfloat16 from_f32<__hip_bfloat16>(float x) { return __float2bfloat16(x); }

// The tensors of one launch.  A workgroup owns kBlock granules of one of them: tensor t's are the workgroups
// first[t] .. first[t + 1) (UINT_MAX past the last tensor).
constexpr int kTensors = 32;
struct Tensor {
    void* param;
    float* master;
    const float* grad;
    float* m;
    float* v;
    int64_t n;
    int dtype;
    int vec;   // granules of 4 values, else of one
};
struct Group {
    AdamW a;
    unsigned first[kTensors];
    Tensor t[kTensors];
};
static_assert(sizeof(Group) <= 4096, "kernel arguments");

// master == nullptr: the parameter itself is the state (read as T, written as T).
// master != nullptr: the fp32 master copy is updated and `param` receives its rounding.
// The contraction barrier keeps `next` an fp32 value before it is rounded to T.
template <typename T>
__device__ __forceinline__ void adamw_granule(const Tensor& t, int64_t at, const AdamW& a) {
    T* param = static_cast<T*>(t.param);
    if (t.vec) {
        const int64_t base = at * 4;
        if (base >= t.n) return;
        const float4 g4 = load_stream(reinterpret_cast<const float4*>(t.grad + base));
        float4 m4 = load_stream(reinterpret_cast<const float4*>(t.m + base));
        float4 v4 = load_stream(reinterpret_cast<const float4*>(t.v + base));
        float p[4];
        if (t.master) {
            const float4 p4 = load_stream(reinterpret_cast<const float4*>(t.master + base));
            p[0] = p4.x; p[1] = p4.y; p[2] = p4.z; p[3] = p4.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) p[j] = to_f32<T>(param[base + j]);
        }
        p[0] = adamw_one(p[0], g4.x, m4.x, v4.x, a);
        p[1] = adamw_one(p[1], g4.y, m4.y, v4.y, a);
        p[2] = adamw_one(p[2], g4.z, m4.z, v4.z, a);
        p[3] = adamw_one(p[3], g4.w, m4.w, v4.w, a);
        asm volatile("" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]));
        store_stream(reinterpret_cast<float4*>(t.m + base), m4);
        store_stream(reinterpret_cast<float4*>(t.v + base), v4);
        if (t.master) store_stream(reinterpret_cast<float4*>(t.master + base), make_float4(p[0], p[1], p[2], p[3]));
#pragma unroll
        for (int j = 0; j < 4; j++) param[base + j] = from_f32<T>(p[j]);
    } else {
        if (at >= t.n) return;
        float mm = t.m[at], vv = t.v[at];
        float p = t.master ? t.master[at] : to_f32<T>(param[at]);
        p = adamw_one(p, t.grad[at], mm, vv, a);
        asm volatile("" : "+v"(p));
        t.m[at] = mm;
        t.v[at] = vv;
        if (t.master) t.master[at] = p;
        param[at] = from_f32<T>(p);
    }
}

// A launch of one tensor needs no search and no table in its arguments, and its type and width are compiled in: with
// the general kernel below a tensor of 16 million values, fp16 with an fp32 master copy, took 90.9 us instead of 86.7,
// and one of a million odd fp32 values 8.6 instead of 7.3.
struct Single {
    AdamW a;
    Tensor t;
};
template <typename T, int VEC>
__global__ __launch_bounds__(kBlock) void adamw_single_kernel(Single g) {
    g.t.vec = VEC == 4;
    adamw_granule<T>(g.t, (int64_t)blockIdx.x * kBlock + threadIdx.x, g.a);
}

// Which tensor is found by counting: 32 scalar compares against kernel arguments, no dependent loads.
__global__ __launch_bounds__(kBlock) void adamw_kernel(Group g) {
    int which = 0;
#pragma unroll
    for (int i = 1; i < kTensors; i++) which += blockIdx.x >= g.first[i] ? 1 : 0;
    const Tensor& t = g.t[which];
    const int64_t at = (int64_t)(blockIdx.x - g.first[which]) * kBlock + threadIdx.x;
    if (t.dtype == BR_F32) adamw_granule<float>(t, at, g.a);
    else if (t.dtype == BR_F16) adamw_granule<__half>(t, at, g.a);
    else adamw_granule<__hip_bfloat16>(t, at, g.a);
}

int check_tensor(const br_adamw_tensor& t) {
    if (t.n < 0) return BR_ERR_ATTR;
    if (t.n == 0) return BR_OK;
    if (!t.grad) return BR_ERR_INPUT;
    if (!t.param || !t.m || !t.v) return BR_ERR_OUTPUT;
    if (t.param_dtype == BR_F32 && t.master) return BR_ERR_ATTR;  // an fp32 parameter is its own master copy
    if (t.param_dtype != BR_F32 && t.param_dtype != BR_F16 && t.param_dtype != BR_BF16) return BR_ERR_TODO;
    return BR_OK;
}

// Whether one update writes what the other reads or writes.
bool shares_memory(const br_adamw_tensor& x, const br_adamw_tensor& y) {
    struct Span { const void* p; int64_t bytes; };
    auto spans = [](const br_adamw_tensor& t, Span* s) {
        s[0] = {t.param, t.n * (t.param_dtype == BR_F32 ? 4 : 2)};
        s[1] = {t.m, t.n * 4};
        s[2] = {t.v, t.n * 4};
        s[3] = {t.master, t.master ? t.n * 4 : 0};
        s[4] = {t.grad, t.n * 4};   // read only
    };
    Span a[5], b[5];
    spans(x, a);
    spans(y, b);
    for (int i = 0; i < 5; i++)
        for (int j = 0; j < 5; j++) {
            const uintptr_t p = reinterpret_cast<uintptr_t>(a[i].p), q = reinterpret_cast<uintptr_t>(b[j].p);
            if (!(i == 4 && j == 4) && p < q + (uintptr_t)b[j].bytes && q < p + (uintptr_t)a[i].bytes) return true;
        }
    return false;
}

}  // namespace

extern "C" {

int br_hip_adamw_group(const br_adamw_tensor* tensors, int64_t count, float lr, float beta1, float beta2, float eps,
                       float weight_decay, int64_t step, br_stream_t stream) {
    if (count < 0 || step < 1 || !(beta1 >= 0.f && beta1 < 1.f) || !(beta2 >= 0.f && beta2 < 1.f)) return BR_ERR_ATTR;
    if (count > 0 && !tensors) return BR_ERR_INPUT;
    // nothing is launched unless every tensor can be
    for (int64_t i = 0; i < count; i++) {
        const int rc = check_tensor(tensors[i]);
        if (rc != BR_OK) return rc;
    }
    Group g;
    int64_t from[kTensors];
    g.a.lr = lr;
    g.a.beta1 = beta1;
    g.a.beta2 = beta2;
    g.a.eps = eps;
    g.a.decay = 1.0f - lr * weight_decay;
    // bias corrections in fp64 on the host, as torch computes them for a python-number step
    const double bc1 = 1.0 - pow((double)beta1, (double)step);
    const double bc2 = 1.0 - pow((double)beta2, (double)step);
    g.a.step_size = (float)((double)lr / bc1);
    g.a.sqrt_bc2 = (float)sqrt(bc2);
    // Launches are closed when 32 tensors are in, when the grid is full (a tensor may go on in the next one), and
    // before a tensor that shares memory with one already in: those are updated one after the other.
    constexpr int64_t kMaxBlocks = (1 << 24) - 1;
    int used = 0;
    int64_t blocks = 0;
    auto launch = [&]() {
        if (used == 1) {
            const Single one{g.a, g.t[0]};
            const hipStream_t st = as_stream(stream);
            const unsigned grid = (unsigned)blocks;
#define BR_ADAMW_SINGLE(T)                                                            \
    if (one.t.vec) adamw_single_kernel<T, 4><<<grid, kBlock, 0, st>>>(one);           \
    else adamw_single_kernel<T, 1><<<grid, kBlock, 0, st>>>(one)
            if (one.t.dtype == BR_F32) { BR_ADAMW_SINGLE(float); }
            else if (one.t.dtype == BR_F16) { BR_ADAMW_SINGLE(__half); }
            else { BR_ADAMW_SINGLE(__hip_bfloat16); }
#undef BR_ADAMW_SINGLE
            used = 0;
            blocks = 0;
            BR_HIP_LAUNCH_CHECK();
            return (int)BR_OK;
        }
        for (int k = used; k < kTensors; k++) g.first[k] = 0xffffffffu;
        adamw_kernel<<<(unsigned)blocks, kBlock, 0, as_stream(stream)>>>(g);
        used = 0;
        blocks = 0;
        BR_HIP_LAUNCH_CHECK();
        return (int)BR_OK;
    };
    for (int64_t i = 0; i < count; i++) {
        const br_adamw_tensor& s = tensors[i];
        const int64_t size = s.param_dtype == BR_F32 ? 4 : 2;
        const bool vec = s.n % 4 == 0 && aligned16(s.grad) && aligned16(s.m) && aligned16(s.v) &&
                         (!s.master || aligned16(s.master)) && reinterpret_cast<uintptr_t>(s.param) % (4 * size) == 0;
        const int64_t per_block = vec ? 4 * kBlock : kBlock;
        for (int64_t at = 0; at < s.n;) {
            bool full = used == kTensors || blocks == kMaxBlocks;
            for (int k = 0; !full && k < used; k++) full = shares_memory(s, tensors[from[k]]);
            if (full) {
                const int rc = launch();
                if (rc != BR_OK) return rc;
            }
            const int64_t room = (kMaxBlocks - blocks) * per_block, n = s.n - at < room ? s.n - at : room;
            g.t[used] = Tensor{static_cast<char*>(s.param) + at * size, s.master ? s.master + at : nullptr, s.grad + at,
                               s.m + at, s.v + at, n, s.param_dtype, vec ? 1 : 0};
            g.first[used] = (unsigned)blocks;
            from[used++] = i;
            blocks += (n + per_block - 1) / per_block;
            at += n;
        }
    }
    return used ? launch() : BR_OK;
}

int br_hip_adamw(void* param, int param_dtype, float* master, const float* grad, float* m, float* v, int64_t n,
                 float lr, float beta1, float beta2, float eps, float weight_decay, int64_t step,
                 br_stream_t stream) {
    const br_adamw_tensor t = {param, master, grad, m, v, n, param_dtype};
    return br_hip_adamw_group(&t, 1, lr, beta1, beta2, eps, weight_decay, step, stream);
}

}  // extern "C"
