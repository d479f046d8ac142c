#include "hip_tensor.hpp"

#include <cmath>
#include <cstring>
#include <vector>

#include "br_hip.h"
#include "host_tensor.hpp"

namespace br {

void* hip_tensor_alloc(size_t bytes) {
    br_assert(ComputingContext::booted(), "device tensors need ComputingContext::boot() first");
    void* p = nullptr;
    BR_HIP_CHECK(br_hip_malloc(&p, bytes));
    return p;
}

void hip_tensor_free(void* p) {
    // kernels that still use the block may be in flight on the stream
    if (ComputingContext::booted()) ComputingContext::sync();
    BR_HIP_CHECK(br_hip_free(p));
}

namespace {

br_stream_t stream() { return ComputingContext::stream; }

// Negative codes are argument rejections and map one to one onto
// ComputingReturn; positive codes are HIP runtime failures and are fatal.
ComputingReturn done(int code, const char* what) {
    if (code > 0) hip_check_at(what, code, __FILE__, __LINE__);
    return static_cast<ComputingReturn>(code);
}
#define BR_OP(call)                                       \
    do {                                                  \
        ComputingReturn r_ = done((call), #call);         \
        if (r_ != OP_OK) return r_;                       \
    } while (0)

int code(const tensor_t& t) { return static_cast<int>(t->dtype()); }
bool dev(const tensor_t& t) { return t->is_cuda(); }
bool dev_f32(const tensor_t& t) { return t->is_cuda() && t->dtype() == DataType::Float; }

// MFMA element type for a product: a 16-bit operand decides; products of
// fp32-only operands follow the context's policy.
int pick_compute(std::initializer_list<tensor_t> ops) {
    bool f16 = false, bf16 = false;
    for (const auto& t : ops) {
        f16 = f16 || t->dtype() == DataType::F16;
        bf16 = bf16 || t->dtype() == DataType::BF16;
    }
    if (bf16) return BR_GEMM_BF16;
    if (f16) return BR_GEMM_F16;
    return ComputingContext::fp32_gemm_compute;
}

// Small regions at the tail of the 128 MiB workspace, clear of what the
// reduction kernels use at its head.
constexpr size_t kTailBytes = 8u << 20;
char* tail() { return static_cast<char*>(ComputingContext::workspace) + ComputingContext::workspace_size - kTailBytes; }
size_t head_bytes() { return ComputingContext::workspace_size - kTailBytes; }

// Every matrix product of the backend.  With a 16-bit MFMA type the product
// goes through br_hip_gemm_staged: fp32 operands are staged as 16-bit copies
// first, which lets the product run on the direct-to-LDS kernel, and products
// with few output tiles are split along K; fp32 compute goes straight through.
int product(int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha, const void* a, int a_dtype,
            int64_t lda, int64_t stride_a, const void* b, int b_dtype, int64_t ldb, int64_t stride_b, int accumulate,
            void* c, int c_dtype, int64_t ldc, int64_t stride_c, const float* bias, int64_t batch, int compute) {
    void* stream = ComputingContext::stream;
    if (compute == BR_GEMM_F32)
        return br_hip_gemm(trans_a, trans_b, m, n, k, alpha, a, a_dtype, lda, stride_a, b, b_dtype, ldb, stride_b,
                           accumulate, c, c_dtype, ldc, stride_c, bias, batch, compute, stream);
    const size_t need = br_hip_gemm_staged_workspace(trans_a, trans_b, m, n, k, a_dtype, b_dtype, batch);
    void* ws = ComputingContext::gemm_staging(0, need);
    return br_hip_gemm_staged(trans_a, trans_b, m, n, k, alpha, a, a_dtype, lda, stride_a, b, b_dtype, ldb, stride_b,
                              accumulate, c, c_dtype, ldc, stride_c, bias, batch, compute, ws, need, stream);
}

// Column sums and the two products of a backward operator, in this order or, where they are small, as one launch.
// Operands that have to be converted are, in one launch, and once where both products read them.
int two_products(const br_product& first, const br_product& second, const br_column_sums* sums, int compute,
                 const br_partial_sums* later = nullptr) {
    const size_t need = br_hip_gemm_pair_workspace(&first, &second, compute);
    void* ws = need ? ComputingContext::gemm_staging(0, need) : nullptr;
    return br_hip_gemm_pair(&first, &second, sums, later && later->partials ? later : nullptr, compute, ws, need,
                            ComputingContext::stream);
}

// An operand that several products of one operator read: with a 16-bit MFMA
// type an fp32 operand is converted once here (same rounding as the staged
// GEMM entry point applies), otherwise it is passed through.
struct Operand {
    const void* ptr;
    int dtype;
};
// Factor that takes the backward pass's gradient lift out of a parameter gradient.
float unlift() { return 1.0f / ComputingContext::grad_lift; }

Operand shared_operand(const void* p, int dtype, int64_t items, int compute) {
    if (dtype != BR_F32 || compute == BR_GEMM_F32 || items % 8 != 0) return {p, dtype};
    const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
    void* dst = ComputingContext::gemm_staging(1, (size_t)items * 2);
    BR_HIP_CHECK(br_hip_cast(p, BR_F32, dst, native, items, ComputingContext::stream));
    return {dst, native};
}

// The two products of a linear layer's backward once the gradient dy[n,out] is
// available in the products' type: weight_g[out,in] = dy^T . x, then
// x_g[n,in] = dy . W (in that order: x_g may overwrite x).
// (weight and weight_g may be the first rows of the `out` rows meant)
int linear_backward_products(const Operand& dy, const tensor_t& x, const tensor_t& weight, const tensor_t& x_g,
                             const tensor_t& weight_g, int64_t n, int64_t in, int64_t out, int compute,
                             const br_column_sums* sums = nullptr, const br_partial_sums* later = nullptr) {
    return two_products(
        {1, 0, out, in, n, unlift(), dy.ptr, dy.dtype, out, 0, x->data(), code(x), in, 0, weight_g->data(), code(weight_g), in, 0, 1},
        {0, 0, n, in, out, 1.0f, dy.ptr, dy.dtype, out, 0, weight->data(), code(weight), in, 0, x_g->data(), code(x_g), in, 0, 1},
        sums, compute, later);
}

// fp32 device pointer to a bias vector, converting 16-bit storage on the fly
// into workspace tail slot `slot` (each slot 1 MiB).
const float* bias_f32(const tensor_t& b, int slot) {
    if (b->dtype() == DataType::Float) return static_cast<const float*>(b->data());
    br_assert(b->items() * sizeof(float) <= (1u << 20), "bias vector too long for the conversion slot");
    float* dst = reinterpret_cast<float*>(tail() + (size_t)slot * (1u << 20));
    BR_HIP_CHECK(br_hip_cast(b->data(), code(b), dst, BR_F32, (int64_t)b->items(), stream()));
    return dst;
}

void shape4(const ShapeType& s, int64_t out[4]) {
    // rank <= 4 to rank 4 the way the reference describes tensors to cuDNN
    // (blackriver/cuda_tensor.hpp:39-49)
    const auto& v = s.vec();
    switch (v.size()) {
        case 4: out[0] = v[0]; out[1] = v[1]; out[2] = v[2]; out[3] = v[3]; break;
        case 3: out[0] = v[0]; out[1] = v[1]; out[2] = 1; out[3] = v[2]; break;
        case 2: out[0] = v[0]; out[1] = v[1]; out[2] = 1; out[3] = 1; break;
        case 1: out[0] = 1; out[1] = v[0]; out[2] = 1; out[3] = 1; break;
        default: br_panic("can't convert shape to rank 4");
    }
}

template <typename T>
void print_ends(const std::vector<T>& first, const std::vector<T>& last) {
    std::cout << "--------------------------" << std::endl;
    std::cout << "First " << first.size() << " : ";
    for (auto v : first) std::cout << v << " ";
    std::cout << std::endl;
    std::cout << "Last " << last.size() << " : ";
    for (auto v : last) std::cout << v << " ";
    std::cout << std::endl;
}

}  // namespace

// ------------------------------------------------------------------- io
template <DataType DT>
ComputingReturn HIPTensor<DT>::io_dump(tensor_t self) {
    const size_t n = std::min(self->shape().vec().back(), (size_t)8);
    const size_t items = self->items();
    // convert the two ends to fp32 on the device when stored in 16 bits
    float* stage = reinterpret_cast<float*>(tail());
    const size_t es = DataType_size(DT);
    const char* base = static_cast<const char*>(mem_);
    BR_OP(br_hip_cast(base, (int)DT, stage, BR_F32, (int64_t)n, stream()));
    BR_OP(br_hip_cast(base + (items - n) * es, (int)DT, stage + 8, BR_F32, (int64_t)n, stream()));
    std::vector<float> first(n), last(n);
    BR_OP(br_hip_memcpy_d2h(first.data(), stage, n * sizeof(float), stream()));
    BR_OP(br_hip_memcpy_d2h(last.data(), stage + 8, n * sizeof(float), stream()));
    ComputingContext::sync();
    print_ends(first, last);
    return OP_OK;
}

// Files hold raw fp32; 16-bit tensors are converted on the device.
template <DataType DT>
ComputingReturn HIPTensor<DT>::io_load(tensor_t self, const char* fileName) {
    std::vector<float> src;
    read_data(fileName, src);
    br_assert(src.size() == self->items(), "loaded data must has same size");
    const size_t bytes = src.size() * sizeof(float);
    if (DT == DataType::Float) {
        BR_OP(br_hip_memcpy_h2d(mem_, src.data(), bytes, stream()));
    } else {
        void* stage = ComputingContext::scratch(bytes);
        BR_OP(br_hip_memcpy_h2d(stage, src.data(), bytes, stream()));
        BR_OP(br_hip_cast(stage, BR_F32, mem_, (int)DT, (int64_t)src.size(), stream()));
    }
    ComputingContext::sync();  // `src` goes away when this returns
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::io_save(tensor_t self, const char* fileName) {
    const size_t n = self->items();
    std::vector<float> dst(n);
    if (DT == DataType::Float) {
        BR_OP(br_hip_memcpy_d2h(dst.data(), mem_, n * sizeof(float), stream()));
    } else {
        void* stage = ComputingContext::scratch(n * sizeof(float));
        BR_OP(br_hip_cast(mem_, (int)DT, stage, BR_F32, (int64_t)n, stream()));
        BR_OP(br_hip_memcpy_d2h(dst.data(), stage, n * sizeof(float), stream()));
    }
    ComputingContext::sync();
    std::ofstream out(fileName, std::ios::binary | std::ios::trunc);
    if (!out) return OP_OUTPUT_ERROR;
    out.write(reinterpret_cast<const char*>(dst.data()), n * sizeof(float));
    return out.good() ? OP_OK : OP_OUTPUT_ERROR;
}

// Point-to-point activation hand-off between pipeline stages.  All stages
// live in this process, so the payload goes through the in-process mailbox.
template <DataType DT>
ComputingReturn HIPTensor<DT>::io_nccl_send(tensor_t self, int dst) {
    const size_t bytes = self->items() * DataType_size(DT);
    std::vector<unsigned char> buf(bytes);
    BR_OP(br_hip_memcpy_d2h(buf.data(), mem_, bytes, stream()));
    ComputingContext::sync();
    CollectiveContext::post(CollectiveContext::nccl_rank, dst, buf.data(), bytes);
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::io_nccl_recv(tensor_t self, int src) {
    const size_t bytes = self->items() * DataType_size(DT);
    std::vector<unsigned char> buf(bytes);
    if (!CollectiveContext::take(src, CollectiveContext::nccl_rank, buf.data(), bytes)) return OP_INPUT_ERROR;
    BR_OP(br_hip_memcpy_h2d(mem_, buf.data(), bytes, stream()));
    ComputingContext::sync();
    return OP_OK;
}

// ------------------------------------------------------------- plumbing
template <DataType DT>
ComputingReturn HIPTensor<DT>::op_zero(tensor_t self) {
    // a fill kernel rather than a memset node, so callers may graph-capture it
    BR_OP(br_hip_fill(mem_, (int)DT, 0.0f, (int64_t)self->items(), stream()));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_fill(tensor_t self, float value) {
    BR_OP(br_hip_fill(mem_, (int)DT, value, (int64_t)self->items(), stream()));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_copy(tensor_t self, tensor_t src) {
    const size_t n = self->items();
    if (src->is_cpu()) {
        if (src->dtype() != DataType::Float) return OP_INPUT_ERROR;
        if (DT == DataType::Float) {
            BR_OP(br_hip_memcpy_h2d(mem_, src->data(), n * sizeof(float), stream()));
        } else {
            void* stage = ComputingContext::scratch(n * sizeof(float));
            BR_OP(br_hip_memcpy_h2d(stage, src->data(), n * sizeof(float), stream()));
            BR_OP(br_hip_cast(stage, BR_F32, mem_, (int)DT, (int64_t)n, stream()));
        }
        return OP_OK;
    }
    if (src->dtype() == DT) {
        BR_OP(br_hip_memcpy_d2d(mem_, src->data(), n * DataType_size(DT), stream()));
    } else {
        // storage conversion, e.g. fp32 master weights into fp16 compute copies
        BR_OP(br_hip_cast(src->data(), code(src), mem_, (int)DT, (int64_t)n, stream()));
    }
    return OP_OK;
}

template <DataType DT>
TransformerComputing::view_result_t HIPTensor<DT>::op_view(tensor_t self, size_t offset,
                                                           const std::vector<size_t>& newShape) {
    void* p = static_cast<char*>(mem_) + offset * DataType_size(DT);
    return std::make_shared<TensorType>(new HIPTensor<DT>(p), ShapeType(newShape));
}

// -------------------------------------------------------------- forward
template <DataType DT>
ComputingReturn HIPTensor<DT>::op_add(tensor_t self, tensor_t b, tensor_t c) {
    if (DT == DataType::BF16) return OP_TODO_ERROR;
    if (!dev(b) || b->dtype() != DT) return OP_INPUT_ERROR;
    if (!dev(c) || c->dtype() != DT || c->items() != self->items()) return OP_OUTPUT_ERROR;
    int64_t as[4], bs[4];
    shape4(self->shape(), as);
    shape4(b->shape(), bs);
    BR_OP(br_hip_add_bcast(mem_, b->data(), c->data(), (int)DT, as, bs, stream()));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_linear(tensor_t self, tensor_t w, tensor_t bias, tensor_t y) {
    if (!dev(w) || !dev(bias)) return OP_INPUT_ERROR;
    if (!dev(y)) return OP_OUTPUT_ERROR;
    const int64_t n = (int64_t)(self->shape()[0] * self->shape()[1]);
    const int64_t in = (int64_t)self->shape()[2];
    const int64_t out = (int64_t)w->shape()[0];
    if ((int64_t)w->shape()[1] != in || (int64_t)bias->items() != out) return OP_INPUT_ERROR;
    if ((int64_t)y->items() != n * out) return OP_OUTPUT_ERROR;
    // y[n,out] = x[n,in] . w[out,in]^T + bias, the bias added in the GEMM epilogue
    BR_OP(product(0, 1, n, out, in, 1.0f, mem_, (int)DT, in, 0, w->data(), code(w), in, 0, 0, y->data(), code(y),
                      out, 0, bias_f32(bias, 0), 1, pick_compute({self, w, y})));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_layernorm(tensor_t self, tensor_t mean, tensor_t var, tensor_t scale, tensor_t bias,
                                            tensor_t y, float eps) {
    if (DT != DataType::Float) return OP_TODO_ERROR;
    if (!dev_f32(scale) || !dev_f32(bias)) return OP_INPUT_ERROR;
    if (!dev_f32(y) || !dev_f32(mean) || !dev_f32(var)) return OP_OUTPUT_ERROR;
    const int64_t rows = (int64_t)(self->shape()[0] * self->shape()[1]);
    const int64_t cols = (int64_t)self->shape()[2];
    // mean / var may be larger scratch tensors; only the first `rows` entries are written
    if ((int64_t)mean->items() < rows || (int64_t)var->items() < rows) return OP_OUTPUT_ERROR;
    if ((int64_t)scale->items() != cols || (int64_t)bias->items() != cols) return OP_INPUT_ERROR;
    BR_OP(br_hip_layernorm_fwd(static_cast<const float*>(mem_), static_cast<const float*>(scale->data()),
                               static_cast<const float*>(bias->data()), static_cast<float*>(y->data()),
                               static_cast<float*>(mean->data()), static_cast<float*>(var->data()), rows, cols, eps,
                               stream()));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_transpos_0213(tensor_t self, tensor_t y) {
    if (self->shape().dim() != 4) return OP_INPUT_ERROR;
    if (!dev(y) || y->dtype() != DT || y->items() != self->items() || y->data() == mem_) return OP_OUTPUT_ERROR;
    const auto& s = self->shape();
    BR_OP(br_hip_transpose_0213(mem_, y->data(), (int)DataType_size(DT), (int64_t)s[0], (int64_t)s[1], (int64_t)s[2],
                                (int64_t)s[3], stream()));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_qk(tensor_t self, tensor_t k, tensor_t qk) {
    if (self->shape().dim() != 4 || !dev(k) || k->items() != self->items()) return OP_INPUT_ERROR;
    const auto& s = self->shape();
    const int64_t bh = (int64_t)(s[0] * s[1]), t = (int64_t)s[2], hd = (int64_t)s[3];
    if (!dev(qk) || (int64_t)qk->items() != bh * t * t) return OP_OUTPUT_ERROR;
    const float alpha = (float)(1.0 / sqrt((double)hd));
    BR_OP(product(0, 1, t, t, hd, alpha, mem_, (int)DT, hd, t * hd, k->data(), code(k), hd, t * hd, 0, qk->data(),
                      code(qk), t, t * t, nullptr, bh, pick_compute({self, k})));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_softmax(tensor_t self, tensor_t out) {
    if (DT != DataType::Float) return OP_TODO_ERROR;
    if (!dev_f32(out) || out->items() != self->items()) return OP_OUTPUT_ERROR;
    const int64_t cols = (int64_t)self->shape().vec().back();
    BR_OP(br_hip_softmax_fwd(static_cast<const float*>(mem_), static_cast<float*>(out->data()),
                             (int64_t)self->items() / cols, cols, stream()));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_attn(tensor_t self, tensor_t v, tensor_t attn) {
    if (self->shape().dim() != 4 || v->shape().dim() != 4 || !dev(v)) return OP_INPUT_ERROR;
    const auto& s = self->shape();
    const int64_t bh = (int64_t)(s[0] * s[1]), t = (int64_t)s[2], hd = (int64_t)v->shape()[3];
    if ((int64_t)v->items() != bh * t * hd) return OP_INPUT_ERROR;
    if (!dev(attn) || (int64_t)attn->items() != bh * t * hd) return OP_OUTPUT_ERROR;
    BR_OP(product(0, 0, t, hd, t, 1.0f, mem_, (int)DT, t, t * t, v->data(), code(v), hd, t * hd, 0, attn->data(),
                      code(attn), hd, t * hd, nullptr, bh, pick_compute({self, v})));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_gelu(tensor_t self, tensor_t dst) {
    if (DT == DataType::BF16) return OP_TODO_ERROR;
    if (!dev(dst) || dst->items() != self->items()) return OP_OUTPUT_ERROR;
    if (DT == DataType::Float && (dst->dtype() == DataType::F16 || dst->dtype() == DataType::BF16)) {
        // fp32 activation in, 16-bit operand buffer out
        BR_OP(br_hip_gelu_fwd_f32_to_16(static_cast<const float*>(mem_), dst->data(), code(dst), (int64_t)self->items(),
                                        stream()));
        return OP_OK;
    }
    if (dst->dtype() != DT) return OP_OUTPUT_ERROR;
    BR_OP(br_hip_gelu_fwd(mem_, dst->data(), (int)DT, (int64_t)self->items(), stream()));
    return OP_OK;
}

// Logits of the last real token of every sequence: the first position whose
// successor is padding, or position 0 when the row has no padding at all
// (that is what the reference computes, cuda_tensor.cpp:424-432).
template <DataType DT>
ComputingReturn HIPTensor<DT>::op_last_logits(tensor_t self, tensor_t mask_, tensor_t lm_head, tensor_t output) {
    if (DT != DataType::Float) return OP_TODO_ERROR;
    if (!mask_->is_cpu() || mask_->dtype() != DataType::Int || !dev(lm_head)) return OP_INPUT_ERROR;
    const int64_t batch = (int64_t)self->shape()[0], tokens = (int64_t)self->shape()[1];
    const int64_t hidden = (int64_t)self->shape()[2], vocab = (int64_t)lm_head->shape()[0];
    if (!dev_f32(output) || (int64_t)output->items() < batch * vocab) return OP_OUTPUT_ERROR;
    const int* mask = static_cast<const int*>(mask_->data());
    void* rows = ComputingContext::workspace;
    br_assert((size_t)(batch * hidden) * sizeof(float) <= head_bytes(), "workspace too small for last_logits");
    std::vector<int64_t> targets((size_t)batch);
    for (int64_t b = 0; b < batch; b++) {
        const int* m = mask + b * tokens;
        int64_t target = 0;
        for (int64_t i = 0; i < tokens - 1; i++) {
            if (m[i + 1] == 0) {
                target = i;
                break;
            }
        }
        targets[b] = b * tokens + target;
    }
    // the rows arrive in the type the product multiplies in (the rounding it would apply itself)
    const int compute = pick_compute({self, lm_head});
    const int type = compute == BR_GEMM_F16 ? BR_F16 : compute == BR_GEMM_BF16 ? BR_BF16 : BR_F32;
    BR_OP(br_hip_pick_rows(static_cast<const float*>(mem_), targets.data(), rows, type, batch, hidden, stream()));
    BR_OP(product(0, 1, batch, vocab, hidden, 1.0f, rows, type, hidden, 0, lm_head->data(), code(lm_head), hidden, 0, 0,
                  output->data(), BR_F32, vocab, 0, nullptr, 1, compute));
    return OP_OK;
}

namespace {
// What the newest op_loss_backward has its value from: which positions count and log p(label) of each, there once the
// stream has been waited for.  They lie, behind the labels, in the context's pinned slot 0, which copies of a call that
// left its value for later may still be reading or writing (`waiting`).
struct LossRecord {
    const int32_t* keep = nullptr;
    const float* logp = nullptr;
    int64_t positions = 0, count = 0;
    bool waiting = false;
} g_loss;
}  // namespace

float hip_finish_loss() {
    double total = 0.0;
    g_loss.waiting = false;
    if (g_loss.count > 0)
        for (int64_t i = 0; i < g_loss.positions; i++)
            if (g_loss.keep[i]) total += (double)g_loss.logp[i];
    const float ret = g_loss.count > 0 ? (float)(total / (double)g_loss.count) : 0.0f;
    ComputingContext::last_loss = ret;
    if (ComputingContext::echo_loss) std::cout << "#################  " << g_loss.count << " " << ret << std::endl;
    return ret;
}

// ------------------------------------------------------------- backward
// Shift-by-one masked cross entropy through the LM head, all on the device.
// Integer part (on the host, from the CPU ids / mask tensors, bit-exact):
//   position t < T-1 carries a loss iff mask[t] and mask[t+1] are non-zero;
//   its label is ids[t+1]; count = number of such positions.
// Float part, per chunk of rows that fits `all_logits`:
//   logits = x . W^T  ->  lse, log p(label)  ->  dlogits in place
//   x_g = dlogits . W          (zero in chunks without a label)
//   lm_head_g += dlogits^T . x
// Returns +mean log-prob of the labels (the reference's sign convention).
template <DataType DT>
TransformerComputing::loss_result_t HIPTensor<DT>::op_loss_backward(tensor_t self, tensor_t ids_, tensor_t mask_,
                                                                    tensor_t lm_head, tensor_t all_logits,
                                                                    tensor_t x_g, tensor_t lm_head_g) {
    if (DT != DataType::Float) return OP_TODO_ERROR;
    if (!ids_->is_cpu() || ids_->dtype() != DataType::Int || !mask_->is_cpu() || mask_->dtype() != DataType::Int)
        return OP_INPUT_ERROR;
    if (!dev(lm_head) || !dev_f32(all_logits)) return OP_INPUT_ERROR;
    if (!dev_f32(x_g) || x_g->items() != self->items()) return OP_OUTPUT_ERROR;
    if (lm_head_g->items() != lm_head->items() || lm_head_g->dtype() != DataType::Float) return OP_OUTPUT_ERROR;

    const int64_t batch = (int64_t)self->shape()[0], tokens = (int64_t)self->shape()[1];
    const int64_t hidden = (int64_t)self->shape()[2], vocab = (int64_t)lm_head->shape()[0];
    const int64_t n = batch * tokens;
    if ((int64_t)ids_->items() < n || (int64_t)mask_->items() < n) return OP_INPUT_ERROR;
    const int64_t cap = (int64_t)all_logits->items() / vocab;
    br_assert(cap >= 1, " logits workspace is not enough !");

    const int* ids = static_cast<const int*>(ids_->data());
    const int* mask = static_cast<const int*>(mask_->data());
    if (g_loss.waiting) ComputingContext::sync();
    // pinned: labels and keep go to the device without a wait, and the values come back
    int32_t* const labels = static_cast<int32_t*>(ComputingContext::pinned(0, (size_t)(3 * n) * sizeof(int32_t)));
    int32_t* const keep = labels + n;
    float* const logp = reinterpret_cast<float*>(keep + n);
    std::fill(labels, labels + n, -100);
    std::fill(keep, keep + n, 0);
    g_loss = LossRecord{keep, logp, n, 0, true};
    int64_t count = 0;
    for (int64_t b = 0; b < batch; b++) {
        for (int64_t t = 0; t + 1 < tokens; t++) {
            const int64_t i = b * tokens + t;
            if (mask[i] != 0 && mask[i + 1] != 0) {
                labels[i] = ids[i + 1];
                keep[i] = 1;
                count++;
            }
        }
    }
    const float scale = count > 0 ? 1.0f / (float)count : 0.0f;
    const int compute = pick_compute({self, lm_head});
    if (ComputingContext::grad_lift_auto) {
        // 16 * 2^ceil(log2(count)): undoes the mean over loss positions and leaves
        // four more bits of headroom below; no lift for fp32 products
        float lift_now = 1.0f;
        if (compute != BR_GEMM_F32 && count > 0) {
            lift_now = 16.0f;
            while (lift_now < 16.0f * (float)count) lift_now *= 2.0f;
        }
        ComputingContext::grad_lift = lift_now;
    }
    const float grad_lift = ComputingContext::grad_lift;   // x_g leaves carrying this factor

    // small per-row arrays in the workspace tail (slots 2..7)
    br_assert((size_t)n * 4 * sizeof(float) + 64 <= 6u * (1u << 20), "too many rows for the loss scratch");
    char* t0 = tail() + 2u * (1u << 20);
    int32_t* d_labels = reinterpret_cast<int32_t*>(t0);
    int32_t* d_keep = d_labels + n;
    float* d_lse = reinterpret_cast<float*>(d_keep + n);
    float* d_logp = d_lse + n;
    float* d_result = d_logp + n;
    // labels and keep lie next to each other, here and on the device
    if (n <= 2048) {
        BR_OP(br_hip_upload_words(d_labels, labels, 2 * n, stream()));
    } else {
        BR_OP(br_hip_memcpy_h2d(d_labels, labels, 2 * n * sizeof(int32_t), stream()));
    }

    // weight gradient target: the tensor itself when it lives on the device,
    // otherwise a zeroed device staging buffer that is added into the CPU
    // tensor at the end
    float* d_wg = nullptr;
    void* staging = nullptr;
    if (lm_head_g->is_cuda()) {
        d_wg = static_cast<float*>(lm_head_g->data());
    } else {
        staging = hip_tensor_alloc((size_t)(vocab * hidden) * sizeof(float));
        d_wg = static_cast<float*>(staging);
        BR_OP(br_hip_fill(d_wg, BR_F32, 0.f, vocab * hidden, stream()));
    }

    const float* x = static_cast<const float*>(mem_);
    float* dx = static_cast<float*>(x_g->data());
    float* logits = static_cast<float*>(all_logits->data());
    // lm_head_g is accumulated into, as the reference does; a driver that would
    // zero it right before (ComputingContext::loss_head_overwrite) gets the
    // first chunk written instead of added, which saves clearing and re-reading
    // a [vocab, hidden] tensor
    // (a host-resident gradient goes through the zeroed staging buffer either way;
    // in overwrite mode the staged sum is assigned to it instead of added)
    const bool overwrite_host = ComputingContext::loss_head_overwrite && !lm_head_g->is_cuda();
    bool overwrite = ComputingContext::loss_head_overwrite && lm_head_g->is_cuda();
    if (overwrite && count == 0) BR_OP(br_hip_fill(d_wg, BR_F32, 0.f, vocab * hidden, stream()));
    // x_g is zero where no position carries a loss; the others' rows are written by their product
    if (count == 0) BR_OP(br_hip_fill(dx, BR_F32, 0.f, n * hidden, stream()));
    for (int64_t r0 = 0; r0 < n && count > 0; r0 += cap) {
        const int64_t rows = std::min(cap, n - r0);
        bool any = false;
        for (int64_t r = r0; r < r0 + rows; r++) any = any || keep[r] != 0;
        if (!any) {  // nothing but zero gradients in this chunk
            BR_OP(br_hip_fill(dx + r0 * hidden, BR_F32, 0.f, rows * hidden, stream()));
            continue;
        }
        BR_OP(product(0, 1, rows, vocab, hidden, 1.0f, x + r0 * hidden, BR_F32, hidden, 0, lm_head->data(),
                          code(lm_head), hidden, 0, 0, logits, BR_F32, vocab, 0, nullptr, 1, compute));
        BR_OP(br_hip_logsoftmax_nll_fwd(logits, d_labels + r0, d_keep + r0, d_lse + r0, d_logp + r0, d_result, rows,
                                        vocab, stream()));
        // dlogits.  With fp32 products it is scaled by 1/count in place, as the
        // reference does.  With 16-bit products the stored operand leaves 1/count
        // out (p/count would fall below fp16's smallest subnormal at a real
        // vocabulary size) and, for fp16, carries an exact factor 2^14 that lifts
        // probabilities down to 4e-12 into range (|softmax - onehot| <= 1, so no
        // overflow); both factors go into the products' alpha.
        Operand dl{logits, BR_F32};
        float alpha = 1.0f;
        if (compute == BR_GEMM_F32) {
            BR_OP(br_hip_logsoftmax_nll_bwd(logits, d_labels + r0, d_keep + r0, d_lse + r0, logits, BR_F32, scale,
                                            rows, vocab, stream()));
        } else {
            const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            const float lift = compute == BR_GEMM_F16 ? 16384.0f : 1.0f;
            alpha = scale / lift;
            if ((rows * vocab) % 8 == 0) {
                void* dl16 = ComputingContext::gemm_staging(1, (size_t)(rows * vocab) * 2);
                BR_OP(br_hip_logsoftmax_nll_bwd(logits, d_labels + r0, d_keep + r0, d_lse + r0, dl16, native, lift,
                                                rows, vocab, stream()));
                dl = Operand{dl16, native};
            } else {
                BR_OP(br_hip_logsoftmax_nll_bwd(logits, d_labels + r0, d_keep + r0, d_lse + r0, logits, BR_F32, lift,
                                                rows, vocab, stream()));
                dl = shared_operand(logits, BR_F32, rows * vocab, compute);
            }
        }
        BR_OP(product(0, 0, rows, hidden, vocab, alpha * grad_lift, dl.ptr, dl.dtype, vocab, 0, lm_head->data(), code(lm_head),
                      hidden, 0, 0, dx + r0 * hidden, BR_F32, hidden, 0, nullptr, 1, compute));
        BR_OP(product(1, 0, vocab, hidden, rows, alpha, dl.ptr, dl.dtype, vocab, 0, x + r0 * hidden, BR_F32, hidden,
                      0, overwrite ? 0 : 1, d_wg, BR_F32, hidden, 0, nullptr, 1, compute));
        overwrite = false;
    }
    // overwrite mode with no chunk carrying a label at all: the gradient is zero
    if (overwrite && count > 0) BR_OP(br_hip_fill(d_wg, BR_F32, 0.f, vocab * hidden, stream()));

    // sum of log p(label) in fp64 on the host, as the reference accumulates it
    if (count > 0) BR_OP(br_hip_memcpy_d2h(logp, d_logp, n * sizeof(float), stream()));
    g_loss.count = count;
    const bool later = ComputingContext::loss_later && !staging;
    if (!later) ComputingContext::sync();

    if (staging) {
        float* host_g = static_cast<float*>(lm_head_g->data());
        float* bounce = static_cast<float*>(ComputingContext::host_workspace);
        const size_t per = ComputingContext::workspace_size / sizeof(float);
        const size_t all = (size_t)(vocab * hidden);
        for (size_t off = 0; off < all; off += per) {
            const size_t cnt = std::min(per, all - off);
            BR_OP(br_hip_memcpy_d2h(bounce, d_wg + off, cnt * sizeof(float), stream()));
            ComputingContext::sync();
            if (overwrite_host) {
                memcpy(host_g + off, bounce, cnt * sizeof(float));
            } else {
                for (size_t i = 0; i < cnt; i++) host_g[off + i] += bounce[i];
            }
        }
        hip_tensor_free(staging);
    }

    return later ? 0.0f : hip_finish_loss();
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_layernorm_backward(tensor_t self, tensor_t scale, tensor_t bias, tensor_t var,
                                                     tensor_t y, tensor_t dscale, tensor_t dbias, tensor_t din,
                                                     float eps) {
    if (DT != DataType::Float) return OP_TODO_ERROR;
    if (!dev_f32(scale) || !dev_f32(bias) || !dev_f32(var) || !dev_f32(y)) return OP_INPUT_ERROR;
    if (!dev_f32(dscale) || !dev_f32(dbias) || !dev_f32(din)) return OP_OUTPUT_ERROR;
    const int64_t rows = (int64_t)(self->shape()[0] * self->shape()[1]);
    const int64_t cols = (int64_t)self->shape()[2];
    if (y->items() != self->items() || (int64_t)var->items() < rows) return OP_INPUT_ERROR;
    if (din->items() != self->items() || (int64_t)dscale->items() != cols || (int64_t)dbias->items() != cols)
        return OP_OUTPUT_ERROR;
    const size_t need = br_hip_layernorm_bwd_workspace(rows, cols);
    void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
    BR_OP(br_hip_layernorm_bwd(static_cast<const float*>(mem_), static_cast<const float*>(y->data()),
                               static_cast<const float*>(scale->data()), static_cast<const float*>(bias->data()),
                               static_cast<const float*>(var->data()), static_cast<float*>(dscale->data()),
                               static_cast<float*>(dbias->data()), static_cast<float*>(din->data()), rows, cols, eps,
                               unlift(), ws, need, stream()));
    return OP_OK;
}

// self = dy[n,out].  Order matters: the bias and weight gradients read x
// before the input gradient may overwrite it (x_g aliases x in the scripts).
template <DataType DT>
ComputingReturn HIPTensor<DT>::op_linear_backward(tensor_t self, tensor_t x, tensor_t weight, tensor_t bias,
                                                  tensor_t x_g, tensor_t weight_g, tensor_t bias_g) {
    if (!dev(x) || !dev(weight)) return OP_INPUT_ERROR;
    if (!dev(x_g) || !dev(weight_g) || !dev_f32(bias_g)) return OP_OUTPUT_ERROR;
    const int64_t n = (int64_t)(self->shape()[0] * self->shape()[1]);
    const int64_t out = (int64_t)self->shape()[2], in = (int64_t)x->shape()[2];
    if ((int64_t)x->items() != n * in || (int64_t)weight->items() != out * in) return OP_INPUT_ERROR;
    if ((int64_t)x_g->items() != n * in || (int64_t)weight_g->items() != out * in || (int64_t)bias_g->items() != out)
        return OP_OUTPUT_ERROR;
    const int compute = pick_compute({self, x, weight});
    // bias_g[o] = sum_n dy[n,o]
    const size_t need = br_hip_colsum_workspace(n, out);
    void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
    if (DT == DataType::Float && compute != BR_GEMM_F32 && out % 8 == 0) {
        // one pass over dy: its column sums and the 16-bit copy both products read
        const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
        void* dy16 = ComputingContext::gemm_staging(1, (size_t)(n * out) * 2);
        BR_OP(br_hip_colsum_cast(static_cast<const float*>(mem_), static_cast<float*>(bias_g->data()), dy16, native, n,
                                 out, unlift(), ws, need, stream()));
        BR_OP(linear_backward_products(Operand{dy16, native}, x, weight, x_g, weight_g, n, in, out, compute));
    } else {
        const br_column_sums sums{mem_, (int)DT, static_cast<float*>(bias_g->data()), n, out, unlift(), ws, need};
        BR_OP(linear_backward_products(shared_operand(mem_, (int)DT, n * out, compute), x, weight, x_g, weight_g, n, in, out,
                                       compute, &sums));
    }
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_gelu_backward(tensor_t self, tensor_t x, tensor_t x_g) {
    if (DT == DataType::BF16) return OP_TODO_ERROR;
    if (!dev(x) || x->dtype() != DT || x->items() != self->items()) return OP_INPUT_ERROR;
    if (!dev(x_g) || x_g->dtype() != DT || x_g->items() != self->items()) return OP_OUTPUT_ERROR;
    BR_OP(br_hip_gelu_bwd(mem_, x->data(), x_g->data(), (int)DT, (int64_t)self->items(), stream()));
    return OP_OK;
}

namespace {
struct AttnDims {
    int64_t bh, t, hd;
};
bool attn_dims(const tensor_t& d_o, const tensor_t& attn, const tensor_t& v, AttnDims& d) {
    if (d_o->shape().dim() != 4) return false;
    const auto& s = d_o->shape();
    d.bh = (int64_t)(s[0] * s[1]);
    d.t = (int64_t)s[2];
    d.hd = (int64_t)s[3];
    return (int64_t)attn->items() == d.bh * d.t * d.t && (int64_t)v->items() == d.bh * d.t * d.hd;
}
// v_g = P^T . dO, then dP = dO . V^T
int attn_products(const Operand& d_o, const tensor_t& attn, const tensor_t& v, void* dp, int dp_dtype, const tensor_t& v_g,
                  const AttnDims& d, int compute) {
    return two_products({1, 0, d.t, d.hd, d.t, 1.0f, attn->data(), code(attn), d.t, d.t * d.t, d_o.ptr, d_o.dtype, d.hd,
                         d.t * d.hd, v_g->data(), code(v_g), d.hd, d.t * d.hd, d.bh},
                        {0, 1, d.t, d.t, d.hd, 1.0f, d_o.ptr, d_o.dtype, d.hd, d.t * d.hd, v->data(), code(v), d.hd,
                         d.t * d.hd, dp, dp_dtype, d.t, d.t * d.t, d.bh},
                        nullptr, compute);
}
}  // namespace

// self = dO[B,NH,T,HD]:  v_g = P^T . dO,  attn_g = dO . V^T
template <DataType DT>
ComputingReturn HIPTensor<DT>::op_attn_backward(tensor_t self, tensor_t attn, tensor_t v, tensor_t attn_g,
                                                tensor_t v_g) {
    AttnDims d;
    if (!dev(attn) || !dev(v) || !attn_dims(self, attn, v, d)) return OP_INPUT_ERROR;
    if (!dev(attn_g) || !dev(v_g) || attn_g->items() != attn->items() || v_g->items() != v->items())
        return OP_OUTPUT_ERROR;
    const int compute = pick_compute({self, attn, v});
    BR_OP(attn_products(Operand{mem_, (int)DT}, attn, v, attn_g->data(), code(attn_g), v_g, d, compute));
    return OP_OK;
}

template <DataType DT>
ComputingReturn HIPTensor<DT>::op_softmax_backward(tensor_t self, tensor_t out, tensor_t x_g) {
    if (DT != DataType::Float) return OP_TODO_ERROR;
    if (!dev_f32(out) || out->items() != self->items()) return OP_INPUT_ERROR;
    if (!dev(x_g) || x_g->items() != self->items()) return OP_OUTPUT_ERROR;
    const int64_t cols = (int64_t)self->shape().vec().back();
    const int64_t rows = (int64_t)self->items() / cols;
    const float* dy = static_cast<const float*>(mem_);
    const float* y = static_cast<const float*>(out->data());
    if (x_g->dtype() != DataType::Float) {
        // a 16-bit gradient for the score products: written directly when the
        // kernel can, otherwise fp32 into scratch memory and converted
        const int rc = br_hip_softmax_bwd_to16(dy, y, x_g->data(), code(x_g), rows, cols, stream());
        if (rc == BR_ERR_TODO) {
            float* tmp = static_cast<float*>(ComputingContext::scratch(self->items() * sizeof(float)));
            BR_OP(br_hip_softmax_bwd(dy, y, tmp, rows, cols, stream()));
            BR_OP(br_hip_cast(tmp, BR_F32, x_g->data(), code(x_g), (int64_t)self->items(), stream()));
        } else {
            BR_OP(rc);
        }
        return OP_OK;
    }
    BR_OP(br_hip_softmax_bwd(dy, y, static_cast<float*>(x_g->data()), rows, cols, stream()));
    return OP_OK;
}

// The two ops above in one: dP is staged in scratch memory so that attn_g may
// alias attn (it does in the scripts): dS = P o (dP - rowsum(dP o P)) is then
// written over P row by row, each row read completely before it is replaced.
template <DataType DT>
ComputingReturn HIPTensor<DT>::op_softmax_attn_backward(tensor_t self, tensor_t attn, tensor_t v, tensor_t attn_g,
                                                        tensor_t v_g) {
    AttnDims d;
    if (!dev_f32(attn) || !dev(v) || !attn_dims(self, attn, v, d)) return OP_INPUT_ERROR;
    if (!dev_f32(attn_g) || !dev(v_g) || attn_g->items() != attn->items() || v_g->items() != v->items())
        return OP_OUTPUT_ERROR;
    const int compute = pick_compute({self, attn, v});
    float* dp = static_cast<float*>(ComputingContext::scratch((size_t)(d.bh * d.t * d.t) * sizeof(float)));
    BR_OP(attn_products(Operand{mem_, (int)DT}, attn, v, dp, BR_F32, v_g, d, compute));
    BR_OP(br_hip_softmax_bwd(dp, static_cast<const float*>(attn->data()), static_cast<float*>(attn_g->data()),
                             d.bh * d.t, d.t, stream()));
    return OP_OK;
}

// self = dS[B,NH,T,T]:  q_g = dS . K / sqrt(HD),  k_g = dS^T . Q / sqrt(HD)
template <DataType DT>
ComputingReturn HIPTensor<DT>::op_qk_backward(tensor_t self, tensor_t q, tensor_t k, tensor_t q_g, tensor_t k_g) {
    if (q->shape().dim() != 4 || !dev(q) || !dev(k) || k->items() != q->items()) return OP_INPUT_ERROR;
    const auto& s = q->shape();
    const int64_t bh = (int64_t)(s[0] * s[1]), t = (int64_t)s[2], hd = (int64_t)s[3];
    if ((int64_t)self->items() != bh * t * t) return OP_INPUT_ERROR;
    if (!dev(q_g) || !dev(k_g) || q_g->items() != q->items() || k_g->items() != q->items()) return OP_OUTPUT_ERROR;
    const float alpha = (float)(1.0 / sqrt((double)hd));
    const int compute = pick_compute({self, q, k});
    BR_OP(two_products({0, 0, t, hd, t, alpha, mem_, (int)DT, t, t * t, k->data(), code(k), hd, t * hd, q_g->data(), code(q_g),
                        hd, t * hd, bh},
                       {1, 0, t, hd, t, alpha, mem_, (int)DT, t, t * t, q->data(), code(q), hd, t * hd, k_g->data(), code(k_g),
                        hd, t * hd, bh},
                       nullptr, compute));
    return OP_OK;
}

ComputingReturn hip_gelu_linear_backward(const tensor_t& dy, const tensor_t& u, const tensor_t& du, const tensor_t& x,
                                         const tensor_t& weight, const tensor_t& bias, const tensor_t& x_g,
                                         const tensor_t& weight_g, const tensor_t& bias_g) {
    bool fast = dev_f32(dy) && dev_f32(u) && dev_f32(du) && dev(x) && dev(weight) && dev(x_g) && dev(weight_g) &&
                dev_f32(bias_g) && du->shape().dim() == 3 && x->shape().dim() == 3 && u->items() == dy->items() &&
                du->items() == dy->items();
    if (fast) {
        const int64_t n = (int64_t)(du->shape()[0] * du->shape()[1]);
        const int64_t out = (int64_t)du->shape()[2], in = (int64_t)x->shape()[2];
        const int compute = pick_compute({du, x, weight});
        fast = compute != BR_GEMM_F32 && out % 8 == 0 && (int64_t)x->items() == n * in &&
               (int64_t)weight->items() == out * in && (int64_t)x_g->items() == n * in &&
               (int64_t)weight_g->items() == out * in && (int64_t)bias_g->items() == out;
        if (fast) {
            const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            const size_t need = br_hip_colsum_workspace(n, out);
            void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
            void* dy16 = ComputingContext::gemm_staging(1, (size_t)(n * out) * 2);
            // Where the products share a launch the column sums are added up beside them, so that the GELU's pass need not own whole
            // columns.  In a step over [1000 x 4096]: 18.7 us with its sums and 35.7 for the products, 13.4 and 38.2 so.  Not where
            // that pass adds up with fewer roundings: up to 256 rows, and 512 of up to 2048 columns (its narrowest strips), a thread
            // has one position and few waves have any.  Against 64 bits, owned / beside: [2048] from 288 rows 8.5e-8 / 9.3e-8,
            // from 416 9.3 / 9.4, from 512 9.9 / 9.4; [2304] from 257 9.6 / 9.0, [4096] from 1000 10.3 / 9.8.  With the products, us:
            // 512 -> 2048 features, 300 rows 13.1 / 13.6, 449 16.8 / 17.0, 600 21.4 / 19.0; 768 -> 3072, 257 rows 20.4 / 19.6.
            br_partial_sums later = {};
            const bool beside = n > (out > 2048 ? 256 : 512) && br_hip_gemm_pair_kernel(out, in, n, 1, n, in, out, 1, compute) >= 0;
            int rc = beside ? br_hip_gelu_bwd_cast_sums(static_cast<const float*>(dy->data()), static_cast<const float*>(u->data()),
                                                        static_cast<float*>(du->data()), static_cast<float*>(bias_g->data()), dy16, native,
                                                        n, out, unlift(), &later, ws, need, stream())
                            : (int)BR_ERR_TODO;
            if (rc == BR_ERR_TODO)
                rc = br_hip_gelu_bwd_colsum_cast(static_cast<const float*>(dy->data()), static_cast<const float*>(u->data()),
                                                 static_cast<float*>(du->data()), static_cast<float*>(bias_g->data()), dy16, native, n, out,
                                                 unlift(), ws, need, stream());
            if (rc != BR_ERR_TODO) {
                BR_OP(rc);
                BR_OP(linear_backward_products(Operand{dy16, native}, x, weight, x_g, weight_g, n, in, out, compute, nullptr, &later));
                return OP_OK;
            }
        }
    }
    // everything already in the products' 16-bit type (the 4h activation and its gradient kept in the
    // products' type): one pass gives du and the bias gradient, du is the
    // products' operand as it stands
    const DataType gdt = dy->dtype();
    const bool half = dev(dy) && dev(u) && dev(du) && (gdt == DataType::F16 || gdt == DataType::BF16) &&
                      u->dtype() == gdt && du->dtype() == gdt && dev(x) && dev(weight) && dev(x_g) && dev(weight_g) &&
                      dev_f32(bias_g) && du->shape().dim() == 3 && x->shape().dim() == 3 &&
                      u->items() == dy->items() && du->items() == dy->items();
    if (half) {
        const int64_t n = (int64_t)(du->shape()[0] * du->shape()[1]);
        const int64_t out = (int64_t)du->shape()[2], in = (int64_t)x->shape()[2];
        const int compute = pick_compute({du, x, weight});
        const int native = compute == BR_GEMM_F16 ? BR_F16 : compute == BR_GEMM_BF16 ? BR_BF16 : BR_F32;
        if (native == (int)gdt && out % 8 == 0 && (int64_t)x->items() == n * in && (int64_t)weight->items() == out * in &&
            (int64_t)x_g->items() == n * in && (int64_t)weight_g->items() == out * in &&
            (int64_t)bias_g->items() == out) {
            const size_t need = br_hip_bias_gelu_bwd_workspace(n, out);
            void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
            BR_OP(br_hip_bias_gelu_bwd(dy->data(), u->data(), nullptr, du->data(), static_cast<float*>(bias_g->data()),
                                       native, n, out, unlift(), ws, need, stream()));
            BR_OP(linear_backward_products(Operand{du->data(), native}, x, weight, x_g, weight_g, n, in, out, compute));
            return OP_OK;
        }
    }
    ComputingReturn r = dy->op_gelu_backward(dy, u, du);
    if (r != OP_OK) return r;
    return du->op_linear_backward(du, x, weight, bias, x_g, weight_g, bias_g);
}

ComputingReturn hip_linear_gelu(const tensor_t& x, const tensor_t& w, const tensor_t& bias, const tensor_t& u,
                                const tensor_t& y) {
    if (!dev(x) || !dev(w) || !dev(bias) || x->shape().dim() != 3) return OP_INPUT_ERROR;
    if (!dev(u) || !dev(y) || u->items() != y->items() || u->data() == y->data()) return OP_OUTPUT_ERROR;
    const int64_t n = (int64_t)(x->shape()[0] * x->shape()[1]);
    const int64_t in = (int64_t)x->shape()[2];
    const int64_t out = (int64_t)w->shape()[0];
    if ((int64_t)w->shape()[1] != in || (int64_t)bias->items() != out) return OP_INPUT_ERROR;
    if ((int64_t)u->items() != n * out) return OP_OUTPUT_ERROR;
    const DataType dt = x->dtype();
    if ((dt == DataType::F16 || dt == DataType::BF16) && w->dtype() == dt && u->dtype() == dt && y->dtype() == dt) {
        const int rc = br_hip_linear_gelu(x->data(), w->data(), bias_f32(bias, 0), u->data(), y->data(), (int)dt, n, out,
                                          in, stream());
        if (rc != BR_ERR_TODO) return done(rc, "br_hip_linear_gelu");
    }
    // the two operators
    ComputingReturn r = x->op_linear(x, w, bias, u);
    if (r != OP_OK) return r;
    return u->op_gelu(u, y);
}

ComputingReturn hip_linear_accumulate(const tensor_t& x, const tensor_t& w, const tensor_t& bias, const tensor_t& y) {
    if (!dev(x) || !dev(w) || !dev(bias) || x->shape().dim() != 3) return OP_INPUT_ERROR;
    if (!dev_f32(y)) return OP_OUTPUT_ERROR;
    const int64_t n = (int64_t)(x->shape()[0] * x->shape()[1]);
    const int64_t in = (int64_t)x->shape()[2];
    const int64_t out = (int64_t)w->shape()[0];
    if ((int64_t)w->shape()[1] != in || (int64_t)bias->items() != out) return OP_INPUT_ERROR;
    if ((int64_t)y->items() != n * out) return OP_OUTPUT_ERROR;
    BR_OP(product(0, 1, n, out, in, 1.0f, x->data(), code(x), in, 0, w->data(), code(w), in, 0, 1, y->data(), BR_F32,
                  out, 0, bias_f32(bias, 0), 1, pick_compute({x, w, y})));
    return OP_OK;
}

// y = x . w^T + bias + residual in one product (the residual is read in the epilogue); y may be the residual.
ComputingReturn hip_linear_residual(const tensor_t& x, const tensor_t& w, const tensor_t& bias,
                                    const tensor_t& residual, const tensor_t& y) {
    if (!dev(x) || !dev(w) || !dev(bias) || !dev_f32(residual) || x->shape().dim() != 3) return OP_INPUT_ERROR;
    if (!dev_f32(y)) return OP_OUTPUT_ERROR;
    const int64_t n = (int64_t)(x->shape()[0] * x->shape()[1]);
    const int64_t in = (int64_t)x->shape()[2];
    const int64_t out = (int64_t)w->shape()[0];
    if ((int64_t)w->shape()[1] != in || (int64_t)bias->items() != out || (int64_t)residual->items() != n * out)
        return OP_INPUT_ERROR;
    if ((int64_t)y->items() != n * out) return OP_OUTPUT_ERROR;
    const int compute = pick_compute({x, w, y});
    const size_t need = compute == BR_GEMM_F32 ? 0 : br_hip_gemm_staged_workspace(0, 1, n, out, in, code(x), code(w), 1);
    void* ws = need ? ComputingContext::gemm_staging(0, need) : nullptr;
    BR_OP(br_hip_linear_residual(x->data(), code(x), w->data(), code(w), bias_f32(bias, 0), residual->data(), y->data(),
                                 BR_F32, n, out, in, compute, ws, need, stream()));
    return OP_OK;
}

ComputingReturn hip_layernorm_backward_add(const tensor_t& dy, const tensor_t& scale, const tensor_t& bias,
                                           const tensor_t& var, const tensor_t& y, const tensor_t& dscale,
                                           const tensor_t& dbias, const tensor_t& residual, const tensor_t& din,
                                           float eps) {
    bool fast = dev_f32(dy) && dev_f32(scale) && dev_f32(bias) && dev_f32(var) && dev_f32(y) && dev_f32(dscale) &&
                dev_f32(dbias) && dev_f32(residual) && dev_f32(din) && dy->shape().dim() == 3;
    if (fast) {
        const int64_t rows = (int64_t)(dy->shape()[0] * dy->shape()[1]);
        const int64_t cols = (int64_t)dy->shape()[2];
        fast = y->items() == dy->items() && (int64_t)var->items() >= rows && din->items() == dy->items() &&
               residual->items() == dy->items() && (int64_t)dscale->items() == cols && (int64_t)dbias->items() == cols &&
               (int64_t)scale->items() == cols && (int64_t)bias->items() == cols && din->data() != y->data();
        if (fast) {
            const size_t need = br_hip_layernorm_bwd_workspace(rows, cols);
            void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
            const int rc = br_hip_layernorm_bwd_residual(
                static_cast<const float*>(dy->data()), static_cast<const float*>(y->data()),
                static_cast<const float*>(scale->data()), static_cast<const float*>(bias->data()),
                static_cast<const float*>(var->data()), static_cast<const float*>(residual->data()),
                static_cast<float*>(dscale->data()), static_cast<float*>(dbias->data()),
                static_cast<float*>(din->data()), rows, cols, eps, unlift(), ws, need, stream());
            if (rc != BR_ERR_TODO) return done(rc, "br_hip_layernorm_bwd_residual");
        }
    }
    // the two operators; din must then be a buffer of its own
    if (din->data() == residual->data()) return OP_OUTPUT_ERROR;
    ComputingReturn r = dy->op_layernorm_backward(dy, scale, bias, var, y, dscale, dbias, din, eps);
    if (r != OP_OK) return r;
    return din->op_add(din, residual, din);
}

namespace {
bool apart(const tensor_t& x, const tensor_t& y) {
    auto begin = [](const tensor_t& t) { return reinterpret_cast<uintptr_t>(t->data()); };
    auto end = [&](const tensor_t& t) { return begin(t) + t->items() * DataType_size(t->dtype()); };
    return end(x) <= begin(y) || end(y) <= begin(x);
}
bool same_tensor(const tensor_t& x, const tensor_t& y) {
    return x->data() == y->data() && x->items() == y->items() && x->dtype() == y->dtype();
}
bool same_shape(const tensor_t& x, const tensor_t& y) {
    bool same = x->shape().dim() == y->shape().dim();
    for (size_t i = 0; same && i < x->shape().dim(); i++) same = x->shape()[i] == y->shape()[i];
    return same;
}
// `next` starts where `t` ends
bool adjacent(const tensor_t& t, const tensor_t& next) {
    return t->dtype() == next->dtype() && t->items() == next->items() &&
           static_cast<const char*>(t->data()) + t->items() * DataType_size(t->dtype()) == static_cast<const char*>(next->data());
}
}  // namespace

namespace {
// A linear layer's operands (lin: x w b y), checked as op_linear checks them.
bool linear_ok(const tensor_t* lin) {
    const tensor_t &x = lin[0], &w = lin[1], &b = lin[2], &y = lin[3];
    if (!dev(x) || !dev(w) || !dev_f32(b) || !dev(y) || x->shape().dim() != 3 || w->shape().dim() != 2) return false;
    const size_t n = x->shape()[0] * x->shape()[1], in = x->shape()[2], out = w->shape()[0];
    return w->shape()[1] == in && b->items() == out && y->items() == n * out;
}
// `count` linear layers of one x (lin: count x (x w b y)) whose weights, biases and outputs lie one behind the other.
bool linears_ok(const tensor_t* lin, int count) {
    for (int i = 0; i < count; i++) {
        const tensor_t* l = lin + 4 * i;
        if (!linear_ok(l) || !same_tensor(l[0], lin[0])) return false;
        // nothing that one of them writes is read or written by another
        for (int j = 0; j < count; j++)
            for (int k = 0; k < 3; k++)
                if (!apart(l[3], lin[4 * j + k])) return false;
        if (i > 0)
            for (int k = 1; k < 4; k++)
                if (!adjacent(lin[4 * i - 4 + k], l[k])) return false;
    }
    return true;
}
// Runs them with x as `x` says (the layers' own, or its image in the products' type).
int linears(const Operand& x, const tensor_t* lin, int count, int compute) {
    const int64_t n = (int64_t)(lin[0]->shape()[0] * lin[0]->shape()[1]), in = (int64_t)lin[0]->shape()[2];
    const int64_t out = (int64_t)lin[1]->shape()[0];
    const size_t need = compute == BR_GEMM_F32 ? 0 : br_hip_linear_group_workspace(count, n, out, in, x.dtype, code(lin[1]));
    void* ws = need ? ComputingContext::gemm_staging(0, need) : nullptr;
    return br_hip_linear_group(x.ptr, x.dtype, lin[1]->data(), code(lin[1]), static_cast<const float*>(lin[2]->data()),
                               lin[3]->data(), code(lin[3]), count, n, out, in, compute, ws, need, stream());
}
// op_linear followed by op_add, one product where the sum is of its output and a residual.
ComputingReturn linear_then_add(const Operand& x, const tensor_t* lin, const tensor_t* add) {
    const tensor_t& y = lin[3];
    bool fast = linear_ok(lin) && dev_f32(y) && dev_f32(add[0]) && dev_f32(add[1]) && dev_f32(add[2]);
    if (fast) {
        const bool first = same_tensor(add[0], y);
        const tensor_t &r = first ? add[1] : add[0], &sum = add[2];
        fast = first != same_tensor(add[1], y) && same_shape(add[0], add[1]) && y->shape().dim() <= 4 && r->items() == y->items() &&
               sum->items() == y->items() &&
               apart(y, r) && apart(y, sum) && (same_tensor(sum, r) || apart(sum, r)) && y->items() % 4 == 0;
        for (int k = 0; fast && k < 3; k++) fast = apart(y, lin[k]) && apart(sum, lin[k]);
        if (fast) {
            const int compute = pick_compute({lin[0], lin[1], y});
            const int64_t n = (int64_t)(lin[0]->shape()[0] * lin[0]->shape()[1]), in = (int64_t)lin[0]->shape()[2];
            const int64_t out = (int64_t)lin[1]->shape()[0];
            const size_t need = compute == BR_GEMM_F32 ? 0 : br_hip_gemm_staged_workspace(0, 1, n, out, in, x.dtype, code(lin[1]), 1);
            void* ws = need ? ComputingContext::gemm_staging(0, need) : nullptr;
            BR_OP(br_hip_linear_sum(x.ptr, x.dtype, lin[1]->data(), code(lin[1]), static_cast<const float*>(lin[2]->data()),
                                    static_cast<const float*>(r->data()), static_cast<float*>(y->data()),
                                    static_cast<float*>(sum->data()), n, out, in, compute, ws, need, stream()));
            return OP_OK;
        }
    }
    if (x.ptr != lin[0]->data()) {
        // (x's image is what the product would have made of it)
        const int64_t n = (int64_t)(lin[0]->shape()[0] * lin[0]->shape()[1]), in = (int64_t)lin[0]->shape()[2];
        const int64_t out = (int64_t)lin[1]->shape()[0];
        BR_OP(product(0, 1, n, out, in, 1.0f, x.ptr, x.dtype, in, 0, lin[1]->data(), code(lin[1]), in, 0, 0, y->data(), code(y), out,
                      0, static_cast<const float*>(lin[2]->data()), 1, pick_compute({lin[0], lin[1], y})));
    } else {
        const ComputingReturn r = lin[0]->op_linear(lin[0], lin[1], lin[2], y);
        if (r != OP_OK) return r;
    }
    return add[0]->op_add(add[0], add[1], add[2]);
}
}  // namespace

ComputingReturn hip_linears(const tensor_t* lin, int count) {
    if (linears_ok(lin, count)) {
        BR_OP(linears(Operand{lin[0]->data(), code(lin[0])}, lin, count, pick_compute({lin[0], lin[1], lin[3]})));
        return OP_OK;
    }
    for (int i = 0; i < count; i++) {
        const tensor_t* l = lin + 4 * i;
        const ComputingReturn r = l[0]->op_linear(l[0], l[1], l[2], l[3]);
        if (r != OP_OK) return r;
    }
    return OP_OK;
}

// The LayerNorm kernel has every row of y in registers: with 16-bit products it writes y's image for the layers, too.
ComputingReturn hip_layernorm_then_linears(const tensor_t* ln, float eps, const tensor_t* lin, int count) {
    const tensor_t &x = ln[0], &mean = ln[1], &var = ln[2], &scale = ln[3], &bias = ln[4], &y = ln[5];
    bool fast = linears_ok(lin, count) && same_tensor(lin[0], y) && x->shape().dim() == 3;
    for (int i = 0; fast && i < 6; i++) fast = dev_f32(ln[i]);
    const int compute = fast ? pick_compute({y, lin[1], lin[3]}) : BR_GEMM_F32;
    if (fast && compute != BR_GEMM_F32) {
        const int64_t rows = (int64_t)(x->shape()[0] * x->shape()[1]), cols = (int64_t)x->shape()[2];
        if ((int64_t)mean->items() >= rows && (int64_t)var->items() >= rows && (int64_t)scale->items() == cols &&
            (int64_t)bias->items() == cols && y->items() == x->items() && cols % 8 == 0) {
            const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            void* y16 = ComputingContext::gemm_staging(1, y->items() * 2);
            const int rc = br_hip_layernorm_fwd_copy16(
                static_cast<const float*>(x->data()), static_cast<const float*>(scale->data()),
                static_cast<const float*>(bias->data()), static_cast<float*>(y->data()), y16, native,
                static_cast<float*>(mean->data()), static_cast<float*>(var->data()), rows, cols, eps, stream());
            if (rc != BR_ERR_TODO) {
                BR_OP(rc);
                BR_OP(linears(Operand{y16, native}, lin, count, compute));
                return OP_OK;
            }
        }
    }
    const ComputingReturn r = x->op_layernorm(x, mean, var, scale, bias, y, eps);
    return r != OP_OK ? r : hip_linears(lin, count);
}

ComputingReturn hip_linear_then_add(const tensor_t* lin, const tensor_t* add) {
    return linear_then_add(Operand{lin[0]->data(), code(lin[0])}, lin, add);
}

// op_gelu(u, v), op_linear(lin) and op_add(add): the GELU writes the image of an fp32 v that the product reads.
ComputingReturn hip_gelu_linear_then_add(const tensor_t& u, const tensor_t& v, const tensor_t* lin, const tensor_t* add) {
    if (dev_f32(u) && dev_f32(v) && u->items() == v->items() && linear_ok(lin) && same_tensor(lin[0], v)) {
        const int compute = pick_compute({v, lin[1], lin[3]});
        if (compute != BR_GEMM_F32 && lin[0]->shape()[2] % 8 == 0) {
            const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            void* v16 = ComputingContext::gemm_staging(1, v->items() * 2);
            const int rc = br_hip_gelu_fwd_copy16(static_cast<const float*>(u->data()), static_cast<float*>(v->data()), v16, native,
                                                  (int64_t)v->items(), stream());
            if (rc != BR_ERR_TODO) {
                BR_OP(rc);
                return linear_then_add(Operand{v16, native}, lin, add);
            }
        }
    }
    const ComputingReturn r = u->op_gelu(u, v);
    return r != OP_OK ? r : hip_linear_then_add(lin, add);
}

namespace {
// The backward pass of a linear layer whose input is a GELU's output and whose input gradient is written over it, then of
// that GELU and of the layer ahead (low: x w b x_g w_g b_g of the first, its dy being `dy`; tail: dy u du of the GELU and
// dy x w b x_g w_g b_g of the layer ahead).  The first layer's two products can only share a launch where neither
// overwrites what the other reads: its input gradient goes to the workspace, and the GELU's pass, which reads it anyway,
// leaves it where it belongs.  A block's forward and backward pass on [64 x 256] 78.6 -> 76.1 us, on [78 x 1024]
// 135.7 -> 135.0.  BR_ERR_TODO: not of that form, or not small; nothing has been done.
int gelu_between(const Operand& dy, const tensor_t* low, const tensor_t* tail, int64_t n, int compute, const br_partial_sums* later) {
    const tensor_t &x = low[0], &w = low[1], &x_g = low[3], &w_g = low[4], &u = tail[1], &du = tail[2];
    const tensor_t* top = tail + 3;   // dy x w b x_g w_g b_g
    const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
    if (compute == BR_GEMM_F32 || dy.dtype != native || !dev(x) || code(x) != native || !same_tensor(x_g, x) || !same_tensor(tail[0], x) ||
        !dev(u) || !dev(du) || code(u) != native || code(du) != native || u->items() != x->items() || du->items() != x->items() ||
        !same_tensor(top[0], du) || du->shape().dim() != 3 || x->shape().dim() != 3)
        return BR_ERR_TODO;
    const int64_t mid = (int64_t)x->shape()[2], out = (int64_t)w->shape()[0];
    if ((int64_t)w->items() != out * mid || (int64_t)du->shape()[2] != mid || mid % 8 != 0 || !dev(top[1]) || !dev(top[2]) ||
        !dev(top[4]) || !dev(top[5]) || !dev_f32(top[6]) || top[1]->shape().dim() != 3)
        return BR_ERR_TODO;
    const int64_t in = (int64_t)top[1]->shape()[2];
    if ((int64_t)top[1]->items() != n * in || (int64_t)top[2]->items() != mid * in || (int64_t)top[4]->items() != n * in || (int64_t)top[5]->items() != mid * in ||
        (int64_t)top[6]->items() != mid || pick_compute({du, top[1], top[2]}) != compute)
        return BR_ERR_TODO;
    if (!(same_tensor(u, du) || apart(u, du)) || !apart(du, x) || !apart(u, x) || !apart(x, w) || !apart(x, w_g) || !apart(du, w_g) || !apart(u, w_g) ||
        !apart(top[6], x) || !apart(top[6], u) || !apart(top[6], du))
        return BR_ERR_TODO;
    auto off = [](const tensor_t& t) { return (reinterpret_cast<uintptr_t>(t->data()) & 15) != 0; };
    if (off(x) || off(u) || off(du) || !br_hip_bias_gelu_bwd_copies(n, mid) ||
        br_hip_gemm_pair_kernel(out, mid, n, 1, n, mid, out, 1, compute) < 0)
        return BR_ERR_TODO;
    // partial sums that wait to be added up lie at the workspace's head
    const size_t sums = later && later->partials ? (size_t)(later->arrays * later->parts * later->cols) * sizeof(float) : 0;
    const size_t at = (sums + 255) / 256 * 256;
    if (at + (size_t)(n * mid) * 2 > head_bytes()) return BR_ERR_TODO;
    void* x_grad = static_cast<char*>(ComputingContext::workspace) + at;
    int rc = two_products({1, 0, out, mid, n, unlift(), dy.ptr, dy.dtype, out, 0, x->data(), native, mid, 0, w_g->data(), code(w_g), mid, 0, 1},
                          {0, 0, n, mid, out, 1.0f, dy.ptr, dy.dtype, out, 0, w->data(), code(w), mid, 0, x_grad, native, mid, 0, 1},
                          nullptr, compute, later);
    if (rc != BR_OK) return rc;
    rc = br_hip_bias_gelu_bwd_copy(x_grad, u->data(), nullptr, du->data(), static_cast<float*>(top[6]->data()), x->data(), native, n,
                                   mid, unlift(), stream());
    if (rc != BR_OK) return rc;
    return linear_backward_products(Operand{du->data(), native}, top[1], top[2], top[4], top[5], n, in, mid, compute);
}
}  // namespace

ComputingReturn hip_linear_gelu_linear_backward(const tensor_t* lin, const tensor_t* tail) {
    const tensor_t &dy = lin[0], &x = lin[1], &w = lin[2];
    if (dev_f32(dy) && dy->shape().dim() == 3 && dev(x) && x->shape().dim() == 3 && dev(w) && w->shape().dim() == 2 && dev(lin[4]) &&
        dev(lin[5]) && dev_f32(lin[6])) {
        const int64_t n = (int64_t)(dy->shape()[0] * dy->shape()[1]), out = (int64_t)dy->shape()[2], in = (int64_t)x->shape()[2];
        const int compute = pick_compute({dy, x, w});
        if (compute != BR_GEMM_F32 && out % 8 == 0 && (int64_t)x->items() == n * in && (int64_t)w->items() == out * in &&
            (int64_t)lin[5]->items() == out * in && (int64_t)lin[6]->items() == out &&
            same_tensor(lin[4], x)) {
            // (the first pass of op_linear_backward)
            const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            const size_t need = br_hip_colsum_workspace(n, out);
            void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
            void* dy16 = ComputingContext::gemm_staging(1, (size_t)(n * out) * 2);
            BR_OP(br_hip_colsum_cast(static_cast<const float*>(dy->data()), static_cast<float*>(lin[6]->data()), dy16, native, n, out,
                                     unlift(), ws, need, stream()));
            const int rc = gelu_between(Operand{dy16, native}, lin + 1, tail, n, compute, nullptr);
            if (rc != BR_ERR_TODO) {
                BR_OP(rc);
                return OP_OK;
            }
            BR_OP(linear_backward_products(Operand{dy16, native}, x, w, lin[4], lin[5], n, in, out, compute));
            return hip_gelu_linear_backward(tail[0], tail[1], tail[2], tail[4], tail[5], tail[6], tail[7], tail[8], tail[9]);
        }
    }
    const ComputingReturn r = dy->op_linear_backward(dy, x, w, lin[3], lin[4], lin[5], lin[6]);
    if (r != OP_OK) return r;
    return hip_gelu_linear_backward(tail[0], tail[1], tail[2], tail[4], tail[5], tail[6], tail[7], tail[8], tail[9]);
}

// op_layernorm_backward(ln[0..7], eps) followed by op_add(add[0], add[1], add[2]) of its din and a residual, and, unless
// lin is null, by op_linear_backward(lin[0..6]) of that sum.  One pass of the LayerNorm kernel leaves din, the sum, and for
// the linear layer the sum's 16-bit image and its bias gradient; anything else runs as the operators.
ComputingReturn hip_layernorm_backward_then_add(const tensor_t* ln, float eps, const tensor_t* add, const tensor_t* lin) {
    const tensor_t &dy = ln[0], &scale = ln[1], &bias = ln[2], &var = ln[3], &y = ln[4], &dscale = ln[5], &dbias = ln[6], &din = ln[7];
    const bool first = same_tensor(add[0], din);
    const tensor_t &residual = first ? add[1] : add[0], &sum = add[2];
    bool fast = first != same_tensor(add[1], din) && (dev_f32(dy) && dy->shape().dim() == 3) && dev_f32(residual) && dev_f32(sum) &&
                same_shape(residual, din) && same_shape(add[first ? 0 : 1], dy) && sum->items() == dy->items() &&
                residual->items() == dy->items() && din->items() == dy->items();
    for (int i = 1; fast && i < 8; i++) fast = dev_f32(ln[i]);
    bool linear = false;
    if (fast) {
        const int64_t rows = (int64_t)(dy->shape()[0] * dy->shape()[1]), cols = (int64_t)dy->shape()[2];
        fast = y->items() == dy->items() && (int64_t)var->items() >= rows && (int64_t)dscale->items() == cols &&
               (int64_t)dbias->items() == cols && (int64_t)scale->items() == cols && (int64_t)bias->items() == cols &&
               // the sum is written row by row, beside din: over the rows of dy or of the residual, or apart from all
               apart(sum, din) && apart(sum, y) && apart(din, residual) && apart(din, y) && apart(din, dy) &&
               (same_tensor(sum, residual) || apart(sum, residual)) && (same_tensor(sum, dy) || apart(sum, dy));
        for (const tensor_t* t : {&scale, &bias, &var, &dscale, &dbias}) fast = fast && apart(sum, *t) && apart(din, *t);
        if (fast) {
            int compute = BR_GEMM_F32;
            int64_t in = 0;
            void* sum16 = nullptr;
            float* sums = nullptr;
            if (lin && same_tensor(lin[0], sum) && lin[0]->shape().dim() == 3 && dev(lin[1]) && lin[1]->shape().dim() == 3 &&
                dev(lin[2]) && dev(lin[4]) && dev(lin[5]) && dev_f32(lin[6]) && (int64_t)lin[0]->shape()[2] == cols) {
                compute = pick_compute({lin[0], lin[1], lin[2]});
                in = (int64_t)lin[1]->shape()[2];
                linear = compute != BR_GEMM_F32 && cols % 8 == 0 && (int64_t)lin[1]->items() == rows * in &&
                         (int64_t)lin[2]->items() == cols * in && (int64_t)lin[4]->items() == rows * in &&
                         (int64_t)lin[5]->items() == cols * in && (int64_t)lin[6]->items() == cols;
                // the bias gradient is written before the LayerNorm's operands have all been read
                for (int i = 0; i < 8; i++) linear = linear && apart(lin[6], ln[i]);
                linear = linear && apart(lin[6], residual) && apart(lin[6], sum) && apart(lin[6], lin[1]) && apart(lin[6], lin[2]);
            }
            const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            if (linear) {
                sum16 = ComputingContext::gemm_staging(1, (size_t)(rows * cols) * 2);
                sums = static_cast<float*>(lin[6]->data());
            }
            const size_t need = br_hip_layernorm_bwd_sums_workspace(rows, cols);
            void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
            br_partial_sums later = {};
            auto run = [&]() {
                return br_hip_layernorm_bwd_add(
                    static_cast<const float*>(dy->data()), static_cast<const float*>(y->data()),
                    static_cast<const float*>(scale->data()), static_cast<const float*>(bias->data()),
                    static_cast<const float*>(var->data()), static_cast<const float*>(residual->data()),
                    static_cast<float*>(dscale->data()), static_cast<float*>(dbias->data()), static_cast<float*>(din->data()),
                    static_cast<float*>(sum->data()), sum16, native, sums, rows, cols, eps, unlift(), linear ? &later : nullptr, ws,
                    need, stream());
            };
            int rc = run();
            if (rc == BR_ERR_TODO && linear) {
                linear = false;
                sum16 = nullptr;
                sums = nullptr;
                rc = run();
            }
            fast = rc != BR_ERR_TODO;
            if (fast) BR_OP(rc);
            if (fast && linear)
                BR_OP(linear_backward_products(Operand{sum16, native}, lin[1], lin[2], lin[4], lin[5], rows, in, cols, compute, nullptr,
                                               &later));
        }
    }
    if (!fast) {
        ComputingReturn r = dy->op_layernorm_backward(dy, scale, bias, var, y, dscale, dbias, din, eps);
        if (r != OP_OK) return r;
        r = add[0]->op_add(add[0], add[1], add[2]);
        if (r != OP_OK) return r;
    }
    if (lin && !(fast && linear)) return lin[0]->op_linear_backward(lin[0], lin[1], lin[2], lin[3], lin[4], lin[5], lin[6]);
    return OP_OK;
}

// The backward pass of the query, key and value layers as the model scripts have it: acc = 0, then for each layer
// op_linear_backward into `tmp` and acc += tmp.  lin: 3 x (dy x w b x_g w_g b_g).  Where the three read one x, their
// weights and gradients lie one behind the other and tmp is not read afterwards (the caller's word), it is the backward
// pass of ONE layer of three times the outputs: the gradients are packed side by side in the products' type, summed over
// rows on the way, and two products are left of six.  BR_ERR_TODO: not of that form, nothing has been done.
int hip_qkv_backward(const tensor_t& acc, const tensor_t* lin) {
    const tensor_t &x = lin[1], &tmp = lin[4];
    if (!dev_f32(acc) || !dev(x) || x->shape().dim() != 3 || !dev_f32(tmp) || tmp->items() != x->items() || acc->items() != x->items())
        return BR_ERR_TODO;
    const int64_t n = (int64_t)(x->shape()[0] * x->shape()[1]), in = (int64_t)x->shape()[2];
    const int64_t out = (int64_t)(lin[6]->items());
    for (int i = 0; i < 3; i++) {
        const tensor_t* l = lin + 7 * i;
        if (!dev_f32(l[0]) || l[0]->shape().dim() != 3 || (int64_t)(l[0]->shape()[0] * l[0]->shape()[1]) != n ||
            (int64_t)l[0]->shape()[2] != out || !same_tensor(l[1], x) || l[1]->shape().dim() != 3 ||
            (int64_t)l[1]->shape()[2] != in || !dev(l[2]) || !same_tensor(l[4], tmp) || !dev_f32(l[5]) || !dev_f32(l[6]) ||
            (int64_t)l[2]->items() != out * in || (int64_t)l[5]->items() != out * in || (int64_t)l[6]->items() != out)
            return BR_ERR_TODO;
        if (i > 0 && !(adjacent(lin[7 * i - 5], l[2]) && adjacent(lin[7 * i - 2], l[5]) && adjacent(lin[7 * i - 1], l[6])))
            return BR_ERR_TODO;
        // what is written is neither read nor written by another part
        for (const tensor_t* t : {&l[0], &l[1], &l[2]}) {
            if (!apart(acc, *t) || !apart(tmp, *t)) return BR_ERR_TODO;
            for (int j = 0; j < 3; j++)
                if (!apart(lin[7 * j + 5], *t) || !apart(lin[7 * j + 6], *t)) return BR_ERR_TODO;
        }
        for (const tensor_t* t : {&l[5], &l[6]})
            if (!apart(acc, *t) || !apart(tmp, *t) || !apart(l[5], lin[6]) || !apart(lin[5], l[6])) return BR_ERR_TODO;
    }
    if (!apart(acc, tmp)) return BR_ERR_TODO;
    const int compute = pick_compute({lin[0], x, lin[2]});
    const int native = compute == BR_GEMM_F16 ? BR_F16 : compute == BR_GEMM_BF16 ? BR_BF16 : BR_F32;
    // one workgroup walks all rows of its columns
    if (out % 8 != 0 || n > 4096) return BR_ERR_TODO;
    // fp32: one sum over three times the K is as exact as three sums on the kernel that adds up in pieces
    auto aligned = [](const tensor_t& t) { return reinterpret_cast<uintptr_t>(t->data()) % 16 == 0; };
    if (native == BR_F32 && (in % 4 != 0 || !aligned(x) || !aligned(lin[2]))) return BR_ERR_TODO;
    void* packed = ComputingContext::gemm_staging(1, (size_t)(n * 3 * out) * (native == BR_F32 ? 4 : 2));
    const float* dy[3] = {static_cast<const float*>(lin[0]->data()), static_cast<const float*>(lin[7]->data()),
                          static_cast<const float*>(lin[14]->data())};
    const int rc = br_hip_pack_colsum(dy, 3, static_cast<float*>(lin[6]->data()), packed, native, n, out, unlift(), stream());
    if (rc != BR_OK) return rc;
    return linear_backward_products(Operand{packed, native}, x, lin[2], acc, lin[5], n, in, 3 * out, compute);
}

// `op.layernorm_backward_add` followed by the `op.linear_backward` whose dy is the LayerNorm's din: the
// LayerNorm kernel has every row of din in registers, so it also writes the 16-bit image the two products read
// and the partial column sums that make the bias gradient -- the pass over din that op.linear_backward starts
// with does not run.  Anything the fused kernel declines runs as the two operators.  The GELU's and the next layer's
// backward of `tail` (null: none) are joined to it where gelu_between takes them, which *tail_done says.
namespace {
ComputingReturn layernorm_backward_add_linear_backward(
    const tensor_t& dy, const tensor_t& scale, const tensor_t& bias, const tensor_t& var, const tensor_t& y,
    const tensor_t& dscale, const tensor_t& dbias, const tensor_t& residual, const tensor_t& din, float eps,
    const tensor_t& x, const tensor_t& weight, const tensor_t& lbias, const tensor_t& x_g, const tensor_t& weight_g,
    const tensor_t& bias_g, const tensor_t* tail, bool* tail_done) {
    bool fast = dev_f32(dy) && dev_f32(scale) && dev_f32(bias) && dev_f32(var) && dev_f32(y) && dev_f32(dscale) &&
                dev_f32(dbias) && dev_f32(residual) && dev_f32(din) && dy->shape().dim() == 3 && dev(x) &&
                dev(weight) && dev(x_g) && dev(weight_g) && dev_f32(bias_g) && x->shape().dim() == 3 &&
                din->shape().dim() == 3;
    if (fast) {
        const int64_t rows = (int64_t)(dy->shape()[0] * dy->shape()[1]);
        const int64_t cols = (int64_t)dy->shape()[2], in = (int64_t)x->shape()[2];
        const int compute = pick_compute({din, x, weight});
        fast = y->items() == dy->items() && (int64_t)var->items() >= rows && din->items() == dy->items() &&
               residual->items() == dy->items() && (int64_t)dscale->items() == cols && (int64_t)dbias->items() == cols &&
               (int64_t)scale->items() == cols && (int64_t)bias->items() == cols && din->data() != y->data() &&
               compute != BR_GEMM_F32 && cols % 8 == 0 && (int64_t)x->items() == rows * in &&
               (int64_t)weight->items() == cols * in && (int64_t)x_g->items() == rows * in &&
               (int64_t)weight_g->items() == cols * in && (int64_t)bias_g->items() == cols &&
               // the gradients this call writes must not be each other or an input of the products
               bias_g->data() != dscale->data() && bias_g->data() != dbias->data();
        if (fast) {
            const int native = compute == BR_GEMM_F16 ? BR_F16 : BR_BF16;
            const size_t need = br_hip_layernorm_bwd_sums_workspace(rows, cols);
            void* ws = need <= head_bytes() ? ComputingContext::workspace : ComputingContext::scratch(need);
            void* d16 = ComputingContext::gemm_staging(1, (size_t)(rows * cols) * 2);
            // dgamma, dbeta and the bias gradient are added up beside the products
            br_partial_sums later = {};
            const int rc = br_hip_layernorm_bwd_add(
                static_cast<const float*>(dy->data()), static_cast<const float*>(y->data()),
                static_cast<const float*>(scale->data()), static_cast<const float*>(bias->data()),
                static_cast<const float*>(var->data()), static_cast<const float*>(residual->data()),
                static_cast<float*>(dscale->data()), static_cast<float*>(dbias->data()), nullptr,
                static_cast<float*>(din->data()), d16, native, static_cast<float*>(bias_g->data()), rows, cols, eps,
                unlift(), &later, ws, need, stream());
            if (rc != BR_ERR_TODO) {
                BR_OP(rc);
                if (tail) {
                    const tensor_t low[6] = {x, weight, lbias, x_g, weight_g, bias_g};
                    const int rg = gelu_between(Operand{d16, native}, low, tail, rows, compute, &later);
                    if (rg != BR_ERR_TODO) {
                        BR_OP(rg);
                        *tail_done = true;
                        return OP_OK;
                    }
                }
                BR_OP(linear_backward_products(Operand{d16, native}, x, weight, x_g, weight_g, rows, in, cols, compute, nullptr,
                                               &later));
                return OP_OK;
            }
        }
    }
    const ComputingReturn r = hip_layernorm_backward_add(dy, scale, bias, var, y, dscale, dbias, residual, din, eps);
    if (r != OP_OK) return r;
    return din->op_linear_backward(din, x, weight, lbias, x_g, weight_g, bias_g);
}
}  // namespace

ComputingReturn hip_layernorm_backward_add_linear_backward(
    const tensor_t& dy, const tensor_t& scale, const tensor_t& bias, const tensor_t& var, const tensor_t& y,
    const tensor_t& dscale, const tensor_t& dbias, const tensor_t& residual, const tensor_t& din, float eps,
    const tensor_t& x, const tensor_t& weight, const tensor_t& lbias, const tensor_t& x_g, const tensor_t& weight_g,
    const tensor_t& bias_g, const tensor_t* tail) {
    bool tail_done = false;
    const ComputingReturn r = layernorm_backward_add_linear_backward(dy, scale, bias, var, y, dscale, dbias, residual, din, eps, x,
                                                                     weight, lbias, x_g, weight_g, bias_g, tail, &tail_done);
    if (r != OP_OK || !tail || tail_done) return r;
    return hip_gelu_linear_backward(tail[0], tail[1], tail[2], tail[4], tail[5], tail[6], tail[7], tail[8], tail[9]);
}

template struct HIPTensor<DataType::Float>;
template struct HIPTensor<DataType::F16>;
template struct HIPTensor<DataType::BF16>;

tensor_t create_cuda_float(std::vector<size_t>& shape_) {
    ShapeType shape(shape_);
    return std::make_shared<TensorType>(new HIPTensor<DataType::Float>(shape), shape);
}

tensor_t create_cuda_f16(std::vector<size_t>& shape_) {
    ShapeType shape(shape_);
    return std::make_shared<TensorType>(new HIPTensor<DataType::F16>(shape), shape);
}

tensor_t create_cuda_bf16(std::vector<size_t>& shape_) {
    ShapeType shape(shape_);
    return std::make_shared<TensorType>(new HIPTensor<DataType::BF16>(shape), shape);
}

}  // namespace br
