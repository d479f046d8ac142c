// MFMA GEMM for small and ragged 16-bit products and for all fp32 ones:
// direct-to-LDS loads with hardware bounds checks, waves that split K among
// themselves.
//
//   C[b][i,j] = alpha * sum_p opA[b][i,p] * opB[b][p,j] (+ C) (+ bias[j])
//
// gemm_flex_kernel: a workgroup owns a BM x BN tile of C (64 x 64 or 32 x 32) and EVERY of its
// KW waves computes the whole tile over its own share of K: wave w takes the
// 128-byte K steps w, w + KW, w + 2 KW, ...  Each wave loads its steps into LDS
// buffers of its own and reads them back itself, so the K loop has no barrier:
// a wave waits for its own loads (vmcnt) and nothing else.  At the end the KW
// accumulators meet in LDS and are added in wave order.
//
// Why: a product of a few hundred rows has few output tiles, and what bounds
// it is the latency of one workgroup's walk along K and the 64 B per clock a CU
// takes from L2.  Small tiles give more workgroups, splitting K inside the
// workgroup shortens the walk KW times without partial tiles in memory, and a
// wave that owns the whole tile reads half the LDS bytes per MFMA that four
// waves with a quarter of the tile each would.
//
// Loads are buffer loads through a resource that ends where the operand ends:
// rows of C past m or n and k-values past K read as zero, so K need not be a
// multiple of anything for a row-contiguous operand and of 8 for a k-contiguous
// one (whose tail chunk would otherwise run into the next row; a staged copy
// with zero-filled row ends makes any K qualify).
//
// Measured (fp16, before / after; before = 256 x 128 tiles, or the guarded
// register-staged kernel where K is ragged): [64 x 768] K = 256 12.1 -> 3.4 us,
// [78 x 1024] K = 4096 20.4 -> 8.7, [1000 x 1024] K = 1024 21.9 -> 8.5,
// [1024 x 1024] weight gradient of 1000 tokens 106 -> 8.9, [200 x 512] from
// K = 32008 in eight slices 3490 -> 19.  What bounds it: with 16 or more K steps
// a wave, the CU's loads into LDS (about 40 B per clock); below that launch,
// the first loads' latency and the sum through LDS, 3.3 us for a 32 x 32 and 5
// for a 64 x 64 tile.  A second buffer per wave, or the loads dealt out between
// the products, measured equal or 5-15 % slower on the 64 x 64 tile.
//
// fp32 products run on the same kernel, and on the 16-bit matrix instructions: a value is the sum of three bf16 values to 24
// bits, and six of the nine products of such parts are all that a float holds of the whole.  They take 192 clocks for
// 16 k-values of a 32 x 32 block, v_mfma_f32_32x32x2_f32 512.  With those / with parts, us (and the error against 64 bits, 2-norm):
// [512 x 1024] K = 1024 14.8 / 13.4 (1.6e-7 / 1.0e-7), K = 4096 47.8 / 38.9 (1.7e-7 / 1.6e-7), [512 x 4096] K = 1024 47.0 / 32.5 (1.6e-7 /
// 1.0e-7), [1024 x 8192] K = 2048 313 / 230 (1.6e-7 / 1.5e-7), [64 x 2048] K = 8192 45.1 / 37.3 (1.8e-7 / 1.7e-7); a launch of under
// 6 us takes as long as before.  What bounds it: many tiles, the rate of the 16-bit instructions at the clock they leave (150
// TFLOP/s are 900 of theirs); one small tile to a CU, the loads into LDS, 25-30 B per clock whatever the tile and however many are
// in flight (a second and a third buffer per wave measured equal or slower).
#pragma once
#include <type_traits>

#include "gemm_mfma16.hpp"
#include "gemm_plan.hpp"
#include "lds_direct.hpp"

namespace brk {
namespace gemm16 {

// Operand tile of ROWS rows by 128 bytes of k (64 16-bit or 32 fp32 values), loaded by one wave in 16-byte granules,
// or in single fp32 values (WORDS) where rows are not aligned to granules.
template <int CT, int ROWS, bool KSTR, bool WORDS>
struct FlexTile {
    static constexpr int kSize = CT == BR_GEMM_F32 ? 4 : 2;      // bytes of an element
    static constexpr int kPer = 16 / kSize;                      // elements of a granule
    static constexpr int kStep = 128 / kSize;                    // k-values of a step
    static constexpr int kBytes = ROWS * 128;
    static constexpr int kInstr = kBytes / (WORDS ? 256 : 1024);  // wave-wide loads of a tile
    static constexpr int kGranulesPerK = ROWS / kPer;             // row contiguous: granules of a k-row
    // Loads whose offsets a lane holds.  Value by value there are up to 32 of an operand, and the 64 registers of a 64 x 64 tile
    // left one wave to a SIMD: held are eight, the others' lie kFar rows (row contiguous: k-rows) and a multiple of it further on.
    // All held / eight, us, operands off 16-byte boundaries: [987 x 4608] from K = 1152 131 / 89, [501 x 501] from 65, 16 products,
    // 38.4 / 19.0, [700 x 2049] from 513 29.7 / 19.1; one tile to a CU the same to within 5 %.
    static constexpr int kHeld = WORDS ? 8 : kInstr;
    static constexpr int kFar = kHeld * (WORDS ? 16 : 64) / (KSTR ? kGranulesPerK : 8);
    static_assert(kInstr % kHeld == 0, "whole sets of loads");
    static_assert(!WORDS || kSize == 4, "single values are fp32");

    // Row contiguous, where things lie in LDS.  16-bit: the transposing read of a fragment touches 4 k-rows x 64
    // bytes at a time; fp32: a fragment's reads touch 128 bytes each of k-rows k and k + 4.  Either has to fall on
    // different banks: by which granule of a k-row sits in slot c (c ^ swizzle), and for 32 fp32 rows (half the
    // banks wide) by keeping k-rows k and k + 4 side by side.
    static __device__ __forceinline__ int swizzle(int kk) {
        if (kSize == 4) return ROWS == 32 ? 0 : 8 * ((kk >> 2) & 1);
        return ROWS == 32 ? 0 : ROWS == 64 ? 4 * ((kk >> 1) & 1) : 4 * (kk & 3);
    }
    static __device__ __forceinline__ int place_of_k(int kk) {
        return kSize == 4 && ROWS == 32 ? (kk & ~7) + (kk & 3) * 2 + ((kk >> 2) & 1) : kk;
    }
    static __device__ __forceinline__ int k_in_place(int place) {
        return kSize == 4 && ROWS == 32 ? (place & ~7) + ((place & 7) >> 1) + 4 * (place & 1) : place;
    }
    static __device__ __forceinline__ int slot(int q, int lane) { return WORDS ? q * 16 + (lane >> 2) : q * 64 + lane; }
    static __device__ __forceinline__ int word(int lane) { return WORDS ? lane & 3 : 0; }
    // k (relative to the step) of the first element this lane fetches in its q-th load
    static __device__ __forceinline__ int k_of(int q, int lane) {
        const int s = slot(q, lane);
        if (KSTR) return k_in_place(s / kGranulesPerK);
        return ((s & 7) ^ ((s >> 4) & 7)) * kPer + word(lane);
    }
    // its byte offset from the tile's origin at the step's first k
    static __device__ __forceinline__ unsigned source_offset(int q, int lane, long long ld) {
        const int s = slot(q, lane);
        if (KSTR) {
            const int kk = k_of(q, lane), c = (s % kGranulesPerK) ^ swizzle(kk);
            return (unsigned)((kk * ld + c * kPer + word(lane)) * kSize);
        }
        return (unsigned)(((s >> 3) * ld + k_of(q, lane)) * kSize);
    }
    // LDS byte offset of the fragment of 32-row block `row_base`, sub-step ks (a quarter of the step)
    static __device__ __forceinline__ unsigned frag_offset(int row_base, int ks, int lane) {
        if (!KSTR) {
            const int r = row_base + (lane & 31), c = ks * 2 + (lane >> 5);
            return (unsigned)(r * 128 + ((c ^ ((r >> 1) & 7)) * 16));
        }
        if (kSize == 4) {
            const int r = row_base + (lane & 31), kk = ks * 8 + (lane >> 5) * 4;
            return (unsigned)(place_of_k(kk) * (ROWS * 4) + (((r >> 2) ^ swizzle(kk)) * 16) + (r & 3) * 4);
        }
        const int i = lane & 15, grp = lane >> 4;
        const int kk = ks * 16 + (grp >> 1) * 8 + (i >> 2);
        const int row16 = row_base + (grp & 1) * 16 + (i & 3) * 4;
        return (unsigned)(kk * (ROWS * 2) + (((row16 >> 3) ^ swizzle(kk)) * 16) + (row16 & 7) * 2);
    }
    // 16-bit: row lane % 32, k = 16 ks + 8 (lane / 32) + 0..7;  fp32: k = 8 ks + 4 (lane / 32) + 0..3
    static __device__ __forceinline__ u32x4 fragment(const lds_byte* tile, unsigned off) {
        if (!KSTR) return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(tile + off);
        if (kSize == 4) {
            typedef __attribute__((address_space(3))) unsigned lds_u32;
            constexpr int kNext = ROWS == 32 ? 2 * ROWS : ROWS;   // words from k to k + 1
            const lds_u32* p = (const lds_u32*)(tile + off);
            return mk4(p[0], p[kNext], p[2 * kNext], p[3 * kNext]);
        }
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off + 4 * ROWS * 2));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        return mk4(l2.x, l2.y, h2.x, h2.y);
    }
    static __device__ __forceinline__ void load(unsigned dst, int q, unsigned off, const buffer_rsrc& r) {
        if (WORDS) buffer_dtl_load_dword(dst + q * 256, off, r);
        else buffer_dtl_load(dst + q * 1024, off, r);
    }
};

typedef float flex_f32x4 __attribute__((ext_vector_type(4)));

typedef __attribute__((address_space(3))) flex_f32x4 lds_f32x4;

// The end of a tile, in two parts with a barrier between them.  First every wave leaves its accumulators in BM x BN
// floats of LDS of its own at `mem`:
// acc[i][j][v] is C[row, col] with row = i*32 + lane%32, col = j*32 + (v/4)*8 + (lane/32)*4 + v%4; quad c of row r goes
// to slot c ^ (r % 8) of the row (writes of 16 rows and reads along a row both touch every bank once).
template <int BM, int BN>
__device__ __forceinline__ void flex_park(const f32x16 (&acc)[BM / 32][BN / 32], lds_byte* mem, int lane) {
    constexpr int FM = BM / 32, FN = BN / 32, QN = BN / 4;
    lds_f32x4* const sums = (lds_f32x4*)mem;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = i * 32 + (lane & 31), c = j * 8 + q * 2 + (lane >> 5);
                flex_f32x4 v;
                v.x = acc[i][j][4 * q]; v.y = acc[i][j][4 * q + 1]; v.z = acc[i][j][4 * q + 2]; v.w = acc[i][j][4 * q + 3];
                sums[r * QN + (c ^ (r & 7))] = v;
            }
}

// Then THREADS threads add up the KW accumulators, `wave_bytes` apart from lds_all on, in wave order, and store C.
template <int BM, int BN, int KW, int THREADS, typename TC, bool GELU>
__device__ __forceinline__ void flex_emit(const GemmArgs& g, const lds_byte* lds_all, int wave_bytes, int row0, int col0, int b) {
    constexpr int QN = BN / 4;
    TC* c_base = static_cast<TC*>(g.c) + b * g.sc;
    TC* c2_base = GELU ? static_cast<TC*>(g.c2) + b * g.sc : nullptr;
    const TC* old_base = g.addend ? static_cast<const TC*>(g.addend) + b * g.sc : c_base;
    const float* const bias = g.bias ? g.bias + b * g.sbias : nullptr;
    const lds_f32x4* const all = (const lds_f32x4*)lds_all;
    constexpr int kQuads = BM * QN, kThreads = THREADS;
#pragma unroll
    for (int it = 0; it < (kQuads + kThreads - 1) / kThreads; it++) {
        const int e = it * kThreads + threadIdx.x;
        if (kQuads % kThreads != 0 && e >= kQuads) break;
        const int r = e / QN, c = e % QN;
        const int at = r * QN + (c ^ (r & 7));
        flex_f32x4 s = all[at];
#pragma unroll
        for (int w = 1; w < KW; w++) s += all[w * (wave_bytes / 16) + at];
        const int row = row0 + r, col = col0 + c * 4;
        if (row >= g.m) continue;
        const long long off = row * g.ldc + col;
        const int left = (int)(g.n - col);   // columns of C this quad covers
        float o[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            o[u] = g.alpha * s[u] + (bias && u < left ? bias[col + u] : 0.f);
            if (g.accumulate && u < left) o[u] += c_load<TC>(old_base + off + u);
            if (sizeof(TC) == 2) asm volatile("" : "+v"(o[u]));   // one fp32 value, then one rounding
        }
        if (left >= 4 && g.vec_c) {
            c_store4<TC>(c_base + off, o);
            if (GELU) {
#pragma unroll
                for (int u = 0; u < 4; u++) o[u] = gelu_one(o[u]);
                c_store4<TC>(c2_base + off, o);
            }
        } else {
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (u < left) {
                    c_store<TC>(c_base + off + u, o[u]);
                    if (GELU) c_store<TC>(c2_base + off + u, gelu_one(o[u]));
                }
        }
        if constexpr (!GELU && sizeof(TC) == 4) {
            if (g.sum) {
                float* const to = g.sum + b * g.sc + off;
                if (left >= 4 && g.vec_c) {
                    const float4 r = *reinterpret_cast<const float4*>(old_base + off);
                    *reinterpret_cast<float4*>(to) = make_float4(o[0] + r.x, o[1] + r.y, o[2] + r.z, o[3] + r.w);
                } else {
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (u < left) to[u] = o[u] + old_base[off + u];
                }
            }
        }
    }
}

// The three bf16 parts of eight fp32 values of a lane times 2^24, each the nearest to what the parts before it leave (those
// differences are exact).  bf16 has no bits below 2^-133: of a value below 2^-110 as it is the parts would hold fewer than 24, of
// one of 2^-125 eight.  Times 2^24 the lowest bit there is lies at 2^-125, and whatever an fp32 operand holds, its parts hold too.
// That multiplication is a fifth of the splitting (3 % of a launch, 4 to 7 % where one small tile is all a CU has).
// All of a part ahead of the next one, so that no value waits for its own last step: value by value a layer's backward products
// from 78 tokens take 31.0 us, so 28.6.
//
// A fragment's products with those of the other operand, hi hi, hi mid, mid hi, mid mid, hi lo, lo hi:
//   kAsParts        all but the first are added up in registers of their own: one rounding of the large sum for 16 k-values.
//                   Up to 256 k-values a wave (kApartUpTo): with 512 the largest entry's error passes that of the fp32
//                   instructions ([1024 x 8192] from K = 2048 1.23e-6 of the rms, 1.04e-6), with 1024 the 2-norm's too
//   kAsPartsFolded  all into one accumulator, which goes to a second one every 64 k-values, so that errors grow with the number
//                   of such sums and not with K (3-10 % slower)
//   kOneByOne       the fp32 instructions, folded likewise.  An operand of 2^104 or more, infinite or not a number, and a sum of
//                   2^80 or more make the parts' sums infinite or not a number: a wave that finds that in its sums walks once
//                   more, like this.
enum FlexWalk { kInTheirType, kAsParts, kAsPartsFolded, kOneByOne };
constexpr int kApartUpTo = 256;
constexpr float kPartsScale = 0x1p24f;
constexpr int kNotNumbers = 0x207;   // classes of v_cmp_class_f32: NaN and infinity
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void three_parts(const u32x4& first, const u32x4& second, u32x4& hi, u32x4& mid, u32x4& lo) {
    f32x2 v[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        v[e].x = __uint_as_float(e < 2 ? first[2 * e] : second[2 * e - 4]) * kPartsScale;
        v[e].y = __uint_as_float(e < 2 ? first[2 * e + 1] : second[2 * e - 3]) * kPartsScale;
    }
    auto next_part = [&](u32x4& to, bool last) {
#pragma unroll
        for (int e = 0; e < 4; e++) to[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(v[e], bf16x2));
        if (last) return;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e].x -= __uint_as_float(to[e] << 16);
            v[e].y -= __uint_as_float(to[e] & 0xffff0000u);
        }
    };
    next_part(hi, false);
    next_part(mid, false);
    next_part(lo, true);
}

// LDS of a workgroup of such tiles
template <int BM, int BN, int KW, int ST>
constexpr int flex_lds_bytes() { return KW * ST * (BM + BN) * 128; }

// Workgroup `id` of the `groups` a product has.  SLICES: it may be one of several slices of K (g.splits).
template <int CT, int BM, int BN, int KW, int ST, bool A_KSTR, bool B_KSTR, typename TC, bool GELU, bool WORDS, bool SLICES>
__device__ __forceinline__ void flex_product(const GemmArgs& g, unsigned id, unsigned groups, unsigned char* lds_raw) {
    using TA = FlexTile<CT, BM, A_KSTR, WORDS>;
    using TB = FlexTile<CT, BN, B_KSTR, WORDS>;
    constexpr int kSize = TA::kSize, KT = TA::kStep;
    constexpr int FM = BM / 32, FN = BN / 32;
    constexpr int kStageBytes = TA::kBytes + TB::kBytes;
    constexpr int kLoads = TA::kInstr + TB::kInstr;
    constexpr int kWaveBytes = ST * kStageBytes;
    static_assert(kWaveBytes >= BM * BN * 4, "a wave's buffers hold its accumulators at the end");
    static_assert(KW * kWaveBytes <= 160 * 1024 && KW * kWaveBytes == flex_lds_bytes<BM, BN, KW, ST>(), "LDS");
    static_assert((ST - 1) * kLoads <= 63, "loads a partial wait can leave outstanding");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    long long batch;
    int tm, tn;
    tile_coords(g, id, groups, batch, tm, tn);
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    const int b = __builtin_amdgcn_readfirstlane((int)batch);
    const int row0 = tm * BM, col0 = tn * BN;
    // slices of K take the place of the batch index
    const bool sliced = SLICES && g.splits > 1;
    const int k_begin = sliced ? b * g.k_slice : 0;
    const int k_rest = (int)g.k - k_begin;
    const int k_end = k_begin + (sliced && g.k_slice < k_rest ? g.k_slice : k_rest);

    // this wave's first K step, and where each operand ends as seen from it
    const int k0 = k_begin + wave * KT;
    const int steps = (k_end - k_begin + KT - 1) / KT;
    const int mine = steps > wave ? (steps - wave + KW - 1) / KW : 0;
    const long long a_at = (sliced ? 0 : b * g.sa) + (A_KSTR ? (long long)k0 * g.lda + row0 : (long long)row0 * g.lda + k0);
    const long long b_at = (sliced ? 0 : b * g.sb) + (B_KSTR ? (long long)k0 * g.ldb + col0 : (long long)col0 * g.ldb + k0);
    const unsigned char* a_src = static_cast<const unsigned char*>(g.a) + kSize * a_at;
    const unsigned char* b_src = static_cast<const unsigned char*>(g.b) + kSize * b_at;
    // rounded up to the 16-byte granule the last element lies in
    constexpr long long kRound = WORDS ? 3 : 15;
    long long a_left = ((A_KSTR ? (long long)(k_end - 1 - k0) * g.lda + g.m - row0
                                : (g.m - 1 - row0) * g.lda + (k_end - k0)) * kSize + kRound) & ~kRound;
    long long b_left = ((B_KSTR ? (long long)(k_end - 1 - k0) * g.ldb + g.n - col0
                                : (g.n - 1 - col0) * g.ldb + (k_end - k0)) * kSize + kRound) & ~kRound;
    const long long a_step = (A_KSTR ? g.lda : 1) * ((long long)kSize * KT * KW);
    const long long b_step = (B_KSTR ? g.ldb : 1) * ((long long)kSize * KT * KW);
    int k_left = k_end - k0;
    const unsigned a_far = (unsigned)(kSize * TA::kFar * g.lda), b_far = (unsigned)(kSize * TB::kFar * g.ldb);
    // (computed ahead of the walk, the sums would take the registers that the held offsets save)
    auto here = [](unsigned v) {
        asm volatile("" : "+s"(v));
        return v;
    };
    unsigned a_off[TA::kHeld], b_off[TB::kHeld];
#pragma unroll
    for (int q = 0; q < TA::kHeld; q++) a_off[q] = TA::source_offset(q, lane, g.lda);
#pragma unroll
    for (int q = 0; q < TB::kHeld; q++) b_off[q] = TB::source_offset(q, lane, g.ldb);
    lds_byte* const mem = (lds_byte*)lds_raw + wave * kWaveBytes;
    const unsigned mem0 = (unsigned)(unsigned long long)mem;

    auto issue = [&](int stage) {
        const buffer_rsrc ra = buffer_from(a_src, a_left), rb = buffer_from(b_src, b_left);
        const unsigned dst = mem0 + (unsigned)stage * kStageBytes;
        // a k-contiguous operand's last step: chunks past K are fetched from past the end of the operand
        const bool tail = k_left < KT;
#pragma unroll
        for (int s = 0; s < TA::kInstr / TA::kHeld; s++) {
            const unsigned far = s == 0 ? 0u : here(s * a_far);
#pragma unroll
            for (int q = 0; q < TA::kHeld; q++)
                TA::load(dst, s * TA::kHeld + q, !A_KSTR && tail && TA::k_of(q, lane) >= k_left ? kPastEnd : a_off[q] + far, ra);
        }
#pragma unroll
        for (int s = 0; s < TB::kInstr / TB::kHeld; s++) {
            const unsigned far = s == 0 ? 0u : here(s * b_far);
#pragma unroll
            for (int q = 0; q < TB::kHeld; q++)
                TB::load(dst + TA::kBytes, s * TB::kHeld + q, !B_KSTR && tail && TB::k_of(q, lane) >= k_left ? kPastEnd : b_off[q] + far, rb);
        }
        a_src += a_step; a_left -= a_step;
        b_src += b_step; b_left -= b_step;
        k_left -= KT * KW;
    };

    f32x16 acc[FM][FN];
    f32x16 low[CT == BR_GEMM_F32 ? FM : 1][CT == BR_GEMM_F32 ? FN : 1];   // fp32: what `acc` is added to at the end

    // The wave's steps; `how`: see FlexWalk
    auto walk = [&](auto how) {
        constexpr int kHow = decltype(how)::value;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    acc[i][j][v] = 0.f;
                    if constexpr (CT == BR_GEMM_F32) low[i][j][v] = 0.f;
                }
        auto fold = [&]() {
            if constexpr (CT == BR_GEMM_F32) {
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
#pragma unroll
                        for (int v = 0; v < 16; v++) low[i][j][v] += acc[i][j][v];
            }
        };
#pragma unroll
        for (int s = 0; s < ST; s++)
            if (s < mine) issue(s);
        int stage = 0;
        for (int t = 0; t < mine; t++) {
            // the loads of step t are in once at most those of the steps after it are outstanding
            const int after = mine - 1 - t;
            if (ST > 1 && after >= ST - 1) wait_vmem<(ST - 1) * kLoads>();
            else if (ST > 2 && after == 1) wait_vmem<kLoads>();
            else wait_vmem<0>();
            const lds_byte* tile = mem + stage * kStageBytes;
            u32x4 fa[4][FM], fb[4][FN];
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
#pragma unroll
                for (int i = 0; i < FM; i++) fa[ks][i] = TA::fragment(tile, TA::frag_offset(i * 32, ks, lane));
#pragma unroll
                for (int j = 0; j < FN; j++) fb[ks][j] = TB::fragment(tile + TA::kBytes, TB::frag_offset(j * 32, ks, lane));
            }
            const bool fresh = (kHow == kOneByOne || kHow == kAsPartsFolded) && (t & 1) == 0;
            if (fresh) fold();   // sums of 64 k-values go to a second set of registers
            // The step is in registers: its buffer takes the loads of step t + ST while the products run.  (In one
            // burst: dealt out between the products they measured 5-15 % slower.)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (t + ST < mine) issue(stage);
            stage = stage + 1 == ST ? 0 : stage + 1;
            // Operands swapped: a lane then holds four consecutive columns of one row of C.
            if constexpr (kHow == kAsParts || kHow == kAsPartsFolded) {
                constexpr bool kApart = kHow == kAsParts;
#pragma unroll
                for (int ks = 0; ks < 4; ks += 2) {
                    u32x4 pa[3][FM];
#pragma unroll
                    for (int i = 0; i < FM; i++) three_parts(fa[ks][i], fa[ks + 1][i], pa[0][i], pa[1][i], pa[2][i]);
                    // (the parts of all of B ahead of the products take more registers than 64 x 64 tiles have)
#pragma unroll
                    for (int j = 0; j < FN; j++) {
                        u32x4 pb[3];
                        three_parts(fb[ks][j], fb[ks + 1][j], pb[0], pb[1], pb[2]);
                        auto products = [&](int p, int q, f32x16 (&to)[FM][FN]) {
#pragma unroll
                            for (int i = 0; i < FM; i++)
                                to[i][j] = Cvt<BR_GEMM_BF16>::mfma(pb[q], pa[p][i], !kApart && fresh && ks + p + q == 0 ? f32x16{} : to[i][j]);
                        };
                        auto small_products = [&](f32x16 (&to)[FM][FN]) {
                            products(0, 1, to);
                            products(1, 0, to);
                            products(1, 1, to);
                            products(0, 2, to);
                            products(2, 0, to);
                        };
                        products(0, 0, acc);
                        if constexpr (!kApart) small_products(acc);
                        else if constexpr (CT == BR_GEMM_F32) small_products(low);
                    }
                }
            } else if constexpr (kHow == kOneByOne) {
                // product s of a sub-step multiplies slot s of both halves of the wave, two k-values; the blocks take
                // turns, so that no product waits for the one before it
#pragma unroll
                for (int ks = 0; ks < 4; ks++)
#pragma unroll
                    for (int s = 0; s < 4; s++)
#pragma unroll
                        for (int i = 0; i < FM; i++)
#pragma unroll
                            for (int j = 0; j < FN; j++)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(fb[ks][j][s]), __uint_as_float(fa[ks][i][s]),
                                                                                 fresh && ks == 0 && s == 0 ? f32x16{} : acc[i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int ks = 0; ks < 4; ks++)
#pragma unroll
                    for (int i = 0; i < FM; i++)
#pragma unroll
                        for (int j = 0; j < FN; j++) acc[i][j] = Cvt<kHow == kInTheirType ? CT : BR_GEMM_BF16>::mfma(fb[ks][j], fa[ks][i], acc[i][j]);
            }
        }
        fold();
    };
    if constexpr (CT == BR_GEMM_F32) {
        const unsigned char* const a_first = a_src;
        const unsigned char* const b_first = b_src;
        const long long a_all = a_left, b_all = b_left;
        const int k_all = k_left;
        if (k_end - k_begin <= kApartUpTo * KW) walk(std::integral_constant<int, kAsParts>{});
        else walk(std::integral_constant<int, kAsPartsFolded>{});
        bool odd = false;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    odd |= __builtin_amdgcn_classf(low[i][j][v], kNotNumbers);
                    low[i][j][v] *= 1.0f / (kPartsScale * kPartsScale);
                }
        if (__any(odd)) {
            a_src = a_first; b_src = b_first;
            a_left = a_all; b_left = b_all;
            k_left = k_all;
            walk(std::integral_constant<int, kOneByOne>{});
        }
    } else {
        walk(std::integral_constant<int, kInTheirType>{});
    }

    if constexpr (CT == BR_GEMM_F32) flex_park<BM, BN>(low, mem, lane);
    else flex_park<BM, BN>(acc, mem, lane);
    __syncthreads();
    flex_emit<BM, BN, KW, KW * 64, TC, GELU>(g, (lds_byte*)lds_raw, kWaveBytes, row0, col0, b);
}

template <int CT, int BM, int BN, int KW, int ST, bool A_KSTR, bool B_KSTR, typename TC, bool GELU = false, bool WORDS = false>
__global__ __launch_bounds__(KW * 64, CT == BR_GEMM_F32 ? 2 : 1) void gemm_flex_kernel(GemmArgs g) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[flex_lds_bytes<BM, BN, KW, ST>()];
    touch_args(g);
    flex_product<CT, BM, BN, KW, ST, A_KSTR, B_KSTR, TC, GELU, WORDS, true>(g, blockIdx.x, gridDim.x, lds);
}

// 64 x 128 tiles, a ring of six K steps, waves that load beside waves that multiply.  The kernel above gives a wave
// whole K steps and buffers of its own; a tile of this size leaves no room for two such buffers a wave.  Here four
// waves share a ring of 24 KB steps: wave w multiplies k-values 16 w .. 16 w + 15 of every step by itself, so a fragment
// is still read from LDS exactly once, and four more waves do nothing but keep five steps of loads in flight.  With the
// same waves doing both, a wave that waits for room in the load path holds up its own products: 52 us instead of 31 for
// the first product below.  One barrier a step.
//
// Why: outputs of some 256 such tiles ([512 x 4096], [1024 x 2048]) are bound by the rate at which a CU fills LDS, about
// 30 B per clock whatever the tile; 64 x 128 tiles ask for three quarters of the bytes of 64 x 64 ones, and 128 x 128
// tiles would leave half of the CUs without one.  Inside model steps, 64 x 64 tiles of two waves / this (us, under the
// profiler): [512 x 4096] K = 4096 50 / 39 and, with the weight the other way round, 40 / 35; [1002 x 2048] K = 2048
// in bf16 35.5 / 27 and 24.8 / 22.7; [1024 x 2048] K = 2048 22 / 19.6.
template <int CT, bool A_KSTR, bool B_KSTR, typename TC, bool GELU = false>
__global__ __launch_bounds__(512) void gemm_ring_kernel(GemmArgs g) {
    constexpr int BM = 64, BN = 128, KW = 4, ST = 6, KT = 64;
    using TA = FlexTile<CT, BM, A_KSTR, false>;
    using TB = FlexTile<CT, BN, B_KSTR, false>;
    constexpr int FM = BM / 32, FN = BN / 32;
    constexpr int kStageBytes = TA::kBytes + TB::kBytes;
    constexpr int kA = TA::kInstr / KW, kB = TB::kInstr / KW, kLoads = kA + kB;   // a wave's share of a step's loads
    static_assert(TA::kStep == KT && TA::kInstr % KW == 0 && TB::kInstr % KW == 0, "16-bit operands");
    static_assert(ST * kStageBytes >= KW * BM * BN * 4 && ST * kStageBytes <= 160 * 1024, "LDS");
    static_assert((ST - 1) * kLoads <= 63, "loads a partial wait can leave outstanding");
    __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[ST * kStageBytes];
    const int lane = threadIdx.x & 63;
    const bool loader = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= KW;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % KW;   // among the loaders / the multipliers
    long long batch;
    int tm, tn;
    tile_coords(g, batch, tm, tn);
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    const int b = __builtin_amdgcn_readfirstlane((int)batch);
    const int row0 = tm * BM, col0 = tn * BN;
    // slices of K take the place of the batch index
    const bool sliced = g.splits > 1;
    const int k_begin = sliced ? b * g.k_slice : 0;
    const int k_rest = (int)g.k - k_begin;
    const int k_end = k_begin + (sliced && g.k_slice < k_rest ? g.k_slice : k_rest);
    const int steps = (k_end - k_begin + KT - 1) / KT;
    const int padded = steps + (steps & 1);   // the multipliers take steps in pairs
    // step t of the loop covers K step (t + first) mod steps of the slice (see k_walk_start)
    const int start = (int)(k_walk_start(row0, col0, g.k) / KT), first = start < steps ? start : start % steps;
    const int k0 = k_begin + first * KT;
    const long long a_at = (sliced ? 0 : b * g.sa) + (A_KSTR ? (long long)k0 * g.lda + row0 : (long long)row0 * g.lda + k0);
    const long long b_at = (sliced ? 0 : b * g.sb) + (B_KSTR ? (long long)k0 * g.ldb + col0 : (long long)col0 * g.ldb + k0);
    const unsigned char* a_src = static_cast<const unsigned char*>(g.a) + 2 * a_at;
    const unsigned char* b_src = static_cast<const unsigned char*>(g.b) + 2 * b_at;
    // where each operand ends as seen from the current step, rounded up to the granule the last element lies in
    long long a_left = ((A_KSTR ? (long long)(k_end - 1 - k0) * g.lda + g.m - row0
                                : (g.m - 1 - row0) * g.lda + (k_end - k0)) * 2 + 15) & ~15LL;
    long long b_left = ((B_KSTR ? (long long)(k_end - 1 - k0) * g.ldb + g.n - col0
                                : (g.n - 1 - col0) * g.ldb + (k_end - k0)) * 2 + 15) & ~15LL;
    const long long a_step = (A_KSTR ? g.lda : 1) * (2LL * KT);
    const long long b_step = (B_KSTR ? g.ldb : 1) * (2LL * KT);
    int k_left = k_end - k0;
    int until_wrap = steps - first;
    unsigned a_off[kA], b_off[kB];
#pragma unroll
    for (int q = 0; q < kA; q++) a_off[q] = TA::source_offset(wave * kA + q, lane, g.lda);
#pragma unroll
    for (int q = 0; q < kB; q++) b_off[q] = TB::source_offset(wave * kB + q, lane, g.ldb);
    lds_byte* const lds = (lds_byte*)lds_raw;
    const unsigned lds0 = (unsigned)(unsigned long long)lds;

    auto issue = [&](int stage, int t) {
        // an odd number of steps is filled up with one of zeros, loaded from past the end
        const buffer_rsrc ra = buffer_from(a_src, t < steps ? a_left : 0), rb = buffer_from(b_src, t < steps ? b_left : 0);
        const unsigned dst = lds0 + (unsigned)stage * kStageBytes;
        // a k-contiguous operand's last step: chunks past K are fetched from past the end of the operand
        const bool tail = k_left < KT;
#pragma unroll
        for (int q = 0; q < kA; q++)
            TA::load(dst, wave * kA + q, !A_KSTR && tail && TA::k_of(wave * kA + q, lane) >= k_left ? kPastEnd : a_off[q], ra);
#pragma unroll
        for (int q = 0; q < kB; q++)
            TB::load(dst + TA::kBytes, wave * kB + q, !B_KSTR && tail && TB::k_of(wave * kB + q, lane) >= k_left ? kPastEnd : b_off[q], rb);
        const bool wraps = --until_wrap == 0;
        const long long da = wraps ? a_step - steps * a_step : a_step, db = wraps ? b_step - steps * b_step : b_step;
        a_src += da; a_left -= da;
        b_src += db; b_left -= db;
        k_left -= wraps ? KT - steps * KT : KT;
    };

    // Barrier t, t = 0 .. padded - 1: step t is in LDS, and the fragments of step t - 1 are in registers.
    if (loader) {
#pragma unroll
        for (int s = 0; s < ST; s++)
            if (s < padded) issue(s, s);
        if (padded >= ST) wait_vmem<(ST - 1) * kLoads>();
        else wait_vmem<0>();
        __builtin_amdgcn_s_barrier();
        int stage = 0;
        for (int t = 1; t < padded; t++) {
            // step t is in once at most the ST - 2 steps after it are outstanding
            if (t + ST <= padded + 1) wait_vmem<(ST - 2) * kLoads>();
            else wait_vmem<0>();
            __builtin_amdgcn_s_barrier();
            if (t - 1 + ST < padded) issue(stage, t - 1 + ST);   // where step t - 1 was
            stage = stage + 1 == ST ? 0 : stage + 1;
        }
        __builtin_amdgcn_s_barrier();
    } else {
        unsigned fa_off[FM], fb_off[FN];
#pragma unroll
        for (int i = 0; i < FM; i++) fa_off[i] = TA::frag_offset(i * 32, wave, lane);
#pragma unroll
        for (int j = 0; j < FN; j++) fb_off[j] = TA::kBytes + TB::frag_offset(j * 32, wave, lane);
        f32x16 acc[FM][FN];
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
        u32x4 fa0[FM], fb0[FN], fa1[FM], fb1[FN];
        int stage = 0;
        auto read = [&](u32x4 (&fa)[FM], u32x4 (&fb)[FN]) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const lds_byte* tile = lds + stage * kStageBytes;
#pragma unroll
            for (int i = 0; i < FM; i++) fa[i] = TA::fragment(tile, fa_off[i]);
#pragma unroll
            for (int j = 0; j < FN; j++) fb[j] = TB::fragment(tile, fb_off[j]);
            stage = stage + 1 == ST ? 0 : stage + 1;
            __builtin_amdgcn_sched_barrier(0);
        };
        auto multiply = [&](const u32x4 (&fa)[FM], const u32x4 (&fb)[FN]) {
            // operands swapped: a lane then holds four consecutive columns of one row of C
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) acc[i][j] = Cvt<CT>::mfma(fb[j], fa[i], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        };
        read(fa0, fb0);
        for (int t = 2; t < padded; t += 2) {
            read(fa1, fb1);
            multiply(fa0, fb0);
            read(fa0, fb0);
            multiply(fa1, fb1);
        }
        read(fa1, fb1);
        multiply(fa0, fb0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        multiply(fa1, fb1);
        // every load has landed and every fragment has been read once all waves are here
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        flex_park<BM, BN>(acc, lds + wave * (BM * BN * 4), lane);
    }
    __syncthreads();
    flex_emit<BM, BN, KW, 512, TC, GELU>(g, lds, BM * BN * 4, row0, col0, b);
}

// ---- host-side dispatch -------------------------------------------------------
template <int CT, int BM, int BN, int KW, int ST, typename TC>
int launch_flex_c(const GemmArgs& g, const Problem& p, unsigned grid, hipStream_t st) {
    if (g.c2) {
        // as the large kernels': the linear layer's layout with 16-bit outputs
        if constexpr (sizeof(TC) == 2) {
            if (p.a_kstr || p.b_kstr) return BR_ERR_TODO;
            gemm_flex_kernel<CT, BM, BN, KW, ST, false, false, TC, true><<<grid, KW * 64, 0, st>>>(g);
        } else {
            return BR_ERR_TODO;
        }
    } else if (p.a_kstr && p.b_kstr) {
        gemm_flex_kernel<CT, BM, BN, KW, ST, true, true, TC><<<grid, KW * 64, 0, st>>>(g);
    } else if (p.a_kstr) {
        gemm_flex_kernel<CT, BM, BN, KW, ST, true, false, TC><<<grid, KW * 64, 0, st>>>(g);
    } else if (p.b_kstr) {
        gemm_flex_kernel<CT, BM, BN, KW, ST, false, true, TC><<<grid, KW * 64, 0, st>>>(g);
    } else {
        gemm_flex_kernel<CT, BM, BN, KW, ST, false, false, TC><<<grid, KW * 64, 0, st>>>(g);
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

template <int CT, typename TC>
int launch_ring_c(const GemmArgs& g, const Problem& p, unsigned grid, hipStream_t st) {
    if (g.c2) {
        if constexpr (sizeof(TC) == 2) {
            if (p.a_kstr || p.b_kstr) return BR_ERR_TODO;
            gemm_ring_kernel<CT, false, false, TC, true><<<grid, 512, 0, st>>>(g);
        } else {
            return BR_ERR_TODO;
        }
    } else if (p.a_kstr && p.b_kstr) {
        gemm_ring_kernel<CT, true, true, TC><<<grid, 512, 0, st>>>(g);
    } else if (p.a_kstr) {
        gemm_ring_kernel<CT, true, false, TC><<<grid, 512, 0, st>>>(g);
    } else if (p.b_kstr) {
        gemm_ring_kernel<CT, false, true, TC><<<grid, 512, 0, st>>>(g);
    } else {
        gemm_ring_kernel<CT, false, false, TC><<<grid, 512, 0, st>>>(g);
    }
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// The tiling of a product and whether four columns of C can be stored at once; the number of workgroups, or -1.
template <int BM, int BN>
long long flex_tiles(GemmArgs& g, const Problem& p, long long batch) {
    g.tiles_m = (int)((g.m + BM - 1) / BM);
    g.tiles_n = (int)((g.n + BN - 1) / BN);
    const long long blocks = (long long)g.tiles_m * g.tiles_n * (g.splits > 1 ? g.splits : batch);
    const long long es = p.c_dtype == BR_F32 ? 4 : 2;
    auto quads = [&](const void* q) { return (reinterpret_cast<uintptr_t>(q) & (4 * es - 1)) == 0; };
    g.vec_c = g.ldc % 4 == 0 && g.sc % 4 == 0 && quads(g.c) && (!g.c2 || quads(g.c2)) && (!g.sum || (quads(g.sum) && quads(g.addend)));
    return blocks > 0x7fffffffLL ? -1 : blocks;
}

template <int CT, int BM, int BN, int KW, int ST>
int launch_flex_config(GemmArgs g, const Problem& p, long long batch, hipStream_t st) {
    const long long blocks = flex_tiles<BM, BN>(g, p, batch);
    if (blocks < 0) return BR_ERR_ATTR;
    if (p.c_dtype == BR_F32) return launch_flex_c<CT, BM, BN, KW, ST, float>(g, p, (unsigned)blocks, st);
    return launch_flex_c<CT, BM, BN, KW, ST, std::conditional_t<CT == BR_GEMM_F16, __half, __hip_bfloat16>>(g, p, (unsigned)blocks, st);
}

template <int CT>
int launch_ring(GemmArgs g, const Problem& p, long long batch, hipStream_t st) {
    const long long blocks = flex_tiles<64, 128>(g, p, batch);
    if (blocks < 0) return BR_ERR_ATTR;
    if (p.c_dtype == BR_F32) return launch_ring_c<CT, float>(g, p, (unsigned)blocks, st);
    return launch_ring_c<CT, std::conditional_t<CT == BR_GEMM_F16, __half, __hip_bfloat16>>(g, p, (unsigned)blocks, st);
}

// Any K; slices of K as batch entries when g.splits > 1.
template <int CT>
int launch_flex(const GemmArgs& g, const Problem& p, int kernel, long long batch, hipStream_t st) {
    if (kernel == kFlex64) return launch_flex_config<CT, 64, 64, 4, 1>(g, p, batch, st);
    if (kernel == kFlex64Short) return launch_flex_config<CT, 64, 64, 2, 1>(g, p, batch, st);
    if (kernel == kFlex32x64) return launch_flex_config<CT, 32, 64, 4, 1>(g, p, batch, st);
    if (kernel == kRing64x128) return launch_ring<CT>(g, p, batch, st);
    return launch_flex_config<CT, 32, 32, 4, 2>(g, p, batch, st);
}

// fp32 operands and C.  `words`: an operand's rows are not aligned to 16 bytes (or a k-contiguous one's do not end on
// such a boundary), so it is loaded value by value.
template <int BM, int BN, int KW, bool WORDS>
int launch_flex_fp32(GemmArgs g, const Problem& p, long long batch, hipStream_t st) {
    g.tiles_m = (int)((g.m + BM - 1) / BM);
    g.tiles_n = (int)((g.n + BN - 1) / BN);
    const long long blocks = (long long)g.tiles_m * g.tiles_n * batch;
    if (blocks > 0x7fffffffLL) return BR_ERR_ATTR;
    const unsigned grid = (unsigned)blocks;
    g.vec_c = g.ldc % 4 == 0 && g.sc % 4 == 0 && aligned16(g.c) && (!g.sum || (aligned16(g.sum) && aligned16(g.addend)));
    if (p.a_kstr && p.b_kstr)
        gemm_flex_kernel<BR_GEMM_F32, BM, BN, KW, 1, true, true, float, false, WORDS><<<grid, KW * 64, 0, st>>>(g);
    else if (p.a_kstr)
        gemm_flex_kernel<BR_GEMM_F32, BM, BN, KW, 1, true, false, float, false, WORDS><<<grid, KW * 64, 0, st>>>(g);
    else if (p.b_kstr)
        gemm_flex_kernel<BR_GEMM_F32, BM, BN, KW, 1, false, true, float, false, WORDS><<<grid, KW * 64, 0, st>>>(g);
    else
        gemm_flex_kernel<BR_GEMM_F32, BM, BN, KW, 1, false, false, float, false, WORDS><<<grid, KW * 64, 0, st>>>(g);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

}  // namespace gemm16
}  // namespace brk
