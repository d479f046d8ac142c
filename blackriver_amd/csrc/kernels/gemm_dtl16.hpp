// 16-bit MFMA GEMM, direct-to-LDS variant: the fast path for products whose
// two operands are both stored in the MFMA element type (fp16 or bf16).
//
//   C[b][i,j] = alpha * sum_p opA[b][i,p] * opB[b][p,j] (+ C) (+ bias[j])
//
// Operand tiles never pass through registers on their way in: every wave
// issues global_load_lds_dwordx4 (gfx950: 16 bytes per lane, 1 KiB per
// instruction, written to LDS at M0 + lane*16).  Because the LDS side of such
// a load is fixed to lane order, padding rows is not possible; bank conflicts
// are avoided by choosing WHICH 16-byte chunk of the tile each lane fetches
// (an XOR swizzle), and un-swizzling in the fragment reads:
//
//   k contiguous in memory  -> LDS image [row][4 chunks of 8 k], 64 bytes per
//       row; chunk c of row r sits in slot c ^ ((r >> 2) & 3).  A fragment is
//       one ds_read_b128 per lane; any 16 consecutive rows of one chunk column
//       cover all 64 banks exactly once.
//   row contiguous in memory-> LDS image [k][ROWS/8 chunks of 8 rows]; chunk c
//       of k-row k sits in slot c ^ (4 * (k & 3)).  Fragments are read with
//       ds_read_b64_tr_b16 (two per fragment); the 4 k-rows x 64 bytes that 32
//       lanes touch in one pass land in 16 different 16-byte bank groups.
//
// Pipeline.  STAGES tile buffers form a ring and are all filled up front.  A K
// step (KT = 32 or 64 k-values) is KT/16 sub-steps with two fragment register
// sets used alternately:
//   sub-step s < last:  issue the LDS reads of sub-step s+1, run the MFMAs of
//       sub-step s (whose fragments were read one sub-step ago);
//   last sub-step of tile t:  wait until this wave's loads of tile t+1 have
//       landed (s_waitcnt vmcnt(N), later tiles stay in flight); workgroup
//       barrier -- now tile t+1 is complete in LDS and every wave has read all
//       of tile t; issue the loads of tile t+STAGES into the buffer tile t
//       occupied; issue the LDS reads of (t+1, first sub-step); run the MFMAs.
// KT = 64 makes a k-contiguous operand row a full 128-byte cache line per
// step (with 32, each line is fetched from L2 twice, half used each time).
// One barrier per K step, no staging registers, LDS latency hidden behind 16+
// MFMAs inside the wave, HBM / L2 latency behind STAGES-1 K steps.  The loads
// and the vmcnt waits are inline assembly because the compiler would otherwise
// wait for ALL outstanding direct-to-LDS loads before any LDS read.
//
// Requirements (dtl_applies; everything else takes the register-staged kernel in
// gemm_mfma16.hpp): 16-byte aligned operand bases / leading dimensions / batch
// strides and, for k-contiguous operands, K % 8 == 0 (or rows zero-filled up to
// that).  K that is not a multiple of 64 takes the ragged form (RAG: loads
// through buffer resources with hardware bounds checks).  Measured on bf16
// weight gradients of 1002 tokens, which ran on the register-staged kernel's
// element-wise guarded form before: [8192 x 2048] 355 -> 43 us, [6144 x 2048]
// 194 -> 37 us.  Rows past the end of an operand are redirected to a valid row;
// their products land in rows / columns of C that are never stored.
#pragma once
#include <mutex>
#include <type_traits>

#include "gemm_mfma16.hpp"
#include "gemm_plan.hpp"
#include "lds_direct.hpp"


namespace brk {
namespace gemm16 {

// Operand tile of ROWS x KT elements (KT = 32 or 64 k-values per K step).
template <int ROWS, int KT, int WAVES, bool KSTR>
struct DtlTile {
    static constexpr int kBytes = ROWS * KT * 2;
    static constexpr int kInstr = kBytes / 1024;     // wave-wide loads per tile
    static constexpr int kPerWave = kInstr / WAVES;  // ... issued by each wave
    static_assert(kInstr % WAVES == 0, "tile loads do not divide among the waves");
    static_assert(ROWS >= 128, "swizzle needs at least 16 chunks per k-row");
    // k contiguous: a row is KT/8 chunks; kRowsPer256 rows span the 64 banks
    static constexpr int kRowBytes = KT * 2;
    static constexpr int kChunksPerRow = KT / 8;
    static constexpr int kRowsPer256 = 256 / kRowBytes;
    static constexpr int kRowsPerInstr = 64 / kChunksPerRow;
    // row contiguous: a k-row is ROWS/8 chunks
    static constexpr int kChunksPerK = ROWS / 8;
    static constexpr int kKPerInstr = 64 / kChunksPerK;

    // Byte offset (from the tile origin at K step 0) of the chunk this lane
    // fetches in its q-th load of a tile; LDS slot = instruction*64 + lane.
    static __device__ __forceinline__ unsigned source_offset(int q, int wave, int lane, long long ld, long long row0,
                                                             long long rows) {
        const int j = q * WAVES + wave;
        if (!KSTR) {
            const int r = j * kRowsPerInstr + lane / kChunksPerRow;
            const int c = (lane % kChunksPerRow) ^ ((r / kRowsPer256) % kChunksPerRow);
            long long row = row0 + r;
            row = row < rows ? row : rows - 1;
            return (unsigned)(((row - row0) * ld + c * 8) * 2);
        } else {
            const int kk = j * kKPerInstr + lane / kChunksPerK;
            const int c = (lane % kChunksPerK) ^ (4 * (kk & 3));
            long long row = row0 + c * 8;
            row = row < rows ? row : row0;
            return (unsigned)((kk * ld + (row - row0)) * 2);
        }
    }

    // k (relative to the step) of the first element of the chunk this lane fetches in its q-th load
    static __device__ __forceinline__ int k_of(int q, int wave, int lane) {
        const int j = q * WAVES + wave;
        if (KSTR) return j * kKPerInstr + lane / kChunksPerK;
        return ((lane % kChunksPerRow) ^ ((j * kRowsPerInstr + lane / kChunksPerRow) / kRowsPer256 % kChunksPerRow)) * 8;
    }

    // LDS byte offset (inside one tile image) this lane reads the fragment of
    // 32-row block `row_base` and 16-k sub-step ks from; row-contiguous tiles
    // read a second time 4 k-rows further on.
    static __device__ __forceinline__ unsigned frag_offset(int row_base, int ks, int lane) {
        if (!KSTR) {
            const int r = row_base + (lane & 31);
            const int c = ks * 2 + (lane >> 5);
            return (unsigned)(r * kRowBytes + ((c ^ ((r / kRowsPer256) % kChunksPerRow)) * 16));
        } else {
            const int i = lane & 15, grp = lane >> 4;
            const int kk = ks * 16 + (grp >> 1) * 8 + (i >> 2);
            const int row16 = row_base + (grp & 1) * 16 + (i & 3) * 4;
            const int c = (row16 >> 3) ^ (4 * (i >> 2));
            return (unsigned)(kk * (ROWS * 2) + c * 16 + (row16 & 7) * 2);
        }
    }

    static __device__ __forceinline__ u32x4 fragment(const lds_byte* tile, unsigned off) {
        if (!KSTR) {
            return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(tile + off);
        } else {
            typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off + 4 * ROWS * 2));
            const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
            return mk4(l2.x, l2.y, h2.x, h2.y);
        }
    }
};

// K split in two with the sum done in the kernel.  A product whose 256x256 tiles fill at most half the CUs and
// whose K is long runs two workgroups per tile, workgroup (tile, s) summing half s of K.  After its K loop a
// workgroup draws a ticket from the tile's counter.  The first to draw writes its fp32 partial tile to the caller's
// workspace (in the accumulators' own register order), reports in on a second counter and is done; the second
// waits until the first has reported -- it drew first, so it is past its K loop and its stores are in flight: a
// wait for work already under way, never for a workgroup that may not have started -- adds that partial to its own
// and runs the epilogue.  A sum of two terms is the same whichever is added to which, so the bits do not depend on
// which half finished first.
// The partial tile crosses from one XCD's L2 to another's.  Every access to it is made coherent at device scope by
// itself (the sc1 bit: the access goes to the level all XCDs share), so no fence has to write back or invalidate
// a whole L2 -- which a device-scope fence does on this part, and which costs more than the product when hundreds
// of workgroups do it.  Such accesses move 1.5-3 TB/s where ordinary stores move 6-7: with four or more slices
// (every slice writing, one reading them all) this form measured slower than partials written with ordinary
// stores and summed by a second kernel, which is what products with more slices use (gemm.hip).
// The counters live in the library, start at zero and are put back to zero by the second arrival, so a launch needs
// no clearing pass.  There is one set per stream (kSplitSlots of them, handed out in the order streams first ask:
// split_slot_of): products on one stream run one after the other and may share a set, products split at the same
// time on different streams meet through different sets; a stream beyond the last set gets no split.
constexpr int kSplitSlots = 8;
static __device__ unsigned dtl_tickets[kSplitSlots][kMaxSplitTiles];
static __device__ unsigned dtl_arrived[kSplitSlots][kMaxSplitTiles];

typedef float f32x4 __attribute__((ext_vector_type(4)));
// The wait states after the store are part of the statement: a store of more than 64 bits reads its data
// registers a few cycles after it issues, and the compiler, which keeps such a store's data registers intact for
// that long when it emits the instruction itself, does not look into an asm statement -- it reused them for the
// next address at once, and single lanes of a partial tile came out as garbage.
__device__ __forceinline__ void store_device_coherent(f32x4* p, const f32x4& v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 2" : : "v"(p), "v"(v) : "memory");
}
// Four such loads and the wait for them in ONE statement: the compiler takes an asm statement's outputs to be
// ready when the statement ends, so a wait in a statement of its own would let it copy the registers in between.
__device__ __forceinline__ void load4_device_coherent(f32x4 (&v)[4], const f32x4* p, int stride) {
    const f32x4 *p1 = p + stride, *p2 = p + 2 * stride, *p3 = p + 3 * stride;
    asm volatile(
        "global_load_dwordx4 %0, %4, off sc1\n\t"
        "global_load_dwordx4 %1, %5, off sc1\n\t"
        "global_load_dwordx4 %2, %6, off sc1\n\t"
        "global_load_dwordx4 %3, %7, off sc1\n\t"
        "s_waitcnt vmcnt(0)"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
        : "v"(p), "v"(p1), "v"(p2), "v"(p3)
        : "memory");
}

// One element of C through a buffer resource.
template <typename T>
__device__ __forceinline__ float buffer_read(__amdgpu_buffer_rsrc_t r, unsigned at) {
    if constexpr (sizeof(T) == 4) {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0));
    } else {
        const T h = __builtin_bit_cast(T, (u16)__builtin_amdgcn_raw_buffer_load_b16(r, at, 0, 0));
        return c_load<T>(&h);
    }
}
template <typename T>
__device__ __forceinline__ void buffer_write(__amdgpu_buffer_rsrc_t r, unsigned at, float v) {
    if constexpr (sizeof(T) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, at, 0, 0);
    } else {
        T h;
        c_store<T>(&h, v);
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(u16, h), r, at, 0, 0);
    }
}

// Tiles of which a CU runs two at a time, each with 32-wide K steps: while one workgroup stores its tile the other
// multiplies (see shared_applies).
constexpr bool shared_tile(int bm, int bn, int kt) { return bm * bn == 128 * 256 && kt == 32; }

// KW = 2: the sixteen-wide sub-steps of every K step are dealt to two groups of waves (group kw takes sub-steps
// kw * KS/2 ..), each group covering the whole tile with wave tiles twice as large; the groups' accumulators are
// added through LDS after the K loop (group 1 into group 0, which runs the epilogue).  For tiles too small to give
// eight waves a 64 x 128 block each: a 256 x 128 tile on eight 64 x 64 waves reads 128 KB of fragments per K step
// from LDS, on two groups of four 64 x 128 waves 96 KB.
template <int CT, int BM, int BN, int WM, int WN, int KT, int STAGES, bool A_KSTR, bool B_KSTR, typename TC,
          bool GELU = false, bool SPLIT = false, int KW = 1, bool RAG = false>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * KW * 64, (shared_tile(BM, BN, KT) ? 2 : 1)) void gemm_dtl_kernel(GemmArgs g) {
    constexpr int WAVES_MN = (BM / WM) * (BN / WN);
    constexpr int WAVES = WAVES_MN * KW;
    constexpr int FM = WM / 32, FN = WN / 32, KS = KT / 16 / KW;   // KS: sub-steps of a K step per wave
    static_assert(KW == 1 || (KW == 2 && KT == 64 && !SPLIT), "two wave groups: 64-wide K steps, no K split across workgroups");
    using TA = DtlTile<BM, KT, WAVES, A_KSTR>;
    using TB = DtlTile<BN, KT, WAVES, B_KSTR>;
    constexpr int kStageBytes = TA::kBytes + TB::kBytes;
    constexpr int kLoads = TA::kPerWave + TB::kPerWave;  // per wave and tile
    static_assert(STAGES >= 2 && STAGES <= 6, "two to six tile buffers");
    static_assert(KT == 32 || KT == 64, "K tile of 32 or 64");
    static_assert(FM * FN >= FM + FN, "one LDS fragment read per MFMA slot");
    static_assert(STAGES * kStageBytes <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[STAGES * kStageBytes];
    const lds_byte* lds = (const lds_byte*)lds_raw;
    const unsigned lds0 = (unsigned)(unsigned long long)lds;

    // two groups of waves lose by it: [2048 x 4096] from K = 4096 80.5 us with, 79.3 without, a 16-bit C 73.0 and 72.1
    if constexpr (KW == 1) touch_args(g);
    long long batch;
    int tm, tn;
    tile_coords(g, batch, tm, tn);
    // The divisions in tile_coords run on the vector unit although their operands are wave-uniform.  Taking the
    // results back to scalar registers here keeps everything derived from them (operand tile origins, which the
    // load statement needs in scalar registers, and the row bases of C) on the scalar unit.
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    batch = __builtin_amdgcn_readfirstlane((int)batch);
    // with a K split the slices take the place of the batch index in the tile order (slice-major: the workgroups
    // an XCD runs at a time still cover one block of tiles, of one slice)
    const int slice = SPLIT || (RAG && g.splits > 1) ? (int)batch : 0;
    const long long operand_batch = SPLIT || (RAG && g.splits > 1) ? 0 : batch;
    if (SPLIT) batch = 0;
    const long long row0 = (long long)tm * BM, col0 = (long long)tn * BN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kw = KW == 1 ? 0 : wave / WAVES_MN, wave_mn = KW == 1 ? wave : wave % WAVES_MN;
    const int wm = wave_mn / (BN / WN), wn = wave_mn % (BN / WN);

    // tile origins at K step 0 (wave-uniform, advanced once per step) and the
    // per-lane chunk offsets (fixed for the whole K loop)
    const unsigned char* a_src = reinterpret_cast<const unsigned char*>(g.a) +
                                 2 * (operand_batch * g.sa + (A_KSTR ? row0 : row0 * g.lda));
    const unsigned char* b_src = reinterpret_cast<const unsigned char*>(g.b) +
                                 2 * (operand_batch * g.sb + (B_KSTR ? col0 : col0 * g.ldb));
    const long long a_step = A_KSTR ? 2 * KT * g.lda : 2 * KT;
    const long long b_step = B_KSTR ? 2 * KT * g.ldb : 2 * KT;
    unsigned a_off[TA::kPerWave], b_off[TB::kPerWave];
#pragma unroll
    for (int q = 0; q < TA::kPerWave; q++) a_off[q] = TA::source_offset(q, wave, lane, g.lda, row0, g.m);
#pragma unroll
    for (int q = 0; q < TB::kPerWave; q++) b_off[q] = TB::source_offset(q, wave, lane, g.ldb, col0, g.n);

    unsigned fa_off[FM][KS], fb_off[FN][KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
#pragma unroll
        for (int i = 0; i < FM; i++) fa_off[i][ks] = TA::frag_offset(wm * WM + i * 32, kw * KS + ks, lane);
#pragma unroll
        for (int j = 0; j < FN; j++) fb_off[j][ks] = TA::kBytes + TB::frag_offset(wn * WN + j * 32, kw * KS + ks, lane);
    }

    // this workgroup's K steps: [k_begin, k_begin + nk) of the g.k / KT steps (all of them without a split)
    const int nk_all = (int)((g.k + KT - 1) / KT);
    const int rag_begin = RAG ? slice * (g.k_slice / KT) : 0;
    const int k_begin = SPLIT ? slice * nk_all / 2 : rag_begin;
    const int nk = SPLIT ? (slice + 1) * nk_all / 2 - k_begin
                   : RAG && g.splits > 1 && k_begin + g.k_slice / KT < nk_all ? g.k_slice / KT : nk_all - k_begin;
    // step `t` of the loop covers K step k_begin + (t + first) mod nk (see k_walk_start)
    const int start = (int)(k_walk_start(row0, col0, g.k) / KT), first = (SPLIT || RAG) && start >= nk ? start % nk : start;
    a_src += (k_begin + first) * a_step;
    b_src += (k_begin + first) * b_step;
    int until_wrap = nk - first;  // issues left before the walk returns to K step 0
    // RAG: K is not a multiple of KT.  The loads go through buffer resources that end where the operands end, so
    // that k-rows past K of a row-contiguous operand read as zero; chunks past K of a k-contiguous one (K a multiple
    // of 8, or rows zero-filled up to one) are fetched from past the end.  k_left: k-values from the current step on.
    int k_left = RAG ? (int)g.k - (k_begin + first) * KT : 0;
    auto issue = [&](int tile) {
        const unsigned dst = lds0 + (unsigned)(tile % STAGES) * kStageBytes + (unsigned)wave * 1024u;
        if constexpr (RAG) {
            const buffer_rsrc ra = buffer_from(a_src, (((A_KSTR ? (k_left - 1) * g.lda + g.m - row0 : (g.m - 1 - row0) * g.lda + k_left) * 2 + 15) & ~15LL));
            const buffer_rsrc rb = buffer_from(b_src, (((B_KSTR ? (k_left - 1) * g.ldb + g.n - col0 : (g.n - 1 - col0) * g.ldb + k_left) * 2 + 15) & ~15LL));
#pragma unroll
            for (int q = 0; q < TA::kPerWave; q++)
                buffer_dtl_load(dst + q * WAVES * 1024, !A_KSTR && TA::k_of(q, wave, lane) >= k_left ? kPastEnd : a_off[q], ra);
#pragma unroll
            for (int q = 0; q < TB::kPerWave; q++)
                buffer_dtl_load(dst + TA::kBytes + q * WAVES * 1024, !B_KSTR && TB::k_of(q, wave, lane) >= k_left ? kPastEnd : b_off[q], rb);
        } else {
#pragma unroll
            for (int q = 0; q < TA::kPerWave; q++) dtl_load(dst + q * WAVES * 1024, a_off[q], a_src);
#pragma unroll
            for (int q = 0; q < TB::kPerWave; q++) dtl_load(dst + TA::kBytes + q * WAVES * 1024, b_off[q], b_src);
        }
        const bool wraps = --until_wrap == 0;
        a_src += wraps ? a_step - nk * a_step : a_step;
        b_src += wraps ? b_step - nk * b_step : b_step;
        if (RAG) k_left += wraps ? (nk - 1) * KT : -KT;
    };
    auto read_frags = [&](u32x4 (&fa)[FM], u32x4 (&fb)[FN], int tile, int ks) {
        const lds_byte* stage = lds + (tile % STAGES) * kStageBytes;
#pragma unroll
        for (int i = 0; i < FM; i++) fa[i] = TA::fragment(stage, fa_off[i][ks]);
#pragma unroll
        for (int j = 0; j < FN; j++) fb[j] = TB::fragment(stage, fb_off[j][ks]);
    };

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
    // One sub-step, in the instruction order the hardware is to see: the MFMAs of
    // the fragments in hand (fa, fb), with the LDS reads that fetch the next
    // sub-step's fragments (na, nb; from `tile`, sub-step `ks`) slotted in one
    // per MFMA.  The scheduling fences pin that order: left alone, the compiler
    // sinks the reads below the MFMAs to reuse their registers, and the next
    // sub-step's first MFMA then waits out the full LDS latency.
    auto step = [&](const u32x4 (&fa)[FM], const u32x4 (&fb)[FN], u32x4 (&na)[FM], u32x4 (&nb)[FN], int tile, int ks) {
        const lds_byte* stage = lds + (tile % STAGES) * kStageBytes;
#pragma unroll
        for (int idx = 0; idx < FM * FN; idx++) {
            // column-major walk over the wave's blocks: the first FM MFMAs need only fb[0];
            // fragments are fetched in the order the next sub-step uses them: fb[0], fa[0..], fb[1..]
            const int i = idx % FM, j = idx / FM;
            if (idx == 0) nb[0] = TB::fragment(stage, fb_off[0][ks]);
            else if (idx <= FM) na[idx - 1] = TA::fragment(stage, fa_off[idx - 1][ks]);
            else if (idx < FM + FN) nb[idx - FM] = TB::fragment(stage, fb_off[idx - FM][ks]);
            acc[i][j] = Cvt<CT>::mfma(fa[i], fb[j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Fill the ring, wait for tile 0 and read its first sub-step of fragments.
#pragma unroll
    for (int s = 0; s < STAGES; s++)
        if (s < nk) issue(s);
    if (nk > STAGES - 1) {
        wait_vmem<(STAGES - 1) * kLoads>();
    } else {
        wait_vmem<0>();
    }
    __syncthreads();
    // Two fragment sets: while the MFMAs of one sub-step run, the LDS reads of
    // the next sub-step are in flight.
    u32x4 fa0[FM], fb0[FN], fa1[FM], fb1[FN];
    read_frags(fa0, fb0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);

    // The MFMA stream is free of branches: the last tile's final sub-step also
    // fetches (from the buffer a tile nk would occupy; the values are never
    // used) and passes the barrier like every other.
    for (int t = 0; t < nk; t++) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            u32x4(&fa_now)[FM] = (ks & 1) ? fa1 : fa0;
            u32x4(&fb_now)[FN] = (ks & 1) ? fb1 : fb0;
            u32x4(&fa_next)[FM] = (ks & 1) ? fa0 : fa1;
            u32x4(&fb_next)[FN] = (ks & 1) ? fb0 : fb1;
            if (ks + 1 < KS) {
                step(fa_now, fb_now, fa_next, fb_next, t, ks + 1);
            } else {
                // tile t+1 has to be in LDS; the tiles issued after it may stay in flight
                const int after = nk - 2 - t;
                if (after >= STAGES - 2) {
                    wait_vmem<(STAGES - 2) * kLoads>();
                } else if (STAGES > 3 && after == 1) {
                    wait_vmem<kLoads>();
                } else {
                    wait_vmem<0>();
                }
                // every wave has now read all of tile t (__syncthreads waits for the wave's own LDS reads to
                // complete, lgkmcnt(0), before the barrier), so its buffer can be refilled
                __syncthreads();
                if (t + STAGES < nk) issue(t + STAGES);
                __builtin_amdgcn_sched_barrier(0);
                step(fa_now, fb_now, fa_next, fb_next, t + 1, 0);
            }
        }
    }

    if constexpr (KW == 2) {
        // Every tile issued has landed and been read (the loop's last waits and barrier); the stages now carry
        // group 1's accumulators to group 0: quad q of thread t of wave w at quad index (w * 4 FM FN + q) * 64 + t.
        static_assert((size_t)STAGES * kStageBytes >= (size_t)WAVES_MN * FM * FN * 16 * 64 * 4, "the stages hold one group's sums");
        f32x4* const x = reinterpret_cast<f32x4*>(lds_raw) + (size_t)wave_mn * (4 * FM * FN) * 64 + lane;
        __syncthreads();   // the last sub-step's (unused) fragment reads are done too
        if (kw == 1) {
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        f32x4 v;
                        v.x = acc[i][j][4 * q]; v.y = acc[i][j][4 * q + 1]; v.z = acc[i][j][4 * q + 2]; v.w = acc[i][j][4 * q + 3];
                        x[((i * FN + j) * 4 + q) * 64] = v;
                    }
        }
        __syncthreads();
        if (kw == 1) return;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const f32x4 v = x[((i * FN + j) * 4 + q) * 64];
                    acc[i][j][4 * q] += v.x; acc[i][j][4 * q + 1] += v.y; acc[i][j][4 * q + 2] += v.z; acc[i][j][4 * q + 3] += v.w;
                }
    }

    if constexpr (SPLIT) {
        constexpr int THREADS = WAVES * 64;
        constexpr size_t kTileQuads = (size_t)BM * BN / 4;
        const int tile_id = tm * g.tiles_n + tn;
        f32x4* const slot = reinterpret_cast<f32x4*>(g.partials) + (size_t)tile_id * kTileQuads;
        // everybody is through with the LDS tiles; one word of them carries the ticket to the workgroup
        __syncthreads();
        unsigned* const drawn = reinterpret_cast<unsigned*>(lds_raw);
        if (threadIdx.x == 0)
            *drawn = __hip_atomic_fetch_add(&dtl_tickets[g.split_slot][tile_id], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const bool last = *drawn == 1u;
        // Quad q of accumulator block (i, j) of thread t sits at quad index ((i*FN + j)*4 + q)*THREADS + t of the
        // partial tile (a kilobyte per wave and instruction).  One block at a time, with a running pointer and a
        // fence after each block: the kernel has no registers to spare for addresses formed ahead of time.
        if (!last) {
            f32x4* at = slot + threadIdx.x;
#pragma unroll
            for (int blk = 0; blk < FM * FN; blk++) {
                const int i = blk / FN, j = blk % FN;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    f32x4 v;
                    v.x = acc[i][j][4 * q]; v.y = acc[i][j][4 * q + 1]; v.z = acc[i][j][4 * q + 2]; v.w = acc[i][j][4 * q + 3];
                    store_device_coherent(at, v);
                    at += THREADS;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            wait_vmem<0>();   // this thread's stores have reached the level every XCD sees
            __syncthreads();  // ... and so have every other thread's of this workgroup
            if (threadIdx.x == 0)
                __hip_atomic_fetch_add(&dtl_arrived[g.split_slot][tile_id], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        // The second to draw: the other slice drew first, so it is past its K loop and on its way through the few
        // lines above, which wait for nothing -- the wait below is for stores already in flight.  It is bounded all
        // the same (a second or so): should the counters ever be out of step -- a product killed half way leaves
        // them so -- the tile is filled with NaN rather than summed from a partial that is not there.
        if (threadIdx.x == 0) {
            unsigned seen = 0;
            for (int spin = 0; spin < (1 << 22); spin++) {
                seen = __hip_atomic_load(&dtl_arrived[g.split_slot][tile_id], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (seen >= 1u) break;
                __builtin_amdgcn_s_sleep(4);
            }
            *drawn = seen >= 1u ? 1u : 0u;
        }
        __syncthreads();
        if (*drawn == 0u) {
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[i][j][v] = __builtin_nanf("");
        } else {
            // two terms: the sum is the same whichever of them is the one held in registers, so the bits do not
            // depend on which slice drew last
            const f32x4* at = slot + threadIdx.x;
#pragma unroll
            for (int blk = 0; blk < FM * FN; blk++) {
                const int i = blk / FN, j = blk % FN;
                f32x4 v[4];
                load4_device_coherent(v, at, THREADS);
                at += 4 * THREADS;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    acc[i][j][4 * q] += v[q].x;
                    acc[i][j][4 * q + 1] += v[q].y;
                    acc[i][j][4 * q + 2] += v[q].z;
                    acc[i][j][4 * q + 3] += v[q].w;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (threadIdx.x == 0) {
            // ready for the next product; written the way the counters are read and added to (an ordinary store
            // would sit in this XCD's L2, out of sight of the other XCDs' atomics, until the kernel ends)
            __hip_atomic_store(&dtl_tickets[g.split_slot][tile_id], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&dtl_arrived[g.split_slot][tile_id], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }

    // acc[i][j][v] is C[row, col] with
    //   row = wm*WM + i*32 + (v/4)*8 + (lane/32)*4 + v%4,  col = wn*WN + j*32 + lane%32
    TC* c_base = static_cast<TC*>(g.c) + batch * g.sc;
    TC* c2_base = GELU ? static_cast<TC*>(g.c2) + batch * g.sc : nullptr;
    // (two groups of waves: the batch index is eight registers too many; run_plan keeps such batches from them)
    const float* const bias_row = g.bias && KW == 1 ? g.bias + batch * g.sbias : g.bias;
    const TC* old_base = g.addend ? static_cast<const TC*>(g.addend) + batch * g.sc : c_base;  // read when accumulating
    if (row0 + BM <= g.m && col0 + BN <= g.n) {
        // Interior tile: straight-line code without guards, one 32x32 block of accumulators at a time.  A block's
        // 16 stores leave back to back; when accumulating, the old C of the next block is read before the stores
        // of this one are issued, so the wait for those reads lets the stores stay in flight.  (In the guarded path
        // below, a read of C next to each store puts a wait for ALL outstanding memory operations in front of
        // every element: each store then completes before the next is issued.)  Addresses are a wave-uniform row
        // base plus one per-lane offset; dtl_applies has checked that the offset fits 32 bits.  The fences keep
        // the compiler from forming the addresses of all 128 elements ahead of the first store, which takes more
        // registers than there are.
        const unsigned lane_bytes = (unsigned)(((lane >> 5) * 4 * g.ldc + (lane & 31)) * (long long)sizeof(TC));
        const long long tile_at = (row0 + __builtin_amdgcn_readfirstlane(wm) * WM) * g.ldc + col0 +
                                  __builtin_amdgcn_readfirstlane(wn) * WN;
        char* const c_tile = reinterpret_cast<char*>(c_base + tile_at);
        char* const c2_tile = GELU ? reinterpret_cast<char*>(c2_base + tile_at) : nullptr;
        char* const old_tile = reinterpret_cast<char*>(const_cast<TC*>(old_base) + tile_at);
        auto element = [&](char* tile, int blk, int v) {
            const int i = blk / FN, j = blk % FN;
            return reinterpret_cast<TC*>(tile + (i * 32 + (v >> 2) * 8 + (v & 3)) * g.ldc * (long long)sizeof(TC) +
                                         j * 32 * sizeof(TC) + lane_bytes);
        };
        float bias[FN];
#pragma unroll
        for (int j = 0; j < FN; j++) bias[j] = bias_row ? bias_row[col0 + wn * WN + j * 32 + (lane & 31)] : 0.f;
        auto interior = [&](auto adds) {
            constexpr bool ADDS = decltype(adds)::value;
            // alpha made opaque per form, or the compiler merges the scaling of all 128 elements of the two forms
            // into one pass ahead of the branch and spills its results
            float alpha = g.alpha;
            asm volatile("" : "+v"(alpha));
            float was[2][16];
            auto fetch = [&](int blk) {
#pragma unroll
                for (int v = 0; v < 16; v++) was[blk & 1][v] = c_load<TC>(element(old_tile, blk, v));
            };
            if (ADDS) fetch(0);
#pragma unroll
            for (int blk = 0; blk < FM * FN; blk++) {
                const int i = blk / FN, j = blk % FN;
                if (ADDS && blk + 1 < FM * FN) fetch(blk + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    float o = alpha * acc[i][j][v] + bias[j];
                    if (ADDS) o += was[blk & 1][v];
                    // A 16-bit C is the rounded copy of this fp32 value, the same bits a later product would make
                    // of an fp32 C on loading it.  Left alone, the compiler merges the multiply-add and the
                    // narrowing into one mixed-precision instruction whose result differs in the last place.
                    if (sizeof(TC) == 2) asm volatile("" : "+v"(o));
                    if (shared_tile(BM, BN, KT)) c_store_past<TC>(element(c_tile, blk, v), o);
                    else c_store<TC>(element(c_tile, blk, v), o);
                    // the activation is taken of the fp32 value, not of its rounded copy
                    if (GELU) c_store<TC>(element(c2_tile, blk, v), gelu_one(o));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (g.accumulate) {
            interior(std::true_type{});
        } else {
            interior(std::false_type{});
        }
        return;
    }
    // Edge tiles: the same straight line, through buffer resources that end with the last element of C: rows past m
    // lie beyond their end, columns past n are sent there; loads from there read zero, stores to there are dropped.
    // (With a bounds test around every element, each store waited for the one before: the [1002 x 6144] projection
    // from K = 2048 went from 43 to 34 us, a [78 x 4096] product from 22 to 16.)
    const long long tile_at = (row0 + __builtin_amdgcn_readfirstlane(wm) * WM) * g.ldc + col0 + __builtin_amdgcn_readfirstlane(wn) * WN;
    const long long tile_left = (g.m - 1 - row0 - __builtin_amdgcn_readfirstlane(wm) * WM) * g.ldc + g.n - col0 - __builtin_amdgcn_readfirstlane(wn) * WN;
    auto c_buffer = [&](const TC* base) {
        const long long left = tile_left * (long long)sizeof(TC);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<TC*>(base) + tile_at, 0, left <= 0 ? 0 : left > (long long)kPastEnd ? (int)kPastEnd : (int)left, 0x00020000);
    };
    const auto cb = c_buffer(c_base), c2b = c_buffer(GELU ? c2_base : c_base), oldb = c_buffer(old_base);
    float bias[FN];
    unsigned lane_at[FN];
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const long long col = col0 + wn * WN + j * 32 + (lane & 31);
        bias[j] = bias_row && col < g.n ? bias_row[col] : 0.f;
        lane_at[j] = col < g.n ? (unsigned)(((lane >> 5) * 4 * g.ldc + j * 32 + (lane & 31)) * (long long)sizeof(TC)) : kPastEnd;
    }
    // a row offset added to kPastEnd stays past the end: the tile spans less than 2^31 bytes (kEdgeColumns)
    auto at = [&](int blk, int v) {
        return lane_at[blk % FN] + (unsigned)((blk / FN * 32 + (v >> 2) * 8 + (v & 3)) * (int)g.ldc * (int)sizeof(TC));
    };
    auto edge = [&](auto adds) {
        constexpr bool ADDS = decltype(adds)::value;
        float alpha = g.alpha;
        asm volatile("" : "+v"(alpha));
        float was[2][16];
        auto fetch = [&](int blk) {
#pragma unroll
            for (int v = 0; v < 16; v++) was[blk & 1][v] = buffer_read<TC>(oldb, at(blk, v));
        };
        if (ADDS) fetch(0);
#pragma unroll
        for (int blk = 0; blk < FM * FN; blk++) {
            const int i = blk / FN, j = blk % FN;
            if (ADDS && blk + 1 < FM * FN) fetch(blk + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 16; v++) {
                float o = alpha * acc[i][j][v] + bias[j];
                if (ADDS) o += was[blk & 1][v];
                if (sizeof(TC) == 2) asm volatile("" : "+v"(o));  // as in the interior form
                buffer_write<TC>(cb, at(blk, v), o);
                if (GELU) buffer_write<TC>(c2b, at(blk, v), gelu_one(o));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (g.accumulate) {
        edge(std::true_type{});
    } else {
        edge(std::false_type{});
    }
}

// ---- the same product with workgroups that stay -------------------------------------------------
// 32 workgroups per XCD walk the tiles of that XCD's share instead of one workgroup being launched per tile; the
// tile order, the K walk and the order of every sum are those of gemm_dtl_kernel, so the bits are too.  What it
// buys: a workgroup issues the first two K stages of its NEXT tile before the C stores of the current one, and lets
// up to 63 of those stores stay in flight through the next tile's first K step -- the 2.3 us a fresh workgroup
// spends being launched and waiting for its first operand tile disappear behind the epilogue.  Measured on products
// of the BLOOM-7B1 block (same run, before / after): weight gradient [16384 x 4096] from K = 2048 253 -> 245 us,
// from K = 512 99 -> 95 us, [4096 x 4096] 66.2 -> 64.6, h -> 4h forward 241 -> 237.
// Memory operations complete in issue order on this target, which is what the partial waits rest on: after the 16
// operand loads of the next tile come the wave's 128 stores, so "at most 63 outstanding" means the loads are in.
// PAST: an fp32 C is stored past the caches (past_caches).
// Plain products only: 256 x 256 tiles, all of them interior (m, n multiples of 256), one batch, no bias, nothing
// accumulated, no second output (walk_applies); everything else takes gemm_dtl_kernel.
template <int CT, bool A_KSTR, bool B_KSTR, typename TC, bool PAST>
__global__ __launch_bounds__(512) void gemm_dtl_walk_kernel(GemmArgs g) {
    constexpr int BM = 256, BN = 256, WM = 64, WN = 128, KT = 64, STAGES = 2;
    constexpr int WAVES = (BM / WM) * (BN / WN);
    constexpr int FM = WM / 32, FN = WN / 32, KS = KT / 16;
    using TA = DtlTile<BM, KT, WAVES, A_KSTR>;
    using TB = DtlTile<BN, KT, WAVES, B_KSTR>;
    constexpr int kStageBytes = TA::kBytes + TB::kBytes;
    constexpr int kLoads = TA::kPerWave + TB::kPerWave;
    static_assert(FM * FN * 16 >= 63, "the partial wait counts on at least 63 stores per wave and tile");
    __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[STAGES * kStageBytes];
    const lds_byte* lds = (const lds_byte*)lds_raw;
    const unsigned lds0 = (unsigned)(unsigned long long)lds;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / (BN / WN), wn = wave % (BN / WN);
    // workgroup ids are dealt to the 8 XCDs round-robin: this one is number `slot` of `slots` on XCD `xcd`, whose
    // share of the tile order is [xcd * per_xcd, (xcd + 1) * per_xcd), as in tile_coords
    const int per_xcd = g.tiles_m * g.tiles_n / 8;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
    const int my_tiles = (per_xcd - slot + slots - 1) / slots;
    const int nk = (int)(g.k / KT);

    unsigned fa_off[FM][KS], fb_off[FN][KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
#pragma unroll
        for (int i = 0; i < FM; i++) fa_off[i][ks] = TA::frag_offset(wm * WM + i * 32, ks, lane);
#pragma unroll
        for (int j = 0; j < FN; j++) fb_off[j][ks] = TA::kBytes + TB::frag_offset(wn * WN + j * 32, ks, lane);
    }
    // interior tiles: a lane's chunk offsets inside the operand tiles are the same for every tile
    unsigned a_off[TA::kPerWave], b_off[TB::kPerWave];
#pragma unroll
    for (int q = 0; q < TA::kPerWave; q++) a_off[q] = TA::source_offset(q, wave, lane, g.lda, 0, g.m);
#pragma unroll
    for (int q = 0; q < TB::kPerWave; q++) b_off[q] = TB::source_offset(q, wave, lane, g.ldb, 0, g.n);
    const long long a_step = A_KSTR ? 2 * KT * g.lda : 2 * KT;
    const long long b_step = B_KSTR ? 2 * KT * g.ldb : 2 * KT;

    const unsigned char* a_src = nullptr;
    const unsigned char* b_src = nullptr;
    int until_wrap = 0;
    long long row0 = 0, col0 = 0;
    auto setup = [&](int it) {   // the it-th tile of this workgroup: origins and the start of its K walk
        int tm, tn;
        tile_in_order(g, xcd * per_xcd + it * slots + slot, tm, tn);
        tm = __builtin_amdgcn_readfirstlane(tm);
        tn = __builtin_amdgcn_readfirstlane(tn);
        row0 = (long long)tm * BM;
        col0 = (long long)tn * BN;
        const int first = (int)(k_walk_start(row0, col0, g.k) / KT);
        a_src = reinterpret_cast<const unsigned char*>(g.a) + 2 * (A_KSTR ? row0 : row0 * g.lda) + first * a_step;
        b_src = reinterpret_cast<const unsigned char*>(g.b) + 2 * (B_KSTR ? col0 : col0 * g.ldb) + first * b_step;
        until_wrap = nk - first;
    };
    auto issue = [&](int tile) {
        const unsigned dst = lds0 + (unsigned)(tile % STAGES) * kStageBytes + (unsigned)wave * 1024u;
#pragma unroll
        for (int q = 0; q < kLoads; q++) {
            if (q < TA::kPerWave) dtl_load(dst + q * WAVES * 1024, a_off[q], a_src);
            else dtl_load(dst + TA::kBytes + (q - TA::kPerWave) * WAVES * 1024, b_off[q - TA::kPerWave], b_src);
        }
        const bool wraps = --until_wrap == 0;
        a_src += wraps ? a_step - nk * a_step : a_step;
        b_src += wraps ? b_step - nk * b_step : b_step;
    };
    f32x16 acc[FM][FN];
    auto step = [&](const u32x4 (&fa)[FM], const u32x4 (&fb)[FN], u32x4 (&na)[FM], u32x4 (&nb)[FN], int tile, int ks) {
        const lds_byte* stage = lds + (tile % STAGES) * kStageBytes;
#pragma unroll
        for (int idx = 0; idx < FM * FN; idx++) {
            const int i = idx % FM, j = idx / FM;
            if (idx == 0) nb[0] = TB::fragment(stage, fb_off[0][ks]);
            else if (idx <= FM) na[idx - 1] = TA::fragment(stage, fa_off[idx - 1][ks]);
            else if (idx < FM + FN) nb[idx - FM] = TB::fragment(stage, fb_off[idx - FM][ks]);
            acc[i][j] = Cvt<CT>::mfma(fa[i], fb[j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    setup(0);
    issue(0);
    if (nk > 1) issue(1);
    for (int it = 0; it < my_tiles; it++) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
        // K stage 0 of this tile has to be in LDS.  First tile: nothing but its two stages is outstanding.  Later
        // tiles: both stages were issued ahead of the previous tile's stores, so they have landed once at most 63
        // operations (all of them stores) are outstanding.
        if (nk == 1) wait_vmem<0>();
        else if (it == 0) wait_vmem<kLoads>();
        else wait_vmem<63>();
        __syncthreads();
        u32x4 fa0[FM], fb0[FN], fa1[FM], fb1[FN];
#pragma unroll
        for (int i = 0; i < FM; i++) fa0[i] = TA::fragment(lds, fa_off[i][0]);
#pragma unroll
        for (int j = 0; j < FN; j++) fb0[j] = TB::fragment(lds, fb_off[j][0]);
        __builtin_amdgcn_sched_barrier(0);
        for (int t = 0; t < nk; t++) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                u32x4(&fa_now)[FM] = (ks & 1) ? fa1 : fa0;
                u32x4(&fb_now)[FN] = (ks & 1) ? fb1 : fb0;
                u32x4(&fa_next)[FM] = (ks & 1) ? fa0 : fa1;
                u32x4(&fb_next)[FN] = (ks & 1) ? fb0 : fb1;
                if (ks + 1 < KS) {
                    step(fa_now, fb_now, fa_next, fb_next, t, ks + 1);
                } else {
                    // K stage t+1 has to be in LDS: the only loads in flight, except during step 0 of a later tile,
                    // when stage 1 is already in and up to 63 of the previous tile's stores may go on draining
                    if (t == 0 && it > 0) wait_vmem<63>(); else wait_vmem<0>();
                    __syncthreads();
                    if (t + STAGES < nk) issue(t + STAGES);
                    __builtin_amdgcn_sched_barrier(0);
                    step(fa_now, fb_now, fa_next, fb_next, t + 1, 0);
                }
            }
        }
        // Every wave is past the last barrier of the K loop and nothing in LDS is read for its value any more (the
        // loop's trailing fragment reads fetch a stage that does not exist): the next tile's first stages may go.
        const long long st_row0 = row0, st_col0 = col0;
        if (it + 1 < my_tiles) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            setup(it + 1);
            issue(0);
            if (nk > 1) issue(1);
        }
        // acc[i][j][v] is C[row, col] with row = wm*WM + i*32 + (v/4)*8 + (lane/32)*4 + v%4, col = wn*WN + j*32 + lane%32
        const unsigned lane_bytes = (unsigned)(((lane >> 5) * 4 * g.ldc + (lane & 31)) * (long long)sizeof(TC));
        const long long tile_at = (st_row0 + wm * WM) * g.ldc + st_col0 + wn * WN;
        char* const c_tile = reinterpret_cast<char*>(static_cast<TC*>(g.c) + tile_at);
        float alpha = g.alpha;
        asm volatile("" : "+v"(alpha));
#pragma unroll
        for (int blk = 0; blk < FM * FN; blk++) {
            const int i = blk / FN, j = blk % FN;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 16; v++) {
                float o = alpha * acc[i][j][v] + 0.f;   // the plain epilogue's expression with its bias of zero
                if (sizeof(TC) == 2) asm volatile("" : "+v"(o));   // one fp32 value, then one rounding (see gemm_dtl_kernel)
                TC* const to = reinterpret_cast<TC*>(c_tile + (i * 32 + (v >> 2) * 8 + (v & 3)) * g.ldc * (long long)sizeof(TC) +
                                                     j * 32 * sizeof(TC) + lane_bytes);
                if (PAST) c_store_past<TC>(to, o);
                else c_store<TC>(to, o);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Whether every row of an fp32 C starts on a 128-byte line: a wave's store of 32 columns is then one whole line.
inline bool rows_on_lines(const GemmArgs& g) { return (reinterpret_cast<uintptr_t>(g.c) & 127) == 0 && g.ldc % 32 == 0; }

// Whether the walking form stores an fp32 C past the caches: one that the 256 MB of the last level cannot hold, where it would
// push the operands out, and that has products between its stores.  Ordinary stores / these, us: [250880 x 4096] from K = 512
// 1480 / 1270, [32768 x 4096] from 1024 300 / 272, [8192 x 8192] from 1024 144 / 139, [5120 x 16384] from 2048 312 / 303; of a
// C that fits the cache [2048 x 8192] from 1024, 2048 40.3 / 42.1, 66.3 / 68.2, [4096 x 8192] 76.4 / 77.6, 126.1 / 128.2; from
// K = 64 [2048 x 8192] 14.6 / 17.5, [4096 x 32768] 111 / 114.
inline bool past_caches(const GemmArgs& g) { return rows_on_lines(g) && g.m * g.n * 4 >= 256LL << 20 && g.k >= 128; }

// Whether the walking form takes a product the plan has put on 256 x 256 tiles.
inline bool walk_applies(const GemmArgs& g, long long batch) {
    const long long tiles = (g.m / 256) * (g.n / 256);
    return batch == 1 && g.m % 256 == 0 && g.n % 256 == 0 && g.k % 64 == 0 && tiles >= 256 && tiles % 8 == 0 &&
           tiles <= 0x7fffffffLL && !g.bias && !g.accumulate && !g.c2 && !g.addend && g.splits == 1;
}

template <int CT>
int launch_dtl_walk(GemmArgs g, const Problem& p, hipStream_t st) {
    g.tiles_m = (int)(g.m / 256);
    g.tiles_n = (int)(g.n / 256);
    using F16 = __half;
    using BF16 = __hip_bfloat16;
#define BR_DTL_WALK_CASE(AK, BK_)                                                        \
    if (p.a_kstr == AK && p.b_kstr == BK_) {                                             \
        if (p.c_dtype == BR_F32 && past_caches(g))                                       \
            gemm_dtl_walk_kernel<CT, AK, BK_, float, true><<<256, 512, 0, st>>>(g);      \
        else if (p.c_dtype == BR_F32)                                                    \
            gemm_dtl_walk_kernel<CT, AK, BK_, float, false><<<256, 512, 0, st>>>(g);     \
        else if (CT == BR_GEMM_F16)                                                      \
            gemm_dtl_walk_kernel<CT, AK, BK_, F16, false><<<256, 512, 0, st>>>(g);       \
        else                                                                             \
            gemm_dtl_walk_kernel<CT, AK, BK_, BF16, false><<<256, 512, 0, st>>>(g);      \
    }
    BR_DTL_WALK_CASE(false, false)
    BR_DTL_WALK_CASE(false, true)
    BR_DTL_WALK_CASE(true, false)
    BR_DTL_WALK_CASE(true, true)
#undef BR_DTL_WALK_CASE
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// ---- host-side dispatch -------------------------------------------------------
template <int CT, int BM, int BN, int WM, int WN, int KT, int ST, int KW = 1>
int launch_dtl_config(GemmArgs g, const Problem& p, long long batch, hipStream_t st) {
    constexpr int THREADS = (BM / WM) * (BN / WN) * KW * 64;
    g.tiles_m = (int)((g.m + BM - 1) / BM);
    g.tiles_n = (int)((g.n + BN - 1) / BN);
    if (g.splits > 1) {
        // the plan only splits unbatched products whose partial tiles fit the workspace it was given
        const long long tiles = (long long)g.tiles_m * g.tiles_n;
        if (g.splits != 2 || batch != 1 || tiles > kMaxSplitTiles || !g.partials ||
            (size_t)tiles * BM * BN * sizeof(float) > g.partial_bytes)   // one partial tile per output tile
            return BR_ERR_ATTR;
    }
    const long long blocks = (long long)g.tiles_m * g.tiles_n * batch * g.splits;
    if (blocks > 0x7fffffffLL) return BR_ERR_ATTR;
    const unsigned grid = (unsigned)blocks;
    using F16 = __half;
    using BF16 = __hip_bfloat16;
    if (g.splits == 2) {
        // the two-slice form: its own instantiations (of the two 256-row tiles, the only ones it is planned on),
        // so that the unsplit kernels carry none of its code
        if (g.c2 || BM != 256 || KW != 1) return BR_ERR_TODO;
#define BR_DTL_SPLIT_CASE(AK, BK_)                                                                              \
    if constexpr (BM == 256 && KW == 1) if (p.a_kstr == AK && p.b_kstr == BK_) {                                                          \
        if (p.c_dtype == BR_F32)                                                                                 \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, AK, BK_, float, false, true><<<grid, THREADS, 0, st>>>(g); \
        else if (CT == BR_GEMM_F16)                                                                              \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, AK, BK_, F16, false, true><<<grid, THREADS, 0, st>>>(g);   \
        else                                                                                                     \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, AK, BK_, BF16, false, true><<<grid, THREADS, 0, st>>>(g);  \
    }
        BR_DTL_SPLIT_CASE(false, false)
        BR_DTL_SPLIT_CASE(false, true)
        BR_DTL_SPLIT_CASE(true, false)
        BR_DTL_SPLIT_CASE(true, true)
#undef BR_DTL_SPLIT_CASE
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
    if (g.c2) {
        // GELU epilogue: built for the linear layer's layout only (both operands k-contiguous, 16-bit outputs)
        if (p.a_kstr || p.b_kstr || p.c_dtype == BR_F32) return BR_ERR_TODO;
        if (CT == BR_GEMM_F16)
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, false, false, F16, true, false, KW><<<grid, THREADS, 0, st>>>(g);
        else
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, false, false, BF16, true, false, KW><<<grid, THREADS, 0, st>>>(g);
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
#define BR_DTL_CASE(AK, BK_)                                                                           \
    if (p.a_kstr == AK && p.b_kstr == BK_) {                                                            \
        if (p.c_dtype == BR_F32)                                                                        \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, AK, BK_, float, false, false, KW><<<grid, THREADS, 0, st>>>(g);   \
        else if (CT == BR_GEMM_F16)                                                                     \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, AK, BK_, F16, false, false, KW><<<grid, THREADS, 0, st>>>(g);     \
        else                                                                                            \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, KT, ST, AK, BK_, BF16, false, false, KW><<<grid, THREADS, 0, st>>>(g);    \
    }
    BR_DTL_CASE(false, false)
    BR_DTL_CASE(false, true)
    BR_DTL_CASE(true, false)
    BR_DTL_CASE(true, true)
#undef BR_DTL_CASE
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// The ragged form: K not a multiple of 64, or slices of K that are not all alike.  In every layout and with either type
// of C: on 64 x 64 tiles instead, as some of them ran, [4096 x 4096] from K = 1056 took 77 us with A and B both stored
// the other way round and 70 us as a weight gradient in 16 bits; on large tiles 43 and 42.
template <int CT, int BM, int BN, int WM, int WN, int ST>
int launch_dtl_ragged(GemmArgs g, const Problem& p, long long batch, hipStream_t st) {
    constexpr int THREADS = (BM / WM) * (BN / WN) * 64;
    using C16 = std::conditional_t<CT == BR_GEMM_F16, __half, __hip_bfloat16>;
    g.tiles_m = (int)((g.m + BM - 1) / BM);
    g.tiles_n = (int)((g.n + BN - 1) / BN);
    const long long blocks = (long long)g.tiles_m * g.tiles_n * (g.splits > 1 ? g.splits : batch);
    if (blocks > 0x7fffffffLL) return BR_ERR_ATTR;
    const unsigned grid = (unsigned)blocks;
    if (g.c2) {
        if (p.a_kstr || p.b_kstr || p.c_dtype == BR_F32) return BR_ERR_TODO;
        gemm_dtl_kernel<CT, BM, BN, WM, WN, 64, ST, false, false, C16, true, false, 1, true><<<grid, THREADS, 0, st>>>(g);
        BR_HIP_LAUNCH_CHECK();
        return BR_OK;
    }
#define BR_DTL_RAGGED_CASE(AK, BK_)                                                                                       \
    if (p.a_kstr == AK && p.b_kstr == BK_) {                                                                              \
        if (p.c_dtype == BR_F32)                                                                                          \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, 64, ST, AK, BK_, float, false, false, 1, true><<<grid, THREADS, 0, st>>>(g); \
        else                                                                                                              \
            gemm_dtl_kernel<CT, BM, BN, WM, WN, 64, ST, AK, BK_, C16, false, false, 1, true><<<grid, THREADS, 0, st>>>(g);   \
    }
    BR_DTL_RAGGED_CASE(false, false)
    BR_DTL_RAGGED_CASE(false, true)
    BR_DTL_RAGGED_CASE(true, false)
    BR_DTL_RAGGED_CASE(true, true)
#undef BR_DTL_RAGGED_CASE
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// The direct-to-LDS kernels apply when both operands are 16-bit and 16-byte aligned, a k-contiguous operand's rows
// end on a 16-byte granule of their own (K a multiple of 8, or zero-filled up to one), and every per-lane offset fits
// 32 bits: of the operands, and of the four rows of C a lane of a whole tile spans.  The edge epilogue's offsets span up
// to 256 rows: partial tiles of a C of kEdgeColumns or more columns are left to other kernels (run_plan in gemm.hip).
constexpr long long kEdgeColumns = 1LL << 21;
inline bool dtl_spans(bool a_kstr, long long lda, bool b_kstr, long long ldb, long long ldc, long long m, long long n, long long k) {
    const long long lim = 1LL << 31;
    const long long a_span = a_kstr ? 2 * 64 * lda : 2 * 256 * lda;
    const long long b_span = b_kstr ? 2 * 64 * ldb : 2 * 256 * ldb;
    return a_span < lim && b_span < lim && ldc < (1LL << 27) && m < lim && n < lim && k < lim;
}
inline bool dtl_applies(const GemmArgs& g, const Problem& p) {
    if (p.a_f32 || p.b_f32 || !g.vec_a || !g.vec_b || g.k <= 0) return false;
    if (g.k % 8 != 0 && !p.padded && !(p.a_kstr && p.b_kstr)) return false;
    return dtl_spans(p.a_kstr, g.lda, p.b_kstr, g.ldb, g.ldc, g.m, g.n, g.k);
}

// bytes of partial tiles the two-slice split wants in the caller's workspace (one per output tile)
inline size_t pair_bytes(const Plan& plan, long long m, long long n) {
    if (!plan.pair) return 0;
    const KernelCost& c = kCost[plan.kernel];
    return (size_t)(ceil_div(m, c.bm) * ceil_div(n, c.bn)) * c.bm * c.bn * sizeof(float);
}

// The counter set of a stream (-1: all sets are taken by other streams).
inline int split_slot_of(hipStream_t st) {
    static std::mutex mu;
    static hipStream_t owner[kSplitSlots];
    static int used = 0;
    std::lock_guard<std::mutex> lock(mu);
    for (int i = 0; i < used; i++)
        if (owner[i] == st) return i;
    if (used == kSplitSlots) return -1;
    owner[used] = st;
    return used++;
}

// The two-slice form of a plan with `pair` set.
template <int CT>
int launch_dtl_pair(GemmArgs g, const Problem& p, int kernel, int slot, hipStream_t st) {
    g.splits = 2;
    g.split_slot = slot;
    if (kernel == kTile256) return launch_dtl_config<CT, 256, 256, 64, 128, 64, 2>(g, p, 1, st);
    return launch_dtl_config<CT, 256, 128, 64, 64, 64, 3>(g, p, 1, st);
}

// A weight gradient from few tokens -- fp32 C, short K -- spends as long storing its tiles as multiplying, and one
// workgroup per CU does the two in turn: 256 x 256 tiles take 56 us over a [16384 x 4096] gradient before the first K
// value counts (48 us per 512 of them).  On tiles of half the size two workgroups share a CU, and the stores of one pass
// under the products of the other.  128 x 256 tiles, one / two workgroups to a CU, us, operands from memory (the sums are
// the same, and the bits; A k-contiguous the same within 3 %):
//                    K = 64          128            256            512            768
//   [ 2048,  6144]   13.1 / 12.9    14.6 / 14.0    17.2 / 15.5    22.0 / 20.6    27.1 / 26.2
//   [ 4096,  4096]   16.3 / 14.4    18.3 / 15.8    21.0 / 17.9    27.1 / 24.0    33.8 / 30.8
//   [ 8192,  2048]   14.9 / 15.0    16.8 / 16.1    19.5 / 18.0    25.8 / 24.2    32.5 / 31.0
//   [ 2048,  8192]   14.5 / 16.9    16.2 / 17.7    19.2 / 19.2    25.7 / 26.2    32.1 / 32.2
//   [ 1024, 16384]   14.2 / 18.1    16.1 / 18.9    19.3 / 19.5    26.1 / 26.5    33.7 / 33.8
//   [ 2560,  6400]   15.1 / 15.6    16.9 / 16.9    20.1 / 19.2    26.6 / 25.2    33.6 / 31.8
//   [12288,  4096]   43.1 / 36.0    46.0 / 37.9    54.8 / 45.3    75.2 / 65.7    94.6 / 86.1
//   [ 8192,  8192]   55.0 / 52.3    56.6 / 55.4    63.9 / 62.1    93.3 / 85.2   119.5 / 113
//   [16384,  4096]   54.9 / 46.4    58.4 / 48.1    68.4 / 55.9    94.6 / 82.6   122.3 / 113
//   [20480,  5120]   84.9 / 85.6    88.2 / 84.5    98.6 / 88.8   143.8 / 130    187.2 / 177
//   [250880, 4096]                                 790 / 854     1204 / 1306    1818 / 2026
// Where one round of 256 x 256 tiles holds all of C nothing follows a tile whose products its stores could pass under, and
// rows 32 KB apart lose: such products stay there.  So do those of K = 64 within one round or past four, where either
// way the stores are all there is (2-4 % lost), and any from K = 1024 on (a block's step loses more elsewhere than it gains:
// 755 -> 760 us of [1024 x 2048] as separate words).
// 256 x 128 tiles store columns of 256 rows: with rows 32 KB apart [8192 x 8192] 79.6, 100 and 121 us from K = 64, 512 and
// 768, [4096 x 16384] 76, 104 and 127; elsewhere within 3 % of these, a model's step of 512 tokens 0-2 % slower.
// Two workgroups' stores go past the caches, which takes whole 128-byte lines: a C of rows that start elsewhere waits for
// memory at every line ([3000 x 5000] from K = 64, 512, 768 30.7, 40.6, 46.2 us, and 15.7, 26.6, 32.8 on 256 x 256 tiles).
// With B k-contiguous, or a C of 16 bits, there is less to hide: [12288 x 4096] from 1024 112 / 123 and 101 / 105.  Three K
// steps in flight instead of two: [16384 x 4096] from 512 91 -> 98.
inline bool shared_applies(const GemmArgs& g, const Problem& p, long long batch) {
    const long long tiles = ceil_div(g.m, 256) * ceil_div(g.n, 256);
    const bool one_round = tiles <= 256;
    return batch == 1 && p.b_kstr && p.c_dtype == BR_F32 && g.k <= 768 && tiles <= 2048 && rows_on_lines(g) &&
           (one_round ? g.k >= 128 && g.ldc % 8192 != 0 : g.k >= 128 || tiles <= 1024) &&
           !g.bias && !g.accumulate && !g.c2 && !g.addend && g.splits == 1;
}
template <int CT>
int launch_dtl_shared(GemmArgs g, const Problem& p, hipStream_t st) {
    g.tiles_m = (int)ceil_div(g.m, 128);
    g.tiles_n = (int)ceil_div(g.n, 256);
    const unsigned grid = (unsigned)(g.tiles_m * g.tiles_n);
    if (p.a_kstr) gemm_dtl_kernel<CT, 128, 256, 64, 128, 32, 2, true, true, float><<<grid, 256, 0, st>>>(g);
    else gemm_dtl_kernel<CT, 128, 256, 64, 128, 32, 2, false, true, float><<<grid, 256, 0, st>>>(g);
    BR_HIP_LAUNCH_CHECK();
    return BR_OK;
}

// K a multiple of 64 (kTile128Half: of 32), one workgroup per tile and batch entry.
template <int CT>
int launch_dtl(const GemmArgs& g, const Problem& p, int kernel, long long batch, hipStream_t st) {
    if (kernel == kTile256 && shared_applies(g, p, batch)) return launch_dtl_shared<CT>(g, p, st);
    if (kernel == kTile256 && walk_applies(g, batch)) return launch_dtl_walk<CT>(g, p, st);
    if (kernel == kTile256) return launch_dtl_config<CT, 256, 256, 64, 128, 64, 2>(g, p, batch, st);
    if (kernel == kTile256x128Groups) return launch_dtl_config<CT, 256, 128, 64, 128, 64, 3, 2>(g, p, batch, st);
    if (kernel == kTile256x128) return launch_dtl_config<CT, 256, 128, 64, 64, 64, 3>(g, p, batch, st);
    if (kernel == kTile128Half) return launch_dtl_config<CT, 128, 128, 64, 64, 32, 3>(g, p, batch, st);
    return launch_dtl_config<CT, 128, 128, 64, 64, 64, 2>(g, p, batch, st);
}

}  // namespace gemm16
}  // namespace brk
