// Which kernel a 16-bit product runs on, decided from its sizes alone: the
// bits of a result do not depend on where its operands or workspace lie.
//
// Every kernel's time is estimated from constants fitted to measurements on
// MI355X (fp16, 37 shapes from [64 x 256] to [50008 x 2048], each kernel
// unsplit and with K in 2, 4 and 8 slices; the estimates are within 8-15 % of
// the measured times, and choosing by them costs 1 % on average and 8 % at
// worst over choosing by the measurements):
//
//   us = start + rounds * (steps * max(step, load * groups) + round) + C bytes / 6 TB/s
//
//   steps   K steps one wave of a workgroup walks (64 k-values each)
//   rounds  workgroups / the number resident at a time
// and never less than what the operands take to arrive from memory (5.5 TB/s).
//
//   step    a K step when the CU runs one workgroup (latency of the walk)
//   load    a K step per resident workgroup and CU (LDS and L2 throughput)
#pragma once

#include <math.h>

namespace brk {
namespace gemm16 {

// in the order of the BR_GEMM_* constants
enum Kernel { kTile256, kTile256x128, kTile256x128Groups, kTile128, kFlex64, kFlex64Short, kFlex32x64, kFlex32, kRing64x128, kKernels };

struct KernelCost {
    int bm, bn;
    int k_waves;     // waves a tile's K steps are dealt to
    int resident;    // workgroups the chip holds at a time
    double start, step, load, round;
};
constexpr KernelCost kCost[kKernels] = {
    {256, 256, 1, 256, 4.47, 1.310, 1.655, 0.00},    // gemm_dtl16.hpp, 8 waves of 64 x 128
    {256, 128, 1, 256, 3.07, 0.840, 1.048, 0.89},    // 8 waves of 64 x 64
    {256, 128, 1, 256, 3.09, 0.789, 0.993, 2.48},    // two groups of four 64 x 128 waves
    {128, 128, 1, 512, 2.80, 0.737, 0.606, 0.00},    // 4 waves of 64 x 64
    {64, 64, 4, 512, 2.71, 0.856, 0.900, 1.44},      // gemm_flex.hpp, K dealt to 4 waves
    {64, 64, 2, 1024, 2.84, 0.745, 0.449, 1.99},     // ... to 2 waves, for many tiles or a short K
    {32, 64, 4, 768, 2.95, 0.681, 0.637, 0.44},
    {32, 32, 4, 512, 1.67, 0.472, 0.435, 1.15},
    // gemm_flex.hpp, ring of K steps.  From timings inside whole steps, where weights come from memory: K = 512 (32
    // products of [512 x 128]) 10-12 us against 8-10 on 64 x 64 tiles, K = 2048 20 against 22, K = 4096 35-39 against
    // 40-50, K = 6144 51 against 49 and K = 8192 54-60 against 52-59 on 256 x 128 tiles with K in four slices.
    {64, 128, 1, 256, 2.40, 0.380, 0.430, 2.20},
};

inline bool is_flex(int kernel) { return kernel >= kFlex64; }

struct Plan {
    int kernel = kTile128;
    int slices = 1;        // K in this many slices, partial sums in memory, a second kernel adds them
    bool pair = false;     // K in two halves inside the kernel (gemm_dtl16.hpp)
    long long tail_from = 0;   // columns from here on run as a second launch on 256x128 tiles
    double us = 1e30;
};

inline long long ceil_div(long long a, long long b) { return (a + b - 1) / b; }
// k-values of a slice: a multiple of 64, so that the last slice alone is ragged
inline long long slice_length(long long k, int slices) { return ceil_div(ceil_div(k, 64), slices) * 64; }

inline double kernel_us(int kernel, long long m, long long n, long long k, long long batch) {
    const KernelCost& c = kCost[kernel];
    const double groups = (double)(ceil_div(m, c.bm) * ceil_div(n, c.bn) * batch);
    const double resident = c.resident;
    // tiles that fill a CU by themselves go round by round; smaller workgroups start as others end
    const double rounds = groups <= resident ? 1.0 : c.resident == 256 ? ceil(groups / resident) : groups / resident;
    const double per_cu = (groups < resident ? groups : resident) / 256.0;
    const double step = c.step > c.load * per_cu ? c.step : c.load * per_cu;
    const double us = c.start + rounds * (step * (double)ceil_div(ceil_div(k, 64), c.k_waves) + c.round) + (double)m * n * batch * 4.0 / 6e6;
    const double memory = 3.0 + ((double)m * k * 2.0 + (double)n * k * 2.0 + (double)m * n * 4.0) * batch / 5.5e6;
    return us > memory ? us : memory + 0.02 * us;   // between two that memory bounds, the one with less to do
}
// the pass that adds the partial sums of `slices` slices
inline double reduce_us(long long m, long long n, int slices) { return 3.0 + (double)(slices + 1) * m * n * 4.0 / 5.5e6; }

constexpr int kMaxSplitTiles = 8192;   // the two-slice form's arrival counters per stream
// The two-slice form: one partial tile per output tile is written and read back through device-coherent accesses, by
// one half of the workgroups each while the others still multiply.  Timed on [2048 x 4096] outputs (K = 16384: 212 and
// 257 us by operand layout, K = 12288: 184); products of fewer than 1024 rows do better with many slices.
inline double pair_us(int kernel, long long m, long long n, long long k) {
    const KernelCost& c = kCost[kernel];
    const long long tiles = ceil_div(m, c.bm) * ceil_div(n, c.bn);
    if (m < 1024 || k % 64 != 0 || k / 64 < 16 || tiles > kMaxSplitTiles) return 1e30;
    const double rounds = (double)ceil_div(2 * tiles, 256);
    return c.start + rounds * (c.load * (double)ceil_div(k / 64, 2) + c.round) + (double)m * n * 4.0 / 6e6 +
           2.0 * (double)tiles * c.bm * c.bn * 4.0 / 5e6;
}

// A product whose 256x256 tiles fill some rounds of workgroups and then at most half of one more (the q|k|v
// projection of 2048 tokens: 384 tiles, a round and a half) leaves half the chip idle for a whole tile time, and on
// 256x128 tiles throughout it pays their lower rate on every round.  Run in two launches -- the columns that make
// whole rounds on 256x256 tiles, the rest on 256x128 tiles, which then fill one round -- the projection takes 188 us
// instead of 210 either way.  Returns the first column of the second launch, or 0 where this does not apply or does
// not beat `best_us`.  The seam falls on a multiple of 1024 columns, the period of k_walk_start.
inline long long column_tail(long long m, long long n, long long k, double best_us) {
    if (k % 64 != 0) return 0;
    const long long tm = ceil_div(m, 256), tn = ceil_div(n, 256);
    long long a = 256, b = tm;
    while (b) { const long long r = a % b; a = b; b = r; }   // a = gcd(256, tm)
    long long unit = 256 / a;                                // tile columns that make whole rounds
    if (unit < 4) unit = 4;                                  // a power of two; and a multiple of 1024 columns
    const long long tn_main = tn / unit * unit, tn_rest = tn - tn_main;
    if (tn_main == 0 || tn_rest == 0 || tm * tn_rest > 128) return 0;
    const double us = kernel_us(kTile256, m, tn_main * 256, k, 1) + kernel_us(kTile256x128Groups, m, n - tn_main * 256, k, 1);
    return us < best_us ? tn_main * 256 : 0;
}

// slices_allowed: the caller has a workspace for partial sums.
inline Plan gemm_plan(long long m, long long n, long long k, long long batch, bool slices_allowed) {
    Plan best;
    for (int c = 0; c < kKernels; c++) {
        // two groups of waves share a 64-wide K step: no ragged form
        if (c == kTile256x128Groups && k % 64 != 0) continue;
        for (int s = 1; s <= 16; s *= 2) {
            if (s > 1 && (!slices_allowed || batch != 1 || n % 4 != 0 || k / s < 256)) break;
            const long long per = slice_length(k, s);
            const int slices = (int)ceil_div(k, per);
            if (s > 1 && (slices < 2 || c == kTile256x128Groups)) break;
            const double us = s == 1 ? kernel_us(c, m, n, k, batch) : kernel_us(c, m, n, per, slices) + reduce_us(m, n, slices);
            // a split has to win clearly: it takes a second launch
            if (us < (s == 1 ? 1.0 : 0.97) * best.us) best = Plan{c, slices, false, 0, us};
        }
    }
    if (slices_allowed && batch == 1)
        for (int c = kTile256; c <= kTile256x128; c++) {
            const double us = pair_us(c, m, n, k);
            if (us < 0.97 * best.us) best = Plan{c, 1, true, 0, us};
        }
    const long long tail = batch == 1 ? column_tail(m, n, k, best.us) : 0;
    if (tail > 0) best = Plan{kTile256, 1, false, tail, best.us};
    return best;
}

// fp32 products (gemm_flex.hpp): the tile whose matrix instructions finish first.  A step of 32 k-values takes a wave
// 64 / 32 / 16 instructions of 64 clocks; measured with everything around them 2.45 / 1.4 / 0.78 us per step and
// workgroup of a CU, and 2.7 us besides.  A CU that holds one workgroup more than the others sets the time.
inline int fp32_kernel(long long m, long long n, long long k, long long batch) {
    auto us = [&](int kernel, double per_step) {
        const KernelCost& c = kCost[kernel];
        const double load = (double)(ceil_div(m, c.bm) * ceil_div(n, c.bn) * batch) / 256.0;
        return 2.7 + (load >= 4.0 ? load : ceil(load)) * (double)ceil_div(ceil_div(k, 32), 4) * per_step;
    };
    int best = kFlex64;
    double t = us(kFlex64, 2.45);
    if (us(kFlex32x64, 1.4) < 0.98 * t) best = kFlex32x64, t = us(kFlex32x64, 1.4);
    if (us(kFlex32, 0.78) < 0.98 * t) best = kFlex32;
    return best;
}

}  // namespace gemm16
}  // namespace brk
