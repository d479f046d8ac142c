// Which kernel a 16-bit product runs on, and whether K is cut into slices:
// planned from its sizes alone.  Products of the same sizes, types, layouts and
// alignment are summed in the same order at every call; operands that are not
// 16-byte aligned take the register-staged kernel instead, a caller without a
// workspace gets no slices, and a stream beyond the library's counter sets no
// two-slice form (split_slot_of), each with an order of its own.
//
// Every kernel's time is estimated from constants fitted to measurements on
// MI355X: fp16 operands read from memory, 668 sizes from [16 x 16] to
// [16384 x 4096], K = 16 to 16384, in the layouts of a linear layer's three
// products and of batched attention products, 871 products in all, each on
// every kernel, unsplit and with K in up to 16 slices
// (profiles/gemm_plan_measurements.txt).  Where a kernel is within a quarter of
// the fastest the estimates are off by 5-10 % (median; 12-26 % for one in ten).
// Choosing by them costs 1 % on average over choosing by the measurements, more
// than 7 % for one product in twenty.
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

#include <initializer_list>

namespace brk {
namespace gemm16 {

// in the order of the BR_GEMM_* constants
enum Kernel { kTile256, kTile256x128, kTile256x128Groups, kTile128, kTile128Half, kFlex64, kFlex64Short, kFlex32x64, kFlex32, kRing64x128, kKernels };
constexpr int kPairWide = kKernels;   // two products: gemm_wide_pair_kernel (gemm_pair.hpp)

struct KernelCost {
    int bm, bn;
    int k_waves;     // waves a tile's K steps are dealt to
    int resident;    // workgroups the chip holds at a time
    double start, step, load, round;
};
constexpr KernelCost kCost[kKernels] = {
    {256, 256, 1, 256, 4.63, 1.233, 1.724, 0.00},     // gemm_dtl16.hpp, 8 waves of 64 x 128
    {256, 128, 1, 256, 2.23, 0.845, 1.052, 2.18},     // 8 waves of 64 x 64
    {256, 128, 1, 256, 2.47, 0.753, 1.004, 3.44},     // two groups of four 64 x 128 waves
    {128, 128, 1, 512, 4.30, 0.785, 0.545, 0.00},     // 4 waves of 64 x 64
    {128, 128, 1, 512, 1.73, 0.864, 0.521, 0.00},     // the same with K steps of 32
    {64, 64, 4, 512, 2.97, 1.088, 1.066, 1.67},       // gemm_flex.hpp, K dealt to 4 waves
    {64, 64, 2, 1024, 1.12, 0.981, 0.459, 4.73},      // ... to 2 waves, for many tiles or a short K
    {32, 64, 4, 768, 2.34, 0.697, 0.879, 0.79},
    {32, 32, 4, 512, 0.65, 0.514, 0.663, 1.77},
    {64, 128, 1, 256, 2.89, 0.284, 0.411, 3.70},      // ring of K steps
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
// The pass that adds the partial sums of `slices` slices.  (Fitted before it had all its loads in flight at once: four slices of
// [1002 x 2048] 8.3 us by this, 10.2 measured then, 8.0 now.)
inline double reduce_us(long long m, long long n, int slices) { return 3.16 + (double)(slices + 1) * m * n * 4.0 / 8.00e6; }

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
    Plan whole, split;   // the best without and with K in slices
    for (int c = 0; c < kKernels; c++) {
        // steps of half the length are for a K they divide and whole steps do not ([2048 x 2048] from K = 2016 in
        // 30-36 us, 35-42 with a bounds-checked last step); a K of one such step is left to the small tiles
        if (c == kTile128Half && (k % 64 != 32 || k == 32)) continue;
        // two groups of waves share a 64-wide K step: no ragged form
        if (c == kTile256x128Groups && k % 64 != 0) continue;
        const double us = kernel_us(c, m, n, k, batch);
        if (us < whole.us) whole = Plan{c, 1, false, 0, us};
        if (!slices_allowed || batch != 1) continue;
        for (int s = 2; s <= 16 && k / s >= 256 && n % 4 == 0 && c != kTile128Half; s *= 2) {
            const long long per = slice_length(k, s);
            const int slices = (int)ceil_div(k, per);
            if (slices < 2 || (c == kTile256x128Groups && per * s != k)) break;
            const double t = kernel_us(c, m, n, per, slices) + reduce_us(m, n, slices);
            if (t < split.us) split = Plan{c, slices, false, 0, t};
        }
        if (c > kTile256x128) continue;
        const double t = pair_us(c, m, n, k);
        if (t < split.us) split = Plan{c, 1, true, 0, t};
    }
    // slices have to win clearly over none: they take a second launch or an exchange of partial tiles
    Plan best = split.us < 0.97 * whole.us ? split : whole;
    const long long tail = batch == 1 ? column_tail(m, n, k, best.us) : 0;
    if (tail > 0) best = Plan{kTile256, 1, false, tail, best.us};
    return best;
}

// The fastest of the kernels that address C in 64 bits.
inline int flex_kernel(long long m, long long n, long long k, long long batch) {
    int best = kFlex64;
    for (int c = kFlex64; c < kKernels; c++)
        if (kernel_us(c, m, n, k, batch) < kernel_us(best, m, n, k, batch)) best = c;
    return best;
}

// fp32 products (gemm_flex.hpp): us = start + steps * max(step, load * workgroups of a CU) + merge * workgroups of a CU, a step
// being 32 k-values of a wave; a CU that holds one workgroup more than the others sets the time.  Fitted to 80 products of 16 to
// 4096 rows, each on every tile (median error 4-6 %; operands were split as they are then, which took 3-7 % less on every tile).
// Choosing by it, 142 other products, 40 of them loaded value by value, take 3686 us, the best of the measurements 3633.
struct Fp32Cost {
    double start, step, load, merge;
};
constexpr Fp32Cost kFp32Cost64{4.21, 1.542, 1.341, 1.62}, kFp32Cost32x64{3.83, 0.83, 0.796, 0.61}, kFp32Cost32{3.38, 0.60, 0.509, 0.27};
// Waves that walk along K.  Where a CU has at most one workgroup of the small tiles they are eight, two to a SIMD.  Four / eight, us:
// 32 x 32 tiles, [200 x 768] from 512 7.6 / 6.7, [64 x 2048] from 8192 49 / 37, value by value [31 x 1025] from 1025 12.1 / 9.2;
// 32 x 64 tiles, [500 x 520] from 512 8.6 / 7.5, 1024 11.8 / 10.7, 2048 20.7 / 16.6, 8192 69.5 / 56.3, [512 x 1024], a workgroup to
// each CU, 9.4 / 8.8, 13.8 / 12.9, 23.5 / 20.0, 76.5 / 69.9, value by value [333 x 1025] from 1025 17.7 / 13.3.  Below 512 a wave of
// eight has one step or two; with more tiles than CUs eight are 5-40 % slower.  (The price of 32 x 64 tiles is that of four: no choice among 142
// products would be another with eight at 0.8 to 1 of it.)
constexpr long long kFp32EightWaves = 512;
inline int fp32_waves(int kernel, long long m, long long n, long long k, long long batch) {
    if (kernel != kFlex32 && kernel != kFlex32x64) return 4;
    return k >= kFp32EightWaves && ceil_div(m, kCost[kernel].bm) * ceil_div(n, kCost[kernel].bn) * batch <= 256 ? 8 : 4;
}
inline double fp32_us(int kernel, long long m, long long n, long long k, long long batch) {
    const KernelCost& c = kCost[kernel];
    const Fp32Cost& f = kernel == kFlex64 ? kFp32Cost64 : kernel == kFlex32x64 ? kFp32Cost32x64 : kFp32Cost32;
    const double per_cu = (double)(ceil_div(m, c.bm) * ceil_div(n, c.bn) * batch) / 256.0;
    const double step = kernel == kFlex32 && fp32_waves(kernel, m, n, k, batch) == 8 ? 0.51 : f.step;
    const double load = f.load * (per_cu < 4.0 ? ceil(per_cu) : per_cu);
    return f.start + (double)ceil_div(ceil_div(k, 32), 4) * (load > step ? load : step) + f.merge * per_cu;
}
inline int fp32_kernel(long long m, long long n, long long k, long long batch) {
    int best = kFlex64;
    for (int c : {kFlex32x64, kFlex32})
        if (fp32_us(c, m, n, k, batch) < fp32_us(best, m, n, k, batch)) best = c;
    // kTile128: 128 x 128 tiles of four waves (gemm.hip), three to a CU.  From a K of little more than 64 the small tiles pay for
    // four waves' steps and multiply with two and a bit; many whole tiles then go faster by rounds of these: [512 x 512], 128
    // products from K = 65 89.5 us against 94.4, 48 from 72 33.1 against 34.9; from 96, 64 products, 65.3 against 45.3.
    const long long tiles = m / 128 * (n / 128) * batch;
    if (k > 64 && k <= 80 && m % 128 == 0 && n % 128 == 0 && 30.0 * (double)ceil_div(tiles, 768) < 1.0 + 0.0447 * (double)tiles)
        return kTile128;
    return best;
}

// Two products as one launch of small tiles (gemm_pair.hpp): the tile, or -1 where they run one after the other.
//
//   us = start + max(longest walk * step, sum over both of workgroups * (steps + merge) * load / 256)
//
// fitted to 124 pairs (linear layers of 256 .. 3072 features and 19 .. 953 tokens, attention heads of 16 .. 512 tokens),
// each on every tile and as two launches; median error 3-7 %.  By the rule all of them together take 0.74 of the time of
// two launches, by the best of the measurements too; the longest that gained was one of 27 us in two launches (18.3 in
// one: 885 tokens, 640 -> 2560 in fp16), from 30 us on large tiles win ([1024 x 4096] from 622 tokens 28.3 in two, 29.7).
struct PairCost {
    double start, step, load, merge;
};
constexpr int kPairKernels[3] = {kFlex64, kFlex32x64, kFlex32};
constexpr PairCost kPairCost16[3] = {{4.29, 0.884, 0.757, 1.80}, {3.47, 0.722, 0.596, 0.79}, {3.02, 0.542, 0.433, 1.47}};
constexpr PairCost kPairCost32[3] = {{4.94, 1.637, 1.504, 1.10}, {4.24, 0.961, 0.867, 0.75}, {3.81, 0.655, 0.523, 0.28}};
struct PairSizes {
    long long m, n, k, batch;
};
// Two 16-bit products as one launch of gemm_wide_pair_kernel: 128 x 128 tiles for the weight gradient `w`, 32 x 32 tiles whose K
// is dealt to eight waves for the other.  Fitted to 193 linear layers of 16 to 700 tokens and
// 256 to 8192 features (median error 7 %).  Taken where it beats everything else by these costs by 5 %, all of them together take
// 2383 us instead of 2591, by the better of both each time 2360: from some 512 x 1536 features on and up to some 300 tokens
// (16 tokens 4096 -> 1024 15.0 -> 9.3 us, 78 tokens 1024 -> 4096 16.0 -> 13.1, 200 tokens 512 -> 2048 9.2 -> 7.7; but 200 tokens
// 512 -> 512 4.5, and 6.7 so).
inline double wide_pair_us(const PairSizes& w, const PairSizes& x) {
    const double nw = (double)(ceil_div(w.m, 128) * ceil_div(w.n, 128)), nx = (double)(ceil_div(x.m, 32) * ceil_div(x.n, 32));
    const double steps_w = (double)ceil_div(w.k, 64), steps_x = (double)ceil_div(ceil_div(x.k, 64), 8);
    const double walk_w = steps_w * 0.772, walk_x = steps_x * 0.803, longest = walk_w > walk_x ? walk_w : walk_x;
    const double all = (nx * (steps_x + 1.627) * 0.815 + nw * (steps_w + 8.0) * 0.385) / 256.0;
    const double us = 3.9 + (all > longest ? all : longest);
    const double memory = 3.0 + ((double)w.m * w.n * 4.0 + (double)x.k * x.n * 2.0 + 2.0 * (double)x.m * (x.n + x.k)) / 4.5e6;
    return us > memory ? us : memory;
}
#ifndef BR_PAIR_FORCE
#define BR_PAIR_FORCE -1   // a kernel: every pair of products on it, for measuring
#endif
// `w`: the product whose operands are both row-contiguous, which alone can have the wide tiles.
inline int pair_kernel(const PairSizes& w, const PairSizes& x, bool fp32) {
    if (BR_PAIR_FORCE >= 0) return BR_PAIR_FORCE;
    double us = 0.0;   // one after the other
    for (const PairSizes* s : {&w, &x}) {
        if (fp32) {
            const int kernel = fp32_kernel(s->m, s->n, s->k, s->batch);
            if (kernel == kTile128) return -1;
            us += fp32_us(kernel, s->m, s->n, s->k, s->batch);
        } else {
            us += gemm_plan(s->m, s->n, s->k, s->batch, true).us;
        }
    }
    int best = -1;
    double best_us = 1e30;
    for (int i = 0; i < 3; i++) {
        const KernelCost& tile = kCost[kPairKernels[i]];
        const PairCost& c = fp32 ? kPairCost32[i] : kPairCost16[i];
        double longest = 0.0, all = 0.0, fewest = 1e30;
        for (const PairSizes* s : {&w, &x}) {
            const double groups = (double)(ceil_div(s->m, tile.bm) * ceil_div(s->n, tile.bn) * s->batch);
            const double steps = (double)ceil_div(ceil_div(s->k, fp32 ? 32 : 64), tile.k_waves);
            if (steps * c.step > longest) longest = steps * c.step;
            if (groups < fewest) fewest = groups;
            all += groups * (steps + c.merge) * c.load / 256.0;
        }
        const double t = c.start + (all > longest ? all : longest);
        // A hurdle for the close ones: [1024 x 4096] from 74 tokens 14.3 in two launches, 14.8 in one.  fp32: two launches
        // take more than these costs say where the tiles are small or both products fill the chip (1000 tokens, 2048 -> 2048 on
        // 64 x 64 tiles 106 us in one launch, 113 in two).  Over 79 pairs (16 to 1000 tokens of 256 to 6144 features, attention
        // heads of 16 to 512) 2313 us by the rule, 2271 by the best of the measurements, 3187 when matrix instructions of fp32
        // operands did the products.
        const int tile_of = kPairKernels[i];
        const double hurdle = !fp32 ? 0.97 : tile_of == kFlex32 ? 1.05 : tile_of == kFlex32x64 ? 0.98 : fewest >= 256.0 ? 1.1 : 0.95;
        if (t < hurdle * us && t < best_us) best = kPairKernels[i], best_us = t;
    }
    if (!fp32 && w.batch == 1 && x.batch == 1 && wide_pair_us(w, x) < 0.95 * (best_us < us ? best_us : us)) best = kPairWide;
    return best;
}

}  // namespace gemm16
}  // namespace brk
