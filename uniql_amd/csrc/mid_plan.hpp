// How the kernel for 9 to 64 rows runs a call: plain host functions of the sizes.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace uniql {

constexpr int kMidMinRows = 9, kMidMaxRows = 64;

struct MidPlan {
    int upw;     // groups of 128 K per wave; 0: the call does not take this kernel
    int waves;   // waves per workgroup
    int splits;  // workgroups along K per strip of 128 columns
    double us;   // expected time
};

// A lane offset behind every descriptor of this kernel, also where the bounds check adds or subtracts a scalar offset.
constexpr uint32_t kMidNoLoad = 0x80000000u;
// Bytes of X from column 128 g of its first row to the end of its last row; none for a unit that does not exist.
constexpr uint32_t mid_x_records(uint32_t x_bytes, int g, bool real) {
    return real && x_bytes > 256u * (uint32_t)g ? x_bytes - 256u * (uint32_t)g : 0u;
}
// Bytes of a group's eight packed rows over all columns.
constexpr int64_t mid_group_bytes(int n) { return 64 * (int64_t)n; }

static inline int mid_row_tiles(int m) { return m <= 16 ? 1 : m <= 32 ? 2 : m <= 48 ? 3 : 4; }  // of 16 rows

// Accumulators of a wave: the products of the low and of the high codes apart (SETS = 2) wherever the registers hold both
// and a wave has more than one unit or nothing to lose: with 33 to 48 rows and one unit a wave the second set costs 0.7 us
// of 9.4 (its zeros, its moves to vector registers), with 49 to 64 rows it does not fit.
static inline int mid_sets(int m, int upw) {
    const int tiles = mid_row_tiles(m);
    return tiles <= 2 || (tiles == 3 && upw > 1) ? 2 : 1;
}
// The K values whose products enter one accumulator one after another: what a sum's error grows with (the matrix unit
// rounds each of its additions; the waves' and workgroups' sums meet in a few levels).
static inline int mid_chain(int m, int upw) { return 128 * upw / mid_sets(m, upw); }

// What a plan that splits K over workgroups needs: an arrival count per strip and wave in `accum` (zero on entry and
// exit), the partial tiles in units of four rows, a whole number per wave, in a scratch area whose contents do not matter.
static inline size_t mid_accum_bytes(int n, const MidPlan& p) { return p.splits <= 1 ? 0 : (size_t)(n / 128) * p.waves * sizeof(unsigned long long); }
static inline size_t mid_part_bytes(int m, int n, const MidPlan& p) {
    const int units = 4 * mid_row_tiles(m), whole = (units + p.waves - 1) / p.waves * p.waves;
    return p.splits <= 1 ? 0 : (size_t)(n / 128) * p.splits * whole * (4 * 128 * sizeof(float));
}

// Time in us of a launch, one workgroup per compute unit at a time: a constant, per started round a constant and a time
// per unit, both growing with the busy part of the chip, and the exchange between K splits.  Fitted for each row class to
// about 1450 drawn layer calls (N 256 to 28672, K 256 to 14336) with every plan timed: half of the times are within 3 to 6 %
// of these, and the plan with the smallest one takes 1.002 to 1.005 x the best plan's time on average.
struct MidFit {
    double constant, round_g, round, split, split_each, busy_g, busy;
};
static const MidFit kMidFits[4] = {
    {1.09, 2.129, 1.047, 0.863, 0.365, 0.391, 1.095},   // 16 rows
    {0.157, 2.477, 2.086, 1.099, 0.325, 0.38, 2.494},   // 32 rows
    {1.573, 1.639, 2.235, 0.741, 0.354, 0.123, 2.42},   // 48 rows
    {2.517, 1.935, 1.677, 0.928, 0.341, 0.122, 3.391},  // 64 rows
};
static inline double mid_us(int m, int64_t wgs, int upw, int splits) {
    const MidFit& f = kMidFits[mid_row_tiles(m) - 1];
    const double rounds = (double)((wgs + 255) / 256), busy = wgs < 256 ? (double)wgs / 256.0 : 1.0;
    return f.constant + rounds * (f.round + f.round_g * upw) + busy * f.busy_g * upw + f.busy * busy +
           (splits > 1 ? f.split + f.split_each * splits : 0.0);
}

// Eight waves, two a SIMD, up to 32 rows (4096 -> 4096 at 17 rows 8.2 us against 8.8 with four), four from 33 rows on
// (4096 -> 4096 at 48 rows 10.1 against 10.5: eight have no registers there to load a unit ahead).
// longest_chain: plans whose sums take an eighth more than so many K values one after another do not count (0: all do).
// The eighth: at equal chains the sums are 2 to 4 % closer here, since the waves' and workgroups' sums meet in pairs.
static inline MidPlan mid_plan(int m, int n, int k, int upw_override, size_t part_cap, int longest_chain = 0) {
    const int G = k / 128, waves = m <= 32 ? 8 : 4, longest = (G + waves - 1) / waves;
    MidPlan best = {0, 0, 0, 1e30};
    for (int upw = 1; upw <= longest; ++upw) {
        if (upw_override > 0 && upw != (upw_override < longest ? upw_override : longest)) continue;
        if (longest_chain > 0 && 8 * mid_chain(m, upw) > 9 * longest_chain) continue;
        MidPlan p = {upw, waves, (G + waves * upw - 1) / (waves * upw), 0.0};
        p.us = mid_us(m, (int64_t)(n / 128) * p.splits, upw, p.splits);
        if (mid_part_bytes(m, n, p) <= part_cap && p.us < best.us) best = p;
    }
    return best;
}

}  // namespace uniql
