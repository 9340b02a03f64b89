// How the tiled kernels run a call: pure host functions of the sizes, plain C++.  A plan is made
// once per call and handed as it is to the argument checks, the scratch sizes and the launch.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace uniql {

static inline int ceil_div_i(int a, int b) { return (a + b - 1) / b; }

// One launch of the 128-column kernel.
struct TilePlan {
    int mtiles;    // 32-row M tiles per workgroup
    int splits;    // workgroups that share a tile's K groups
    int gps;       // K groups per workgroup (the last split may have fewer)
    int quartets;  // wave quartets per workgroup (1 or 2); two take alternate groups, every range is even then
    double us;     // expected time
};

// The K values whose products enter one accumulator one after another: a wave takes 32 of a group's 128, a quartet its
// share of the groups.
static inline int tile_chain(const TilePlan& plan) { return 32 * ceil_div_i(plan.gps, plan.quartets); }

// What a plan that splits K over workgroups needs: one arrival count per output tile in `accum` (zero on entry,
// zero again on exit) and one fp32 partial tile per (tile, split) in a scratch area whose contents do not matter.
static inline size_t tile_accum_bytes(int m, int n, const TilePlan& plan) {
    return plan.splits <= 1 ? 0 : (size_t)(n / 128) * ceil_div_i(m, 32 * plan.mtiles) * sizeof(unsigned long long);
}
static inline size_t tile_part_bytes(int m, int n, const TilePlan& plan) {
    if (plan.splits <= 1) return 0;
    return (size_t)(n / 128) * ceil_div_i(m, 32 * plan.mtiles) * plan.splits * (32 * plan.mtiles * 128) * sizeof(float);
}

// Time in us of a launch of `wgs` workgroups that walk `g` K groups each, on 256 compute units.  Workgroups run in
// rounds: one per compute unit with two quartets, 96-, 128-row and 256 x 256 tiles (LDS), two with 64-row tiles, four with
// 32-row tiles.  A launch costs a constant (prologue, epilogue, start) and a time per K group, which steps with the number of
// workgroups on the fullest compute unit and grows with the busy part of the chip inside a step (the clock falls with the matrix load).
// Fitted to 6250 drawn layer calls (N 256 to 28672, K 256 to 14336, 17 to 4096 rows, plain, cut, gated and with a residual), each
// with every plan inside 1.5 x of the best: half of the times are within 3.5 % of these, nine in ten within 12 %.  What
// is off is mostly the epilogue, which a plan must not depend on (a layer's sum is the same with and without a residual):
// adding one costs the tall tiles 4 to 8 us a round.  Of another 6250 calls the plan with the smallest time here took 1.003 x
// the best plan's time on average.
// The exchange of 64- (one quartet), 96- and 128-row tiles since its slots are read in batches: of 300 drawn calls of 65 to 700
// rows whose plan that changed (96-row tiles with 2 to 7 splits in place of shorter ones, mostly) 284 are no slower, 12 % faster on
// average (14336 -> 6144 at 84 rows 35.6 -> 27.9 us, 12160 -> 4096 at 66 27.2 -> 21.4, 4096 -> 11264 at 96 20.8 -> 19.3; calls with more
// rows than columns: tile_us).  Kept above what is measured (1 us for two splits,
// 2 for eight) for 64-row tiles, so that one quartet does not replace two, whose sums are half as long chains, and as it was for
// 32-row tiles, up to 64 rows the other kernel's rivals.
struct LaunchFit {
    double full, full_g;        // a whole round: constant, per K group
    double split, split_each;   // the exchange between K splits (partial tiles' stores, count, the last one's reading of all of them)
    double after;               // what is left behind whole rounds, a constant
    int levels;                 // workgroups per compute unit and round
    struct {                    // i + 1 workgroups on the fullest unit in what is left:
        double alone;           //   its constant if that is the whole launch
        double behind;          //   factor on the times per group behind whole rounds
        double g[3];            //   time per K group with the level nearly empty, half full, full
    } level[4];
};
static const LaunchFit kLaunchFits[7] = {
    {8.65, 1.351, 0.537, 0.77, 4.03, 4, {{5.34, 0.814, 0.391, 0.355, 0.404}, {5.78, 1.127, 0.581, 0.639, 0.715},
     {6.82, 1.054, 1.019, 1.032, 1.138}, {8.86, 1.117, 1.304, 1.379, 1.453}}},  // 32 rows, one quartet
    {5.29, 0.35, 0.763, 0.547, 5.46, 1, {{5.46, 1.0, 0.279, 0.282, 0.339}}},  // 32 rows, two quartets
    {5.59, 1.001, 1.6, 0.85, 5.58, 2, {{6.82, 0.989, 0.447, 0.452, 0.577}, {7.16, 1.085, 0.8, 0.938, 1.074}}},  // 64 rows, one quartet
    {7.46, 0.521, 0.852, 0.935, 7.15, 1, {{7.15, 1.0, 0.365, 0.381, 0.498}}},  // 64 rows, two quartets
    {6.97, 0.74, 2.3, 0.79, 4.67, 1, {{6.35, 1.083, 0.478, 0.604, 0.743}}},  // 96 rows
    {5.98, 0.95, 1.877, 1.2, 7.49, 1, {{8.94, 1.043, 0.493, 0.692, 0.9}}},  // 128 rows
    {7.65, 3.39, 0.0, 0.0, 4.41, 1, {{13.28, 1.095, 2.15, 2.64, 3.29}}},  // 256 x 256
};
static inline double launch_us(const LaunchFit& f, int64_t wgs, int g, int splits) {
    const int64_t per_round = 256 * (int64_t)f.levels, full = wgs / per_round, rest = wgs % per_round;
    double us = (double)full * (f.full + f.full_g * g) + (splits > 1 ? f.split + f.split_each * splits : 0.0);
    if (rest == 0) return us;
    const auto& l = f.level[(rest - 1) / 256];
    const double x = (double)((rest - 1) % 256 + 1) / 128.0;   // 0 to 2 inside the level
    const double per_g = x < 1.0 ? l.g[0] + (l.g[1] - l.g[0]) * x : l.g[1] + (l.g[2] - l.g[1]) * (x - 1.0);
    return us + (full > 0 ? f.after + l.behind * per_g * g : l.alone + per_g * g);
}
static inline int fit_index(int mt, int quartets) { return mt <= 2 ? 2 * (mt - 1) + (quartets - 1) : mt + 1; }
// What the exchange cost more before its slots were read in batches, and in two places still counts for.
static inline double former_exchange_us(int mt, int quartets, int splits) {
    if (splits <= 1 || quartets == 2 || mt < 2) return 0.0;
    return mt == 2 ? -0.091 + 0.262 * splits : mt == 3 ? 0.58 + 1.068 * splits : 1.48 * splits;
}
// With at least as many rows as columns (activations of four times the weights' bytes and more) taller tiles with more splits are
// no gain: of 438 drawn calls of 33 to 4096 rows whose plan the lower ratings change, the 293 with fewer rows than columns are
// 1.07 x as fast and 16 of them slower by more than 5 %, of the 145 others, 1.00 x as fast, 38 are, by up to a third (10624 -> 384 at
// 1563 rows 24.4 -> 32.9 us, 6784 -> 768 at 1326 24.1 -> 31.5, 7424 -> 512 at 3025 32.9 -> 42.6).
static inline double tile_us(int mt, int quartets, int m, int n, int64_t wgs, int g, int splits) {
    return launch_us(kLaunchFits[fit_index(mt, quartets)], wgs, g, splits) + (m >= n ? former_exchange_us(mt, quartets, splits) : 0.0);
}
// us by which a launch with K split has to be faster than one whose sums are shorter chains of products to be taken in its
// place: sums get no longer, and so no further from exact ones, for a gain of a few per cent (10752 -> 2048 at 459 rows, chains
// of 896 in place of 672: 34.9 us against 35.7; 12672 -> 3968 at 3558, of 12672 in place of 3168: 328 against 356).
static inline double longer_chain_us(int m, int n, const TilePlan& p) {
    return m >= n ? 0.0 : former_exchange_us(p.mtiles, p.quartets, p.splits);  // there it is part of the plan's time
}
static inline double wide_us(int m, int n, int k) {
    return launch_us(kLaunchFits[6], (int64_t)(n / 256) * ((m + 255) / 256), k / 128, 1);
}

// Height of the tiles, K splits and quartets with the smallest expected time.  K is split over workgroups while the
// grid stays within one workgroup per compute unit, every workgroup keeps at least 8 groups and the
// partial tiles fit part_cap bytes.  Two quartets are rated where the grid has at most 256 workgroups of at most 64 rows
// and every workgroup can get an even number of groups.  Overrides: 0 = choose.
// The 96-row tiles are there for the rounds: 14336 -> 4096 at 333 rows runs as 256 workgroups of them in 51.3 us
// (128 rows: 54.1, 64 rows: 54.5, the plan of rule_launch: 57-63), 4096 -> 24576 at 333 rows as three
// whole rounds (87.0 against 93.3).
static inline TilePlan tile_plan(int m, int n, int k, int splits_override, int mt_override, int kw_override, size_t part_cap) {
    TilePlan best = {4, 1, k / 128, 1, 1e30};
    const int strips = n / 128, G = k / 128;
    for (int mt = 1; mt <= 4; ++mt) {
        if (mt_override >= 1 && mt_override <= 4 && mt != mt_override) continue;
        const int64_t tiles = (int64_t)strips * ceil_div_i(m, 32 * mt);
        for (int s = 1; s <= 255; ++s) {
            if (splits_override > 0) s = splits_override;
            else if (s > 1 && (tiles * s > 256 || G / s < 8)) break;
            const int gps1 = ceil_div_i(G, s > G ? G : s), splits = ceil_div_i(G, gps1);
            // two quartets take alternate groups: every workgroup's range must hold an even number
            const int gps2 = gps1 + (gps1 & 1);
            const bool two_ok = mt <= 2 && G % 2 == 0 && ceil_div_i(G, gps2) == splits && (kw_override == 2 || tiles * splits <= 256);
            for (int kw = 1; kw <= 2; ++kw) {
                if (kw == 2 ? !two_ok || (kw_override & 1) : two_ok && kw_override == 2) continue;
                TilePlan p = {mt, splits, kw == 2 ? gps2 : gps1, kw, 0.0};
                p.us = tile_us(mt, kw, m, n, tiles * splits, p.gps, splits);
                const bool fits = splits == 1 || splits_override > 0 || tile_part_bytes(m, n, p) <= part_cap;
                if (fits && p.us < best.us) best = p;
            }
            if (splits_override > 0) break;
        }
    }
    return best;
}

// How the tiled kernels run a call: one launch, or two over consecutive rows or columns.
struct RowPart {
    int rows;
    bool wide;      // the 256 x 256 kernel; `tile` then only carries the expected time
    TilePlan tile;
};
struct LinearPlan {
    int parts;
    RowPart part[2];
    int head_columns;  // 0: two parts are consecutive rows; else all rows, the first of them over so many columns
};
static inline int part_columns(const LinearPlan& plan, int i, int n) {
    return plan.head_columns == 0 ? n : (i == 0 ? plan.head_columns : n - plan.head_columns);
}

// The plan for m rows in one launch by the order of the tile heights alone.  In
// units of the time one 128-row workgroup takes for its K loop when every compute unit has one: 128 rows 1 per started
// round of 256; 64 rows 1.08 per round of 512 (every weight is expanded twice per 128 rows), 0.85 for a last round of at most
// 256; 32 rows 0.62 for at most 256 workgroups, 0.88 for at most 512, 1.62 per started round of 1024; two quartets, at most
// one workgroup per compute unit, 0.85 and 0.92 of it.  A long K loop over few 64-row tiles prefers those with K split (every weight
// is expanded for twice the rows).  K splits double while the grid stays within one workgroup per compute unit, every
// workgroup keeps at least 8 groups and the partial tiles stay below a quarter of the packed weights.  The 256 x 256
// kernel wherever the real output fills at least 0.62 of the tile slots of its rounds of 256 workgroups.
static inline RowPart rule_launch(int m, int n, int k, bool wide_ok) {
    const int64_t wide_rounds = ((int64_t)(n / 256) * ((m + 255) / 256) + 255) / 256;
    if (wide_ok && (double)m * n / 65536.0 >= 0.62 * 256.0 * (double)wide_rounds)
        return RowPart{m, true, TilePlan{0, 1, k / 128, 1, wide_us(m, n, k)}};
    const int strips = n / 128, G = k / 128;
    const bool even_g = G % 2 == 0;
    const int64_t t4 = (int64_t)strips * ceil_div_i(m, 128), t2 = (int64_t)strips * ceil_div_i(m, 64);
    const int64_t t1 = (int64_t)strips * ceil_div_i(m, 32), rest2 = t2 % 512;
    const double cost4 = (double)((t4 + 255) / 256);
    const double cost2 = (1.08 * (double)(t2 / 512) + (rest2 == 0 ? 0.0 : (rest2 <= 256 ? 0.85 : 1.08))) * (even_g && t2 <= 256 ? 0.92 : 1.0);
    const double cost1 = (t1 <= 256 ? 0.62 : (t1 <= 512 ? 0.88 : 1.62 * (double)((t1 + 1023) / 1024))) * (even_g && t1 <= 256 ? 0.85 : 1.0);
    TilePlan p;
    p.mtiles = m <= 32 ? 1 : (cost2 < cost4 && cost2 <= cost1 ? 2 : (cost1 < cost4 ? 1 : 4));
    if (p.mtiles == 1 && G >= 64 && m >= 64 && t2 <= 128) p.mtiles = 2;
    const int64_t tiles = (int64_t)strips * ceil_div_i(m, 32 * p.mtiles);
    int splits = 1;
    while (tiles * (2 * splits) <= 256 && G / (2 * splits) >= 8 && (int64_t)(2 * splits) * m * 16 <= k) splits *= 2;
    p.gps = ceil_div_i(G, splits);
    p.quartets = even_g && p.mtiles <= 2 && tiles * ceil_div_i(G, p.gps) <= 256 ? 2 : 1;
    if (p.quartets == 2) p.gps += p.gps & 1;
    p.splits = ceil_div_i(G, p.gps);
    p.us = tile_us(p.mtiles, p.quartets, m, n, tiles * p.splits, p.gps, p.splits);
    return RowPart{m, false, p};
}

// Whether all workgroups of a launch of the 128-column kernel are on the chip at once.
static inline bool one_round(int m, int n, const TilePlan& p) {
    return (int64_t)(n / 128) * ceil_div_i(m, 32 * p.mtiles) * p.splits <= 256 * (int64_t)kLaunchFits[fit_index(p.mtiles, p.quartets)].levels;
}

// One launch for m rows: what the search expects to be fastest, if that beats the rule's plan by 2 %.  Between two launches
// of one round each, whose expected times are the most exact, any gain is enough.  Of 6250 calls the search alone is 1.7 %
// faster than the rule and slower by more than 2 % in 113; with these margins it is 1.7 % faster and slower in 31.
static inline RowPart best_launch(int m, int n, int k, bool wide_ok, size_t part_cap) {
    const RowPart rule = rule_launch(m, n, k, wide_ok);
    RowPart p = {m, false, tile_plan(m, n, k, 0, 0, 0, part_cap)};
    if (p.tile.mtiles >= 3 && p.tile.splits > 1) {
        const TilePlan shorter = tile_plan(m, n, k, 0, 2, 2, part_cap);
        if (tile_chain(shorter) < tile_chain(p.tile) && shorter.us <= p.tile.us + longer_chain_us(m, n, p.tile)) p.tile = shorter;
    }
    const double wide = wide_ok ? wide_us(m, n, k) : p.tile.us;
    if (wide < p.tile.us) {
        p.wide = true;
        p.tile.us = wide;
    }
    if (!rule.wide && tile_part_bytes(m, n, rule.tile) > part_cap) return p;
    const bool exact = !p.wide && !rule.wide && one_round(m, n, p.tile) && one_round(m, n, rule.tile);
    return p.tile.us < (exact ? 1.0 : 0.98) * rule.tile.us ? p : rule;
}

// wide_ok: the 256 x 256 kernel can take the call.  part_cap: the most bytes of partial tiles a plan may ask for.
// tune: fields of a plan asked for by the caller (bits 0..7 K splits, 8..11 32-row M tiles per workgroup, 8 there for the
// 256 x 256 kernel, 12..13 wave quartets; 0 = choose), followed as far as the kernels can.
// A last round of workgroups that leaves most of the chip idle costs as much as a full one, so the rows behind the
// last 128-row boundaries are also tried as a launch of their own (shorter tiles, K split): 4096 -> 28672 at 1100
// rows is 1024 on the 256 x 256 kernel and 76 on 96-row tiles, 240 us instead of 297 in one launch.
// Up to 128 rows there is nothing to split.  The 2 us: two launches of different kernels take that much longer than each
// behind its like (4096 -> 28672 at 200 rows: 69.5 us, 65.1 expected of 128 and 72 rows alone); the 2 %: what the expected times may be
// off together.
static inline LinearPlan linear_plan(int m, int n, int k, bool wide_ok, size_t part_cap, unsigned tune) {
    LinearPlan plan;
    plan.parts = 1;
    plan.head_columns = 0;
    if ((tune & 0x3fffu) != 0) {
        const int rows = (int)((tune >> 8) & 0xfu);
        plan.part[0] = RowPart{m, rows == 8 && wide_ok,
                               tile_plan(m, n, k, (int)(tune & 0xffu), rows, (int)((tune >> 12) & 0x3u), (size_t)-1)};
        return plan;
    }
    plan.part[0] = best_launch(m, n, k, wide_ok, part_cap);
    double us = plan.part[0].tile.us;
    int j = (m - 1) / 128;
    for (int tries = 0; j > 0 && tries < 8; --j, ++tries) {
        const RowPart head = best_launch(128 * j, n, k, wide_ok, part_cap);
        if (head.tile.us + 2.0 >= us) continue;
        const RowPart tail = best_launch(m - 128 * j, n, k, wide_ok, part_cap);
        const double both = head.tile.us + tail.tile.us + 2.0 + (head.wide && !plan.part[0].wide ? longer_chain_us(m - 128 * j, n, tail.tile) : 0.0);
        if (both < 0.98 * us) {
            us = both / 0.98;
            plan.parts = 2;
            plan.part[0] = head;
            plan.part[1] = tail;
        }
    }
    return plan;
}

// The same with the columns in two launches, where that is expected to be faster by a margin: first as many as fill whole
// rounds of the 256 x 256 kernel or of 128-row tiles, then the rest on whatever suits it.  4096 -> 18688 at 1024 rows is 292
// of the large tiles, 36 more than a round: 256 of them over 16384 columns and 96-row tiles over the other 2304 take 145 us
// (768 rows of large tiles, then 256 rows of 64-row ones: 161).  Of 1100 drawn calls
// of more than 64 rows 110 run so, 0.99 to 1.35 x as fast, 1.11 on average; with a margin of 3 % in place of 5 one in ten
// of them was up to 2 % slower.  wide_ok: whether the 256 x 256 kernel can take the largest multiple of 256 columns;
// n itself may be an odd number of strips (2048 -> 21376 at 2997 rows 326 -> 247).  Up to 64 rows the columns are one launch.
static inline LinearPlan call_plan(int m, int n, int k, bool wide_ok, size_t part_cap, unsigned tune) {
    LinearPlan plan = linear_plan(m, n, k, wide_ok && n % 256 == 0, part_cap, tune);
    if ((tune & 0x3fffu) != 0 || m <= 64) return plan;
    double us = plan.part[0].tile.us + (plan.parts == 2 ? plan.part[1].tile.us + 2.0 : 0.0);
    const int wide_rows = (m + 255) / 256, tall_rows = (m + 127) / 128;
    const int wide_columns = 256 * (int)((int64_t)wide_rows * (n / 256) / 256 * 256 / wide_rows);
    const int tall_columns = 128 * (int)((int64_t)tall_rows * (n / 128) / 256 * 256 / tall_rows);
    // One launch of large tiles whose last round is a third full and more ends sooner than expected (its workgroups
    // start as the compute units become free, at a higher clock: 4096 -> 6144 at 4096 rows 189 us, 213 expected, 192 in two).
    const int rest = (int)((int64_t)wide_rows * (n / 256) % 256);
    const double gain = plan.parts == 1 && plan.part[0].wide && rest >= 96 ? 0.88 : 0.95;
    const int columns[3] = {wide_ok ? wide_columns : 0, tall_columns, wide_ok && n % 256 != 0 ? n - 128 : 0};
    for (int i = 0; i < 3; ++i) {
        const int c = columns[i];
        if (c <= 0 || c >= n) continue;
        const RowPart head = best_launch(m, c, k, wide_ok && c % 256 == 0, part_cap);
        if (head.tile.us + 2.0 >= us) continue;
        const RowPart tail = best_launch(m, n - c, k, wide_ok && (n - c) % 256 == 0, part_cap);
        const double both = head.tile.us + tail.tile.us + 2.0 + (head.wide && !plan.part[0].wide ? longer_chain_us(m, n - c, tail.tile) : 0.0);
        if (both < gain * us) {
            us = both / gain;
            plan.parts = 2;
            plan.part[0] = head;
            plan.part[1] = tail;
            plan.head_columns = c;
        }
    }
    return plan;
}
static inline size_t plan_accum_bytes(const LinearPlan& plan, int n) {
    size_t most = 0;
    for (int i = 0; i < plan.parts; ++i) {
        const size_t b = plan.part[i].wide ? 0 : tile_accum_bytes(plan.part[i].rows, part_columns(plan, i, n), plan.part[i].tile);
        most = b > most ? b : most;
    }
    return most;
}
static inline size_t plan_part_bytes(const LinearPlan& plan, int n) {
    size_t most = 0;
    for (int i = 0; i < plan.parts; ++i) {
        const size_t b = plan.part[i].wide ? 0 : tile_part_bytes(plan.part[i].rows, part_columns(plan, i, n), plan.part[i].tile);
        most = b > most ? b : most;
    }
    return most;
}

}  // namespace uniql
