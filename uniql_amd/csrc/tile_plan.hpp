// How the tiled kernels run the rows of a call: pure host functions of the sizes, plain C++.  A plan is made
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

// What a plan that splits K over workgroups needs: one arrival count per output tile in `accum` (zero on entry,
// zero again on exit) and one fp32 partial tile per (tile, split) in a scratch area whose contents do not matter.
static inline size_t tile_accum_bytes(int m, int n, const TilePlan& plan) {
    return plan.splits <= 1 ? 0 : (size_t)(n / 128) * ceil_div_i(m, 32 * plan.mtiles) * sizeof(unsigned long long);
}
static inline size_t tile_part_bytes(int m, int n, const TilePlan& plan) {
    if (plan.splits <= 1) return 0;
    return (size_t)(n / 128) * ceil_div_i(m, 32 * plan.mtiles) * plan.splits * (32 * plan.mtiles * 128) * sizeof(float);
}

// Time of a launch of `wgs` workgroups that walk `g` K groups each, in us, on 256 compute units.
// Workgroups run in rounds: one per compute unit with 96- and 128-row tiles (LDS) or two quartets, two with
// 64-row tiles, four with 32-row tiles.  A round costs a prologue and an epilogue (6 us) and a time per group that
// grows once more than half of the chip is busy (the clock falls with the matrix load).  Fitted to forced
// launches of nine shapes (K 4096 to 14336, N 4096 to 28672) at 96 to 4096 rows, within 5 % of all but the
// 32-row tiles from 600 workgroups on; e.g. 4096 -> 4096, 256 tiles of 128 rows 35.6 us (model 35.0), of 96 rows 29.7
// (29.4), 14336 -> 4096 106 (104) and 89.8 (87.8).
static inline double ramp(double lo, double hi, int64_t x, int64_t x0, int64_t x1) {
    return x <= x0 ? lo : lo + (hi - lo) * (double)(x - x0) / (double)(x1 - x0);
}
static inline double tile_us(int mt, int quartets, int64_t wgs, int g) {
    const int64_t per_round = quartets == 2 || mt >= 3 ? 256 : (mt == 2 ? 512 : 1024);
    const double full = (double)(wgs / per_round);
    const int64_t rest = wgs % per_round;
    double us = 0.0;
    if (quartets == 2 && mt == 2) {
        us = full * (5.7 + 0.536 * g);
        if (rest) us += 5.7 + g * (rest <= 192 ? ramp(0.375, 0.447, rest, 64, 192) : ramp(0.447, 0.536, rest, 192, 256));
    } else if (quartets == 2) {
        us = full * (3.9 + 0.40 * g) + (rest ? 3.9 + g * ramp(0.30, 0.40, rest, 64, 256) : 0.0);
    } else if (mt == 4) {
        us = full * (6.5 + 0.875 * g) + (rest ? 6.5 + g * ramp(0.60, 0.86, rest, 128, 256) : 0.0);
    } else if (mt == 3) {
        us = full * (6.0 + 0.73 * g) + (rest ? 6.0 + g * ramp(0.53, 0.73, rest, 128, 256) : 0.0);
    } else if (mt == 2) {
        us = full * (6.5 + 1.02 * g);
        if (rest > 256) us += 6.0 + g * ramp(0.75, 1.02, rest, 256, 512);
        else if (rest) us += full > 0 ? 4.0 + g * ramp(0.33, 0.49, rest, 0, 256)  // starts before the round ends
                                  : 5.1 + g * ramp(0.46, 0.55, rest, 128, 256);
    } else {
        us = full * (5.0 + 1.5 * g);
        if (rest > 512) us += 5.0 + g * ramp(0.85, 1.5, rest, 512, 1024);
        else if (rest > 256) us += 5.0 + g * ramp(0.55, 0.75, rest, 256, 512);
        else if (rest) us += full > 0 ? 4.0 + 0.35 * g : 3.1 + g * ramp(0.395, 0.45, rest, 128, 256);
    }
    return us;
}

// What the exchange between the splits of a tile adds: the partial tiles' stores, the count, and the last workgroup's
// reading of all of them (forced splits of 1 to 8 on six shapes at 24 to 192 rows).
static inline double exchange_us(int mt, int splits) {
    if (mt == 1) return 2.2 + 0.08 * splits * splits;
    if (mt == 2) return 3.0 + 0.11 * splits * splits;
    return mt == 3 ? 3.0 + 1.8 * splits : 6.0 + 2.1 * splits;
}

// Height of the tiles, K splits and quartets with the smallest expected time.  K is split over workgroups while the
// grid stays within one workgroup per compute unit, every workgroup keeps at least 8 groups and the
// partial tiles fit part_cap bytes.  Two quartets whenever the grid has at most 256 workgroups of at most 64 rows
// and every workgroup can get an even number of groups.  Overrides: 0 = choose.
// The 96-row tiles are there for the rounds: 14336 -> 4096 at 333 rows runs as 256 workgroups of them in 51.3 us
// (128 rows: 54.1, 64 rows: 54.5, the rule of thumb this search replaced: 57-63), 4096 -> 24576 at 333 rows as three
// whole rounds (87.0 against 93.3).
static inline TilePlan tile_plan(int m, int n, int k, int splits_override, int mt_override, int kw_override, size_t part_cap) {
    TilePlan best = {4, 1, k / 128, 1, 1e30};
    const int strips = n / 128, G = k / 128;
    const bool even_g = G % 2 == 0;
    for (int mt = 1; mt <= 4; ++mt) {
        if (mt_override >= 1 && mt_override <= 4 && mt != mt_override) continue;
        const int64_t tiles = (int64_t)strips * ceil_div_i(m, 32 * mt);
        for (int s = 1; s <= 255; ++s) {
            if (splits_override > 0) s = splits_override;
            else if (s > 1 && (tiles * s > 256 || G / s < 8)) break;
            TilePlan p;
            p.mtiles = mt;
            p.gps = ceil_div_i(G, s > G ? G : s);
            p.splits = ceil_div_i(G, p.gps);
            p.quartets = 1;
            // two quartets take alternate groups: every workgroup's range must hold an even number
            if ((kw_override == 2 || (kw_override == 0 && tiles * p.splits <= 256)) && mt <= 2 && even_g) {
                const int gps2 = p.gps + (p.gps & 1);
                if (splits_override == 0 || ceil_div_i(G, gps2) == p.splits) {
                    p.gps = gps2;
                    p.splits = ceil_div_i(G, p.gps);
                    p.quartets = 2;
                }
            }
            p.us = tile_us(mt, p.quartets, tiles * p.splits, p.gps);
            if (p.splits > 1) p.us += exchange_us(mt, p.splits);
            const bool fits = p.splits == 1 || splits_override > 0 || tile_part_bytes(m, n, p) <= part_cap;
            if (fits && p.us < best.us) best = p;
            if (splits_override > 0) break;
        }
    }
    return best;
}

// Expected time of the 256 x 256 kernel in us (fitted like the 128-column kernel's: forced launches of nine shapes at 96 to
// 4096 rows, within 5 %): rounds of 256 workgroups, the time per K group growing with the busy part of the chip.
static inline double wide_us(int m, int n, int k) {
    const int64_t tiles = (int64_t)(n / 256) * ((m + 255) / 256);
    const int g = k / 128;
    const int64_t rest = tiles % 256;
    const double slow = rest > 120 ? 1.08 * (double)(rest - 120) / 136.0 : 0.0;
    return (double)(tiles / 256) * (9.0 + 3.2 * g) + (rest ? 8.5 + g * (2.12 + slow) : 0.0);
}

// How the tiled kernels run the rows of a call: one launch, or two over consecutive rows.
struct RowPart {
    int rows;
    bool wide;      // the 256 x 256 kernel; `tile` then only carries the expected time
    TilePlan tile;
};
struct LinearPlan {
    int parts;
    RowPart part[2];
};

// The faster of the two kernels for m rows in one launch, by their expected times.  The 4 %: most layer calls cut, add or
// gate their outputs, which the 256 x 256 kernel does at next to no cost and the tall tiles of the other with 3 to 8 %
// (4096 -> 18560 of 18688 at 565 rows: 101 us against 107, expected of the plain product 101.5 and 100.5).
static inline RowPart best_launch(int m, int n, int k, bool wide_ok, size_t part_cap) {
    RowPart p = {m, false, tile_plan(m, n, k, 0, 0, 0, part_cap)};
    const double w = wide_ok ? wide_us(m, n, k) : 1e30;
    if (w < 1.04 * p.tile.us) {
        p.wide = true;
        p.tile.us = w;
    }
    return p;
}

// wide_ok: the 256 x 256 kernel can take the call.  part_cap: the most bytes of partial tiles a plan may ask for.
// tune: fields of a plan asked for by the caller (bits 0..7 K splits, 8..11 32-row M tiles per workgroup, 8 there for the
// 256 x 256 kernel, 12..13 wave quartets; 0 = choose), followed as far as the kernels can.
// A last round of workgroups that leaves most of the chip idle costs as much as a full one, so the rows behind the
// last 128-row boundaries are also tried as a launch of their own (shorter tiles, K split): 4096 -> 28672 at 1100
// rows is 1024 on the 256 x 256 kernel and 76 on 96-row tiles, 240 us instead of 297 in one launch.
// Up to 128 rows there is nothing to split (a second launch costs 2 us).
static inline LinearPlan linear_plan(int m, int n, int k, bool wide_ok, size_t part_cap, unsigned tune) {
    LinearPlan plan;
    plan.parts = 1;
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
        const double both = head.tile.us + tail.tile.us + 2.0;
        if (both < 0.97 * us) {
            us = both / 0.97;
            plan.parts = 2;
            plan.part[0] = head;
            plan.part[1] = tail;
        }
    }
    return plan;
}
static inline size_t plan_accum_bytes(const LinearPlan& plan, int n) {
    size_t most = 0;
    for (int i = 0; i < plan.parts; ++i) {
        const size_t b = plan.part[i].wide ? 0 : tile_accum_bytes(plan.part[i].rows, n, plan.part[i].tile);
        most = b > most ? b : most;
    }
    return most;
}
static inline size_t plan_part_bytes(const LinearPlan& plan, int n) {
    size_t most = 0;
    for (int i = 0; i < plan.parts; ++i) {
        const size_t b = plan.part[i].wide ? 0 : tile_part_bytes(plan.part[i].rows, n, plan.part[i].tile);
        most = b > most ? b : most;
    }
    return most;
}

}  // namespace uniql
