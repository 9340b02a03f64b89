"""The tiled kernels' plans (csrc/tile_plan.hpp, plain host C++): what is chosen can be run as it is."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "tile_plan.hpp"
using namespace uniql;

static bool runnable(const TilePlan& p, int k) {
    const int G = k / 128;
    if (p.mtiles < 1 || p.mtiles > 4 || p.splits < 1 || p.gps < 1) return false;
    if ((p.splits - 1) * p.gps >= G || p.splits * p.gps < G) return false;   // every split has groups, none is left over
    if (p.quartets == 2) return p.mtiles <= 2 && G % 2 == 0 && p.gps % 2 == 0;  // even ranges, the last one too
    return p.quartets == 1;
}

// Rows lo..hi of one layer: how many launches are not what the search chose once its fields are asked for, or cannot run.
extern "C" int plans_off(int n, int k, int lo, int hi, int wide_ok, int* launches) {
    int off = 0;
    *launches = 0;
    for (int m = lo; m <= hi; ++m) {
        const LinearPlan plan = linear_plan(m, n, k, wide_ok != 0, (size_t)12 << 20, 0);
        int rows = 0;
        for (int i = 0; i < plan.parts; ++i) {
            const RowPart& part = plan.part[i];
            rows += part.rows;
            if (part.wide) continue;
            ++*launches;
            const TilePlan& p = part.tile;
            const unsigned tune = (unsigned)p.splits | ((unsigned)p.mtiles << 8) | ((unsigned)p.quartets << 12);
            const TilePlan q = linear_plan(part.rows, n, k, false, 0, tune).part[0].tile;
            off += !runnable(p, k) || q.mtiles != p.mtiles || q.splits != p.splits || q.gps != p.gps || q.quartets != p.quartets;
        }
        off += rows != m;
    }
    return off;
}

// Rows lo..hi: in how many the search leaves a plan that it rates (a height, a split count, one or two quartets) below its choice.
extern "C" int plans_missed(int n, int k, int lo, int hi) {
    int missed = 0;
    for (int m = lo; m <= hi; ++m) {
        const TilePlan best = tile_plan(m, n, k, 0, 0, 0, (size_t)12 << 20);
        for (int mt = 1; mt <= 4; ++mt) {
            for (int kw = 1; kw <= 2; ++kw) {
                const TilePlan p = tile_plan(m, n, k, 0, mt, kw, (size_t)12 << 20);
                const bool rated = p.quartets == 1 || (int64_t)(n / 128) * ceil_div_i(m, 32 * mt) * p.splits <= 256;
                missed += rated && p.us < best.us;
            }
        }
    }
    return missed;
}

// Rows of the first launch of a call that runs as two, 0 if it runs as one.
extern "C" int first_of_two(int m, int n, int k) {
    const LinearPlan plan = linear_plan(m, n, k, n % 256 == 0, (size_t)12 << 20, 0);
    return plan.parts == 2 ? plan.part[0].rows : 0;
}

// Rows lo..hi: in how many the launch that is taken is neither the rule's nor faster than it by its expected time.
extern "C" int rule_left_for_nothing(int n, int k, int lo, int hi) {
    int bad = 0;
    for (int m = lo; m <= hi; ++m) {
        const RowPart rule = rule_launch(m, n, k, n % 256 == 0), p = best_launch(m, n, k, n % 256 == 0, (size_t)-1);
        bad += p.tile.us > rule.tile.us || !(p.wide || runnable(p.tile, k)) || !(rule.wide || runnable(rule.tile, k));
    }
    return bad;
}

// Products that enter one accumulator one after another, at most, in a call of m rows.
extern "C" int longest_chain(int m, int n, int k) {
    const LinearPlan plan = call_plan(m, n, k, k >= 256, (size_t)12 << 20, 0);
    int longest = 0;
    for (int i = 0; i < plan.parts; ++i) {
        const int chain = plan.part[i].wide ? k : tile_chain(plan.part[i].tile);
        longest = chain > longest ? chain : longest;
    }
    return longest;
}

// Height and K splits of a call that runs as one launch; 0 0 where it runs as two.
extern "C" void one_launch(int m, int n, int k, int* plan) {
    const LinearPlan p = call_plan(m, n, k, k >= 256, (size_t)12 << 20, 0);
    plan[0] = p.parts == 1 ? p.part[0].tile.mtiles : 0;
    plan[1] = p.parts == 1 ? p.part[0].tile.splits : 0;
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("tile_plan")
    (d / "plans.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wno-unused-function", "-shared", "-fPIC",
                    f"-I{os.path.join(ROOT, 'uniql_amd', 'csrc')}", str(d / "plans.cpp"), "-o", str(d / "plans.so")], check=True)
    return ctypes.CDLL(str(d / "plans.so"))


@pytest.mark.parametrize("n", [256, 1024, 4096, 6144, 18688, 28672])
def test_the_plan_that_is_chosen_is_the_plan_that_its_fields_ask_for(plans, n):
    """a field set that names a choice (K splits, tile height, quartets) leads back to that choice, group count per
    split included: 10496 -> 4096 at 65 rows wants two splits of 42 groups for two quartets, not of 41"""
    launches = ctypes.c_int(0)
    total = 0
    for k in list(range(128, 2048, 384)) + list(range(2048, 14337, 128)):
        for lo, hi in ((17, 200), (320, 340), (1090, 1110), (4090, 4096)):
            for wide_ok in (0, 1):
                assert plans.plans_off(n, k, lo, hi, wide_ok, ctypes.byref(launches)) == 0, (n, k, lo, hi, wide_ok)
                total += launches.value
    assert total > 10000


@pytest.mark.parametrize("n", [256, 1024, 4096, 6144, 28672])
def test_the_search_rates_one_and_two_quartets(plans, n):
    """4096 -> 1024 at 97 rows: one quartet is the faster of the two where both fit"""
    for k in (128, 512, 1280, 2688, 4096, 7424, 10496, 14336):
        assert plans.plans_missed(n, k, 17, 1100) == 0, (n, k)
        assert plans.rule_left_for_nothing(n, k, 17, 1100) == 0, (n, k)


@pytest.mark.parametrize("m,k,n,head", [(1100, 4096, 28672, 1024), (1100, 14336, 4096, 1024), (1057, 11008, 4096, 1024),
                                        (1030, 11008, 4096, 1024), (1024, 4096, 18688, 768), (128, 4096, 28672, 0)])
def test_calls_that_run_as_two_launches(plans, m, k, n, head):
    """the sizes at which the GPU tests of two launches look at their results do run as two"""
    assert plans.first_of_two(m, n, k) == head


@pytest.mark.parametrize("m,k,n,chain", [(459, 10752, 2048, 672), (275, 13056, 3072, 832), (277, 9984, 3200, 640), (281, 11776, 2176, 512),
                                         (462, 11264, 2048, 704), (1985, 14336, 512, 896),        # 64-row tiles of two quartets
                                         (3558, 12672, 3968, 3168), (2132, 13440, 14976, 3360)])  # 128-column kernel alone
def test_sums_get_no_longer_for_a_gain_of_a_few_per_cent(plans, m, k, n, chain):
    """sizes at which taller tiles with K split, or the 256 x 256 kernel with such tiles behind it, are expected to be a little
    faster than a plan whose sums are shorter chains of products"""
    assert plans.longest_chain(m, n, k) <= chain


@pytest.mark.parametrize("m,k,n,mtiles,splits", [(1563, 10624, 384, 2, 3), (1326, 6784, 768, 2, 2), (3025, 7424, 512, 2, 1),
                                                 (96, 6272, 6656, 3, 4)])
def test_many_rows_and_few_columns_stay_on_fewer_splits(plans, m, k, n, mtiles, splits):
    """with at least as many rows as columns taller tiles with more splits were slower than expected (24.4 -> 32.9 us at the first
    of these); with fewer they are what is chosen"""
    plan = (ctypes.c_int * 2)()
    plans.one_launch(m, n, k, plan)
    assert tuple(plan) == (mtiles, splits)
