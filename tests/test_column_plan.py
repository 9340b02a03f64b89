"""Which columns run in which launch (csrc/tile_plan.hpp, plain host C++)."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "tile_plan.hpp"
using namespace uniql;
// calls of lo..hi rows: how many have parts that do not cover the layer or that a kernel cannot take
extern "C" int calls_off(int n, int k, int lo, int hi, int wide_ok, int* split) {
    int off = 0;
    for (int m = lo; m <= hi; ++m) {
        const LinearPlan p = call_plan(m, n, k, wide_ok != 0, (size_t)12 << 20, 0);
        *split += p.head_columns > 0;
        if (p.head_columns == 0) {
            off += (p.parts == 1 ? p.part[0].rows : p.part[0].rows + p.part[1].rows) != m;
        } else {
            off += m <= 64 || p.parts != 2 || p.part[0].rows != m || p.part[1].rows != m;
            off += p.head_columns % 128 != 0 || p.head_columns <= 0 || p.head_columns >= n;
        }
        for (int i = 0; i < p.parts; ++i) {
            const int c = part_columns(p, i, n);
            if (p.part[i].wide) {
                off += c % 256 != 0 || !wide_ok;
            } else {
                off += tile_accum_bytes(p.part[i].rows, c, p.part[i].tile) > plan_accum_bytes(p, n);
                off += tile_part_bytes(p.part[i].rows, c, p.part[i].tile) > plan_part_bytes(p, n) || plan_part_bytes(p, n) > ((size_t)12 << 20);
            }
        }
    }
    return off;
}
extern "C" int head_columns(int m, int n, int k, unsigned tune) { return call_plan(m, n, k, true, (size_t)12 << 20, tune).head_columns; }
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("column_plan")
    (d / "plans.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wno-unused-function", "-shared", "-fPIC",
                    f"-I{os.path.join(ROOT, 'uniql_amd', 'csrc')}", str(d / "plans.cpp"), "-o", str(d / "plans.so")], check=True)
    return ctypes.CDLL(str(d / "plans.so"))


@pytest.mark.parametrize("n", [128, 256, 384, 4096, 5760, 16512, 18688, 28672])
@pytest.mark.parametrize("wide_ok", [0, 1])
def test_parts_cover_the_layer_and_can_be_run(plans, n, wide_ok):
    split = ctypes.c_int(0)
    for k in (128, 256, 512, 1024, 4096, 8192, 14336):
        for lo, hi in ((17, 260), (1000, 1100), (2990, 3010), (4090, 4096)):
            assert plans.calls_off(n, k, lo, hi, wide_ok, ctypes.byref(split)) == 0, (n, k, lo, hi)
    assert split.value > 0 or n not in (5760, 16512, 18688)


@pytest.mark.parametrize("m,k,n,head", [(1024, 4096, 18688, 16384), (1024, 512, 18688, 16384), (1024, 1024, 16512, 16384),
                                        (203, 8192, 18688, 16384), (3000, 384, 5760, 5376), (4096, 4096, 6144, 0),
                                        (1100, 4096, 28672, 0), (64, 8192, 18688, 0)])
def test_calls_whose_columns_are_split(plans, m, k, n, head):
    """the sizes at which the GPU test looks at the results; fields of a plan asked for by the caller are one launch"""
    assert plans.head_columns(m, n, k, 0) == head
    assert plans.head_columns(m, n, k, 1) == 0
