"""What the loads of the kernel for 9 to 64 rows can reach (csrc/w4a16_mid.hip; sizes and offsets are those of
csrc/mid_plan.hpp, plain C++).  A load has a lane offset and, for packed rows, a scalar offset against a descriptor's
size; whether the hardware's check leaves the scalar offset out, adds it or takes it off the size (in 32 bits) is not
relied on: a load of what exists stays inside under each of them, and one that must bring nothing is outside."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "mid_plan.hpp"
using namespace uniql;
// bit r: suppressed under rule r (scalar offset left out, added, taken off the size)
static unsigned suppressed(uint32_t records, uint32_t lane, uint32_t scalar) {
    return (lane >= records) | (((uint64_t)lane + scalar >= records) << 1) | ((lane >= (uint32_t)(records - scalar)) << 2);
}
// loads of one call's rows, groups and lanes (real units and the one behind the last) that are not what they should be
extern "C" int x_loads_off(int m, int64_t lda, int k_valid, int k) {
    const uint32_t x_bytes = (uint32_t)(((int64_t)(m - 1) * lda + k_valid) * 2);
    int off = 0;
    for (int g = 0; g <= k / 128; ++g)
        for (int row = 0; row < 16 * mid_row_tiles(m); ++row)
            for (int slot = 0; slot < 16; ++slot) {
                const bool real = g < k / 128, column = 128 * g + 8 * slot < k_valid;
                const uint32_t lane = column ? (uint32_t)row * (uint32_t)lda * 2u + 16u * slot : kMidNoLoad;
                const unsigned s = suppressed(mid_x_records(x_bytes, g, real), lane, 0);
                const bool wanted = real && row < m && column;
                off += s != (wanted ? 0u : 7u);
                if (wanted) off += 256ull * g + lane + 16 > x_bytes;
            }
    return off;
}
extern "C" int row_loads_off(int n) {
    const uint32_t records = (uint32_t)mid_group_bytes(n), row_bytes = 8u * (uint32_t)n;
    int off = mid_group_bytes(n) > (int64_t)kMidNoLoad;
    for (uint32_t row = 0; row < 8; ++row)
        for (uint32_t piece = 0; piece < 64; ++piece) {
            const uint32_t strip = 1024u * (uint32_t)(n / 128 - 1);   // the last strip's descriptor starts there
            off += suppressed(records, 16 * piece, row * row_bytes) != 0;
            off += (uint64_t)strip + 16 * piece + row * row_bytes + 16 > records;
            off += suppressed(records, kMidNoLoad, row * row_bytes) != 7;
        }
    return off;
}
"""


@pytest.fixture(scope="module")
def loads(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("mid_loads")
    (d / "loads.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wno-unused-function", "-Wno-unused-variable", "-shared", "-fPIC",
                    f"-I{os.path.join(ROOT, 'uniql_amd', 'csrc')}", str(d / "loads.cpp"), "-o", str(d / "loads.so")], check=True)
    lib = ctypes.CDLL(str(d / "loads.so"))
    lib.x_loads_off.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    return lib


@pytest.mark.parametrize("m", [9, 16, 33, 48, 49, 64])
@pytest.mark.parametrize("k_valid,lda", [(128, 128), (8, 8), (128, 1 << 23), (2048, 2048), (2040, 2048), (4096, 4104), (14336, 14336), (11840, 20000)])
def test_rows_of_x(loads, m, k_valid, lda):
    k = (k_valid + 127) // 128 * 128
    if ((m - 1) * lda + k) * 2 < 1 << 31:      # as mid_shape_ok asks
        assert loads.x_loads_off(m, lda, k_valid, k) == 0


@pytest.mark.parametrize("n", [128, 256, 4096, 28672, 256000, (1 << 25) - 128, 1 << 25])
def test_packed_rows(loads, n):
    assert loads.row_loads_off(n) == 0
