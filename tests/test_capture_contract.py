"""What a layer call asks of the HIP runtime beside launches and of its caller, on a recorder in the runtime's place
(tests/fake_hip.cpp, no GPU).  Function attributes are set on the first call on a device, for every kernel that a later call may
launch, so that a call recorded into a graph sets none; exchange words, which a graph may have to clear on every replay, are
asked for where workgroups share output columns and nowhere else."""
import os
import shutil
import subprocess
import sys

import pytest

from uniql_amd.build import LIB_PATH

HERE = os.path.dirname(os.path.abspath(__file__))

SETUP = r"""
import ctypes, itertools, sys
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
P, I, L, F, U, Z = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_uint, ctypes.c_size_t
lib.uniql_w4a16_linear.argtypes = [P, L, I, P, P, P, P, L, P, L, I, I, P, L, P, Z, P, Z, I, I, I, I, I, F, U, P]
lib.uniql_w4a16_linear_workspace.argtypes = [I, I, I, I, I, U, ctypes.POINTER(Z), ctypes.POINTER(Z)]
lib.uniql_w4a16_gemm_static.argtypes = [P, L, P, P, P, P, L, I, I, I, I, I, F, U, P]
fake = 1 << 20   # an address that nobody reads

def call(m, k, n, had=0, flags=0, k_in=None, static=False, n_out=None):
    k_in = k if k_in is None else k_in
    before = hip.fake_launches()
    if static:
        code = lib.uniql_w4a16_gemm_static(fake, k, fake, fake, fake, None, 0, m, n, k, k // 128, had, 1.0, flags, None)
    else:
        acc, tmp = Z(0), Z(0)
        assert lib.uniql_w4a16_linear_workspace(m, n, k, k_in, had, flags, ctypes.byref(acc), ctypes.byref(tmp)) == 0
        code = lib.uniql_w4a16_linear(fake, k_in, k_in, fake, fake, None, None, 0, fake, n_out or n, n_out or n, 0, None, 0,
                                      fake, acc.value, fake, tmp.value, m, n, k, k // 128, had, 1.0, flags, None)
    assert code == (-7 if code == -7 and static else 0), (m, k, n, had, flags, code)
    assert code != 0 or hip.fake_launches() > before
    return None if static else acc.value

"""

CALLS = SETUP + r"""
first = eval(sys.argv[3])
call(*first[0], **first[1])
once = hip.fake_attributes()
assert once > 0
for static in (False, True):
    for m, (k, n) in itertools.product((1, 2, 4, 8, 9, 16, 17, 32, 33, 48, 49, 64, 100, 333, 1024, 4096),
                                       ((4096, 4096), (4096, 28672), (14336, 4096), (512, 256), (2048, 18688), (16384, 1024), (32768, 512))):
        call(m, k, n, static=static)
        call(m, k, n, had=128, static=static)
        if k & (k - 1) == 0:
            call(m, k, n, had=k, static=static)
            call(m, k, n, had=1024 if k > 512 else 256, static=static)
        if not static:
            call(m, k, n, k_in=k - 8, n_out=n - 24)
            call(m, k, n, flags=1 << 1)              # forced: streaming
            call(m, k, n, flags=1 << 2)              #         tiled
            for rows, quartets in itertools.product((1, 2, 3, 4, 8), (1, 2)):
                call(m, k, n, flags=1 << 2 | rows << 16 | quartets << 20)
assert hip.fake_refused() == 0
assert hip.fake_attributes() == once, (once, hip.fake_attributes())
print("launches", hip.fake_launches(), "attributes", once)
"""


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists(LIB_PATH):
        pytest.skip("g++ and the built library are needed")
    path = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.cpp"), "-o", path], check=True)
    return path


@pytest.mark.parametrize("first", ["((1, 4096, 4096), {})", "((16, 4096, 28672), {})", "((1024, 4096, 4096), {})",
                                   "((1, 512, 256), dict(static=True))"])
def test_the_first_call_prepares_every_later_one(recorder, first):
    run = subprocess.run([sys.executable, "-c", CALLS, recorder, LIB_PATH, first], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stderr[-2000:]


WORDS = SETUP + r"""
skinny = 1 << 1
for k, n in itertools.product((256, 512, 640, 2048, 2176, 4096, 8192, 8320, 14336), (128, 1024, 4096, 18304, 18432, 24320, 28672)):
    for m in (1, 2, 3, 4, 7, 8, 9, 12, 16, 20, 35):
        for tune in (0, 1, 3, 8 << 8, 4 << 8 | 2, 8 << 8 | 32):   # groups a wave, waves a workgroup
            words = call(m, k, n, flags=skinny | tune << 8)
            split = hip.fake_grid_y() > 1   # of the last slab of 16 rows
            slabs = [16] * (m // 16) + ([m % 16] if m % 16 else [])
            if len(slabs) == 1:
                assert words == (m * n * 8 if split else 0), (m, k, n, tune, words)
            else:
                assert words in (0, slabs[-1] * n * 8, 16 * n * 8) and (words > 0 or not split)
                lone = [call(rows, k, n, flags=skinny | tune << 8) for rows in slabs]
                assert words == max(lone)
for m in range(1, 9):
    assert call(m, 4096, 28672) == 0 and call(m, 4096, 24320) == 0
"""


def test_words_are_asked_for_where_k_is_split(recorder):
    run = subprocess.run([sys.executable, "-c", WORDS, recorder, LIB_PATH], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stderr[-2000:]
