"""Scratch memory that is enough for the streaming or the tiled kernels only: the call runs there, as if asked for."""
import ctypes

import pytest
import torch

from tests.helpers import workspace_for

pytestmark = pytest.mark.gpu

F_FORCE_SKINNY, F_FORCE_TILED, ONE_SPLIT, MID = 1 << 1, 1 << 2, 1 << 8, 9 << 16


def _call(lib, x, b, s, d, ws, accum, temp, m, n, k, flags=0):
    stream = torch.cuda.current_stream().cuda_stream
    return lib.uniql_w4a16_gemm(x.data_ptr(), k, b.data_ptr(), s.data_ptr(), d.data_ptr(), ws.data_ptr(), ws.numel(),
                                accum.data_ptr(), accum.numel() * 8, temp.data_ptr() if temp is not None else None,
                                temp.numel() if temp is not None else 0, m, n, k, k // 128, 0, 1.0, flags, stream)


@pytest.mark.parametrize("m,k,n", [(10, 2048, 1024), (16, 4096, 4096), (48, 4096, 256), (40, 14336, 4096), (203, 8192, 18688)])
def test_too_little_scratch_takes_the_other_kernels(gpu, m, k, n):
    from uniql_amd import _capi
    lib = _capi.load()
    gen = torch.Generator(device=gpu).manual_seed(m + k)
    b = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=gpu, generator=gen)
    s = (0.004 + 0.016 * torch.rand((k // 128, n), device=gpu, generator=gen)).half()
    x = torch.randn((m, k), device=gpu, generator=gen).half()
    ws = workspace_for(n, gpu)
    accum = torch.zeros(min(m, 16) * n, dtype=torch.int64, device=gpu)
    acc, tmp = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert lib.uniql_w4a16_linear_workspace(m, n, k, k, 0, 0, ctypes.byref(acc), ctypes.byref(tmp)) == 0
    assert tmp.value > 0                                            # the kernel that takes the call by itself splits K
    full = torch.empty(tmp.value, dtype=torch.uint8, device=gpu)
    outs = [torch.full((m, n), float("nan"), dtype=torch.float16, device=gpu) for _ in range(3)]
    if m > 64:
        # the one-launch plan splits nothing: no temp
        small, same = None, F_FORCE_TILED
        assert lib.uniql_w4a16_linear_workspace(m, n, k, k, 0, F_FORCE_TILED | ONE_SPLIT, ctypes.byref(acc), ctypes.byref(tmp)) == 0
        assert tmp.value == 0
    elif m <= 16:
        small, same = None, F_FORCE_SKINNY
    else:
        assert lib.uniql_w4a16_linear_workspace(m, n, k, k, 0, F_FORCE_TILED, ctypes.byref(acc), ctypes.byref(tmp)) == 0
        assert tmp.value < full.numel()
        small, same = torch.empty(tmp.value, dtype=torch.uint8, device=gpu) if tmp.value else None, F_FORCE_TILED
    assert _call(lib, x, b, s, outs[0], ws, accum, full, m, n, k) == 0
    assert _call(lib, x, b, s, outs[1], ws, accum, small, m, n, k) == 0
    if m <= 64:
        assert _call(lib, x, b, s, outs[2], ws, accum, full, m, n, k, same) == 0
        assert torch.equal(outs[1], outs[2])
        assert _call(lib, x, b, s, outs[2], ws, accum, None, m, n, k, F_FORCE_TILED | MID) != 0    # asked for: refused
    # one fp16 step between two orders of the same sum
    assert float((outs[0].float() - outs[1].float()).abs().max()) <= 2 ** -10 * max(1.0, float(outs[1].float().abs().max()))
    assert int(accum.count_nonzero()) == 0
