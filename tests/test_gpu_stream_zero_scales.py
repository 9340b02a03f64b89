"""Streaming kernel from 3 rows on: scales of zero stay in the short expansion, strips of padding columns are left out."""
import pytest
import torch

from tests.helpers import workspace_for

pytestmark = pytest.mark.gpu

F_FORCE_SKINNY = 1 << 1


@pytest.mark.parametrize("m,k,n", [(3, 640, 256), (4, 4096, 128), (8, 2304, 384), (16, 1280, 256)])
def test_zero_scales_and_padding_strips(gpu, m, k, n):
    """one-hot rows: every output is one product 1 * w, for units of zeros, zeros of both signs between scales at the ends of
    the short expansion's range, and the same beside one outside it; then layers whose last strips are padding"""
    from uniql_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(m + k)
    b = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=gpu, generator=gen)
    s = (0.004 + 0.016 * torch.rand((k // 128, n), device=gpu, generator=gen)).half()
    s[0] = 0.0
    s[1, 3:90], s[1, 7], s[1, 100], s[1, 101] = 0.0, -0.0, 2.0 ** -10, 0.0624
    s[2, ::2], s[2, 1] = 0.0, 2.0 ** -11
    s[3, 64:], s[3, 5] = 0.0, 0.0625
    s[4, 1::2], s[4, 4], s[4, 6] = -0.0, -0.01, 6e-8
    w = ops.w4a16_dequant(b, s, n, k)
    ws = workspace_for(n, gpu)
    for first in range(0, k, 40):
        at = (torch.arange(m, device=gpu) * 37 + 5 + first) % k
        x = torch.zeros((m, k), dtype=torch.float16, device=gpu)
        x[torch.arange(m, device=gpu), at] = 1.0
        y = ops.w4a16_gemm_ex(x, b, s, ws, m, n, k, out_f32=True, flags=F_FORCE_SKINNY)
        assert torch.equal(y, w[at].float())
    x = torch.randn((m, k), device=gpu, generator=gen).half()
    y = ops.w4a16_linear(x, b, s, ws, n, k, flags=F_FORCE_SKINNY)
    pair = ops.w4a16_linear(x, b, s, ws, n, k, silu_mul=True, flags=F_FORCE_SKINNY)
    for n_out in (n - 8, n - 128, 64):
        if n_out <= 0:
            continue
        assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, flags=F_FORCE_SKINNY), y[:, :n_out])
        half = min(n_out // 16 * 8, n // 2)
        assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, silu_mul=True, out_features=half, flags=F_FORCE_SKINNY), pair[:, :half])
    assert all(int(words.count_nonzero()) == 0 for words in ops._accum_cache.values())
