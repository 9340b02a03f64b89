"""Inputs with fewer columns than the packed weights have rows: the kernels for more than 64 rows read such rows as they are.  The
same bits as behind a zero-padded copy, whatever follows a row in memory."""
import pytest
import torch

from tests.helpers import make_linear_problem, to_gpu, workspace_for

pytestmark = pytest.mark.gpu
F_TILED = 4
# every tile height, one and two quartets, with and without a K split, and the 256 x 256 kernel
PLANS = [(s << 8) | (mt << 16) | (kw << 20) for mt, kw in ((1, 1), (1, 2), (2, 1), (2, 2), (3, 1), (4, 1)) for s in (1, 2)] + [8 << 16]


@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("groups,missing", [(1, 24), (2, 8), (2, 120), (3, 64), (4, 72), (6, 56), (12, 16), (14, 104)])
def test_short_rows(gpu, plan, groups, missing):
    from uniql_amd import ops
    m, k, n = 300, 128 * groups, 256
    k_in = k - missing
    p = make_linear_problem(m, k, n, seed=groups + missing)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    flags = F_TILED | plan
    x = x[:, :k_in].contiguous()           # a row is followed by the next one
    x[7, :8], x[m - 1, :8] = float("inf"), float("nan")
    padded = torch.zeros((m, k), dtype=x.dtype, device=gpu)
    padded[:, :k_in] = x
    apart = torch.full((m * (k_in + 24),), float("nan"), dtype=x.dtype, device=gpu)[:(m - 1) * (k_in + 24) + k_in]
    apart = apart.as_strided((m, k_in), (k_in + 24, 1))   # or by something else, and the last one ends the buffer
    apart.copy_(x)
    want = ops.w4a16_linear(padded, b, s, ws, n, k, flags=flags)
    clean = torch.ones(m, dtype=torch.bool, device=gpu)
    clean[[7, m - 1]] = False
    assert torch.isfinite(want[clean]).all() and not torch.isfinite(want[~clean]).any()
    for rows in (x, apart):
        got = ops.w4a16_linear(rows, b, s, ws, n, k, flags=flags)
        assert torch.equal(got[clean], want[clean])
        assert not torch.isfinite(got[~clean]).any()


@pytest.mark.parametrize("m", [65, 129, 333, 1100])
def test_short_rows_on_the_plan_of_the_call(gpu, m):
    """rows and columns in two launches, bias, residual and gated pairs among them"""
    from uniql_amd import ops
    for k_in, n, kw in ((1992, 4096, dict(residual=True)), (2048 - 120, 2816, dict(bias=True)), (2040, 1536, dict(silu_mul=True))):
        k = 2048
        p = make_linear_problem(m, k, n, seed=m + k_in)
        x, b, s = to_gpu(p, gpu)
        ws = workspace_for(n, gpu)
        x = x[:, :k_in].contiguous()
        padded = torch.zeros((m, k), dtype=x.dtype, device=gpu)
        padded[:, :k_in] = x
        if "residual" in kw:
            kw = dict(residual=torch.randn((m, n), device=gpu, generator=torch.Generator(device=gpu).manual_seed(m)).half())
        if "bias" in kw:
            kw = dict(bias=torch.randn(n, device=gpu, generator=torch.Generator(device=gpu).manual_seed(m)).half())
        assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, **kw), ops.w4a16_linear(padded, b, s, ws, n, k, **kw))


@pytest.mark.parametrize("m,k_in,n,flags", [(300, 2040, 1536, 0), (100, 1992, 512, 0), (2000, 4008, 4096, 0), (300, 2040, 256, F_TILED | 1 << 8 | 2 << 16 | 1 << 20)])
def test_short_rows_take_no_scratch_memory_for_a_copy(gpu, m, k_in, n, flags):
    """a call holds its result and what whole rows of the same layer take: the copy that is not made has no room either"""
    import ctypes

    from uniql_amd import _capi, ops
    k = (k_in + 127) // 128 * 128
    p = make_linear_problem(m, k, n, seed=m)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    x = x[:, :k_in].contiguous()
    y = torch.empty((m, n), dtype=torch.float16, device=gpu)
    ops.w4a16_linear(x, b, s, ws, n, k, flags=flags, out=y)    # the exchange words are there now
    acc, tmp = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert _capi.load().uniql_w4a16_linear_workspace(m, n, k, k, 0, flags, ctypes.byref(acc), ctypes.byref(tmp)) == 0
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.w4a16_linear(x, b, s, ws, n, k, flags=flags, out=y)
    assert torch.cuda.max_memory_allocated() - before <= (tmp.value + 511) // 512 * 512


@pytest.mark.parametrize("m", [17, 24])
def test_short_rows_too_far_apart(gpu, m):
    """2^24 values and more from one row to the next: copied in front of the tiled kernels, whose offsets have 32 bits"""
    from uniql_amd import ops
    k, k_in, n, apart = 512, 488, 256, 1 << 24
    p = make_linear_problem(m, k, n, seed=m)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    far = torch.empty((m - 1) * apart + k_in, dtype=x.dtype, device=gpu).as_strided((m, k_in), (apart, 1))
    far.copy_(x[:, :k_in])
    padded = torch.zeros((m, k), dtype=x.dtype, device=gpu)
    padded[:, :k_in] = x[:, :k_in]
    plan = F_TILED | 1 << 8 | 1 << 16 | 1 << 20
    assert torch.equal(ops.w4a16_linear(far, b, s, ws, n, k, flags=plan), ops.w4a16_linear(padded, b, s, ws, n, k, flags=plan))
    torch.testing.assert_close(ops.w4a16_linear(far, b, s, ws, n, k), ops.w4a16_linear(padded, b, s, ws, n, k, flags=plan),
                               rtol=2 ** -9, atol=2 ** -9)  # another plan's order of fp32 sums: a rounding to fp16 apart, below 1 the same absolutely


@pytest.mark.parametrize("m,k_in,n", [(25, 1744, 28032), (29, 9664, 15360), (17, 14280, 9216), (19, 3752, 26752)])
def test_short_rows_up_to_32_stay_in_the_kernel_for_9_to_64(gpu, m, k_in, n):
    """sizes at which the tiled kernels are rated a little better, as they are for whole rows: the other kernel's bits, not theirs"""
    from uniql_amd import ops
    k = (k_in + 127) // 128 * 128
    g = torch.Generator(device=gpu).manual_seed(m)
    b = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=gpu, generator=g)
    s = (0.004 + 0.016 * torch.rand((k // 128, n), device=gpu, generator=g)).half()
    x = torch.randn((m, k_in), device=gpu, generator=g).half()
    ws = workspace_for(n, gpu)
    got = ops.w4a16_linear(x, b, s, ws, n, k)
    assert torch.equal(got, ops.w4a16_linear(x, b, s, ws, n, k, flags=9 << 16))
    assert not torch.equal(got, ops.w4a16_linear(x, b, s, ws, n, k, flags=F_TILED))
