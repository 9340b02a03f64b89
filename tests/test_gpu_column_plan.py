"""Prefill calls whose columns run as two launches."""
import pytest
import torch

from tests.helpers import check_layer_output_torch, workspace_for

pytestmark = pytest.mark.gpu

F_FORCE_TILED, TILE96 = 1 << 2, 3 << 16


# large tiles and 96-row tiles behind them; an odd number of strips, the last one alone; 128-row tiles and 32-row ones that
# split K behind them; one K group more than the large tiles need
@pytest.mark.parametrize("m,k,n", [(1024, 512, 18688), (1024, 1024, 16512), (203, 8192, 18688), (3000, 384, 5760)])
def test_columns_in_two_launches(gpu, m, k, n):
    """against the dequantised weights, and every epilogue bit for bit from the plain product"""
    from uniql_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(m + n)
    b = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=gpu, generator=gen)
    s = (0.004 + 0.016 * torch.rand((k // 128, n), device=gpu, generator=gen)).half()
    ws = workspace_for(n, gpu)
    x = torch.randn((m, k + 8), device=gpu, generator=gen).half()[:, :k]     # strided rows
    y = ops.w4a16_linear(x, b, s, ws, n, k)
    w = ops.w4a16_dequant(b, s, n, k).double()
    check_layer_output_torch(y, torch.cat([part.double() @ w for part in x.split(256)]))
    one = ops.w4a16_linear(x, b, s, ws, n, k, flags=F_FORCE_TILED | TILE96 | (1 << 8))
    assert float((y.float() - one.float()).abs().max()) <= 2 ** -10 * max(1.0, float(y.float().abs().max()))  # one fp16 step
    bias = torch.randn(n, device=gpu, generator=gen).half()
    n_out = n - 40
    wide = torch.randn((m, n_out + 16), device=gpu, generator=gen).half()
    stream = wide[:, 8:8 + n_out]
    want = (stream.float() + (y[:, :n_out].float() + bias[:n_out].float()).half().float()).half()
    got = ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, bias=bias[:n_out].clone(), residual=stream, out=stream)
    assert got.data_ptr() == stream.data_ptr() and torch.equal(got, want)
    assert torch.equal(ops.w4a16_gemm_ex(x, b, s, ws, m, n, k, transpose_out=True)[:, :m].t(), y)
    r = torch.relu(y.float())
    assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, relu2=True), (r * r).half())
    pair = ops.w4a16_linear(x, b, s, ws, n, k, silu_mul=True)
    gate, up = y.view(m, n // 128, 2, 64).unbind(2)
    want = (torch.nn.functional.silu(gate.float()).half().float() * up.float()).half().reshape(m, n // 2)
    # expf and torch's exp differ in the last bit now and then: one fp16 step of the activation
    assert torch.all((pair.float() - want.float()).abs() <= 2 * 2 ** -10 * want.float().abs() + 2 ** -24)
    assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, silu_mul=True, out_features=n // 2 - 72), pair[:, :n // 2 - 72])
    # one scale per column: the large tiles do not take it, the columns may still be split
    single = (0.004 + 0.016 * torch.rand((1, n), device=gpu, generator=gen)).half()
    y1 = ops.w4a16_gemm_ex(x.contiguous(), b, single, ws, m, n, k)
    w = ops.w4a16_dequant(b, single, n, k).double()
    check_layer_output_torch(y1, torch.cat([part.double() @ w for part in x.split(256)]))
    assert all(int(words.count_nonzero()) == 0 for words in ops._accum_cache.values())
