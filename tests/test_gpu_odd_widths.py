"""Output widths that are no multiple of eight, and residuals requested ahead of the stores: what the kernels for more than
eight rows store equals the unfused sequence on their own fp32 sums, bit for bit."""
import pytest
import torch

from tests.helpers import make_linear_problem, to_gpu, workspace_for

pytestmark = pytest.mark.gpu
F_TILED = 4
# rows and flags: the kernel for 9 to 64 rows, every tile height with one and two quartets and with K split, the 256 x 256 kernel
CALLS = [(12, 0), (24, 0), (40, 0), (60, 0)] + [(131, F_TILED | (s << 8) | (mt << 16) | (kw << 20))
         for mt, kw in ((1, 1), (1, 2), (2, 1), (2, 2), (3, 1), (4, 1)) for s in (1, 3)] + [(300, F_TILED | (8 << 16))]


@pytest.mark.parametrize("n_out", [512, 511, 508, 385, 257])
@pytest.mark.parametrize("m,flags", CALLS)
def test_stores_equal_the_unfused_sequence(gpu, m, flags, n_out):
    from uniql_amd import ops
    k, n = 12 * 128, 512
    p = make_linear_problem(m, k, n, seed=m + n_out)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    g = torch.Generator(device=gpu).manual_seed(n_out)
    bias = torch.randn(n_out, device=gpu, generator=g).half()
    residual = torch.randn((m, n_out), device=gpu, generator=g).half()

    def call(**kw):
        return ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, flags=flags, **kw)

    y32 = ops.w4a16_linear(x, b, s, ws, n, k, out_f32=True, flags=flags)[:, :n_out]
    y16 = y32.half()
    y16b = (y16.float() + bias.float()).half()
    assert torch.equal(call(), y16)
    assert torch.equal(call(bias=bias), y16b)
    assert torch.equal(call(residual=residual), (residual.float() + y16.float()).half())
    assert torch.equal(call(residual=residual, bias=bias), (residual.float() + y16b.float()).half())
    assert torch.equal(call(relu2=True), (y16.float().clamp_min(0) ** 2).half())
    # into a wider buffer whose rows are 16-byte aligned, the residual in place: rows end inside a unit of eight
    wide = torch.zeros((m, 520), dtype=torch.float16, device=gpu)
    wide[:, :n_out] = residual
    ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, flags=flags, residual=wide[:, :n_out], out=wide[:, :n_out])
    assert torch.equal(wide[:, :n_out], (residual.float() + y16.float()).half()) and not wide[:, n_out:].any()


@pytest.mark.parametrize("n_out", [256, 255, 131])
@pytest.mark.parametrize("m,flags", CALLS)
def test_gated_stores_end_at_the_width(gpu, m, flags, n_out):
    from uniql_amd import ops
    k, n = 12 * 128, 512
    p = make_linear_problem(m, k, n, seed=m + n_out)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    bias = torch.randn(2 * n_out, device=gpu, generator=torch.Generator(device=gpu).manual_seed(7)).half()
    y16 = ops.w4a16_linear(x, b, s, ws, n, k, out_f32=True, flags=flags).half().reshape(m, n // 128, 2, 64)
    gate, up = y16[:, :, 0].reshape(m, n // 2)[:, :n_out], y16[:, :, 1].reshape(m, n // 2)[:, :n_out]
    gate, up = (gate.float() + bias[:n_out].float()).half(), (up.float() + bias[n_out:].float()).half()
    want = (torch.nn.functional.silu(gate.double()).half().float() * up.float()).half()
    out = torch.zeros((m, 264), dtype=torch.float16, device=gpu)
    ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, silu_mul=True, bias=bias, flags=flags, out=out[:, :n_out])
    dense = ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, silu_mul=True, bias=bias, flags=flags)
    assert torch.equal(dense, out[:, :n_out]) and not out[:, n_out:].any()
    # the kernel's silu is fp32 with the device's expf: its fp16 rounding may fall to the neighbour, then the product's too
    assert float((dense.float() - want.float()).abs().max()) <= 2.0 ** -9 * float(want.float().abs().max())
    assert float((dense != want).float().mean()) < 0.01


@pytest.mark.parametrize("n_out", [512, 504, 508, 385])
@pytest.mark.parametrize("m,flags", [(12, 0), (40, 0), (131, F_TILED | 1 << 8 | 2 << 16 | 1 << 20), (131, F_TILED | 3 << 8 | 3 << 16), (300, F_TILED | 8 << 16)])
def test_float32_results_with_a_bias(gpu, m, flags, n_out):
    """the sum and the bias added once in fp32, also from a bias that is not 16-byte aligned, then the rest of the epilogue"""
    from uniql_amd import ops
    k, n = 12 * 128, 512
    p = make_linear_problem(m, k, n, seed=m + n_out)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    g = torch.Generator(device=gpu).manual_seed(n_out)
    bias = torch.randn(n_out + 1, device=gpu, generator=g).half()
    residual = torch.randn((m, n_out), device=gpu, generator=g).half()
    y32 = ops.w4a16_linear(x, b, s, ws, n, k, out_f32=True, flags=flags)[:, :n_out]
    for aligned in (bias[:n_out], bias[1:]):
        want = y32 + aligned.float()
        call = dict(out_features=n_out, bias=aligned, out_f32=True, flags=flags)
        assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, **call), want)
        assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, residual=residual, **call), want + residual.float())
        assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, relu2=True, **call), want.clamp_min(0) ** 2)
        wide = torch.zeros((m, 520), dtype=torch.float32, device=gpu)
        ops.w4a16_linear(x, b, s, ws, n, k, out=wide[:, :n_out], **call)
        assert torch.equal(wide[:, :n_out], want) and not wide[:, n_out:].any()
