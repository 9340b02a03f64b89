"""The kernel for 9 to 64 rows: edges of its row tiles, K splits of unequal length, scales on every side of its
expansion's range, the epilogues, short and strided inputs, replays."""
import numpy as np
import pytest
import torch

from tests.helpers import check_layer_output_torch, make_linear_problem, reference_product, to_gpu, workspace_for

pytestmark = pytest.mark.gpu

F_FORCE_SKINNY, F_FORCE_TILED, MID = 1 << 1, 1 << 2, 9 << 16


def _flags(groups_per_wave):
    return F_FORCE_TILED | MID | (groups_per_wave << 8)


# a 16-row tile's edges; one group, fewer groups than waves, K split with a short last workgroup and one unit, many splits
@pytest.mark.parametrize("m,k,n,upw", [(9, 128, 128, 1), (16, 1152, 256, 1), (17, 640, 128, 1), (31, 2176, 256, 2), (32, 1024, 384, 1),
                                       (33, 512, 256, 1), (48, 1664, 128, 2), (49, 384, 256, 1), (64, 2560, 128, 1), (64, 640, 256, 3),
                                       # 3, 4, 9 and 19 partial tiles: the last wave asks for them by two, four and eight
                                       (9, 3200, 128, 1), (16, 9216, 128, 1), (30, 3072, 128, 1), (40, 4608, 128, 1), (50, 1536, 128, 1),
                                       (64, 9600, 128, 1)])
def test_every_row_tile_and_split(gpu, m, k, n, upw):
    from uniql_amd import ops
    p = make_linear_problem(m, k, n, seed=m + k + n)
    x, b, s = to_gpu(p, gpu)
    y32 = ops.w4a16_gemm_ex(x, b, s, workspace_for(n, gpu), m, n, k, out_f32=True, flags=_flags(upw))
    assert np.abs(y32.cpu().numpy() - reference_product(p, exact=True)).max() < 2e-4
    assert torch.equal(ops.w4a16_gemm_ex(x, b, s, workspace_for(n, gpu), m, n, k, flags=_flags(upw)), y32.half())


def _layer(gpu, k, n, seed):
    gen = torch.Generator(device=gpu).manual_seed(seed)
    b = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=gpu, generator=gen)
    s = (0.004 + 0.016 * torch.rand((k // 128, n), device=gpu, generator=gen)).half()
    return gen, b, s


@pytest.mark.parametrize("m", [16, 32, 48, 64])
def test_every_weight_bit_exact(gpu, m):
    """one-hot rows: every output is one product 1 * w, for scales inside the short expansion's range, at its end, beyond it,
    zero, negative and subnormal, mixed inside a unit"""
    from uniql_amd import ops
    k, n = 2304, 128
    gen, b, s = _layer(gpu, k, n, m)
    s[1, 5], s[1, 64] = 0.0624, 0.0625
    s[3], s[4, 7], s[5, :64], s[6] = 0.7, 300.0, 0.0, 1e-4
    s[7, 3], s[8, 70], s[9] = -0.01, -0.5, 3e-7
    w = ops.w4a16_dequant(b, s, n, k)
    rows = torch.arange(m, device=gpu) * 37 + 5
    for first in range(0, k, 640):
        at = (rows + first) % k
        x = torch.zeros((m, k), dtype=torch.float16, device=gpu)
        x[torch.arange(m, device=gpu), at] = 1.0
        y = ops.w4a16_gemm_ex(x, b, s, workspace_for(n, gpu), m, n, k, out_f32=True, flags=_flags(1))
        assert torch.equal(y, w[at].float())


@pytest.mark.parametrize("m,k,n,upw", [(12, 2048, 384, 1), (30, 4096, 256, 1), (45, 2304, 384, 1), (60, 1280, 256, 5)])
def test_epilogues_and_inputs(gpu, m, k, n, upw):
    """bit for bit what the plain product and torch's operators on it give"""
    from uniql_amd import ops
    gen, b, s = _layer(gpu, k, n, m + k)
    ws, flags = workspace_for(n, gpu), _flags(upw)
    x = torch.randn((m, k + 8), device=gpu, generator=gen).half()[:, :k]     # strided rows
    y = ops.w4a16_linear(x, b, s, ws, n, k, flags=flags)
    assert torch.equal(y, ops.w4a16_linear(x.contiguous(), b, s, ws, n, k, flags=flags))
    bias = torch.randn(n, device=gpu, generator=gen).half()
    n_out = n - 136                       # the last strip holds padding columns only
    wide = torch.randn((m, n_out + 16), device=gpu, generator=gen).half()
    stream = wide[:, 8:8 + n_out]
    want = (stream.float() + (y[:, :n_out].float() + bias[:n_out].float()).half().float()).half()
    got = ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, bias=bias[:n_out].clone(), residual=stream, out=stream, flags=flags)
    assert got.data_ptr() == stream.data_ptr() and torch.equal(got, want)
    assert torch.equal(ops.w4a16_gemm_ex(x, b, s, ws, m, n, k, transpose_out=True, flags=flags)[:, :m].t(), y)
    r = torch.relu(y.float())
    assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, relu2=True, flags=flags), (r * r).half())
    # gated pairs: the same roundings as the tiled kernel's epilogue on the same fp16 gate and up values
    pair = ops.w4a16_linear(x, b, s, ws, n, k, silu_mul=True, flags=flags)
    gate, up = y.view(m, n // 128, 2, 64).unbind(2)
    want = (torch.nn.functional.silu(gate.float()).half().float() * up.float()).half().reshape(m, n // 2)
    # expf and torch's exp differ in the last bit now and then: one fp16 step of the activation
    assert torch.all((pair.float() - want.float()).abs() <= 2 * 2 ** -10 * want.float().abs() + 2 ** -24)
    assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, silu_mul=True, out_features=n // 2 - 72, flags=flags), pair[:, :n // 2 - 72])
    # an input shorter than K: zeros behind it
    padded = x.clone()
    padded[:, k - 40:] = 0
    assert torch.equal(ops.w4a16_linear(x[:, :k - 40].contiguous(), b, s, ws, n, k, flags=flags),
                       ops.w4a16_linear(padded, b, s, ws, n, k, flags=flags))
    # one scale per column
    one = (0.004 + 0.016 * torch.rand((1, n), device=gpu, generator=gen)).half()
    y1 = ops.w4a16_gemm_ex(x.contiguous(), b, one, ws, m, n, k, out_f32=True, flags=flags)
    ref = x.double() @ ops.w4a16_dequant(b, one, n, k).double()
    assert (y1.double() - ref).abs().max() < 2e-4


@pytest.mark.parametrize("m", [16, 40])
def test_nan_and_infinite_sums_cross_the_split(gpu, m):
    """every partial tile travels as fp32: NaN stays NaN, infinities of both signs from different workgroups give NaN"""
    from uniql_amd import ops
    k, n = 2048, 128
    gen, b, s = _layer(gpu, k, n, 5)
    x = torch.randn((m, k), device=gpu, generator=gen).half()
    x[1, 3] = float("nan")
    x[2, 7], x[2, 1500] = float("inf"), float("inf")
    y = ops.w4a16_gemm_ex(x, b, s, workspace_for(n, gpu), m, n, k, out_f32=True, flags=_flags(1))
    assert torch.isnan(y[1]).all()
    ref = x.double() @ ops.w4a16_dequant(b, s, n, k).double()
    assert torch.equal(torch.isnan(y[2]), torch.isnan(ref[2])) and torch.equal(torch.isinf(y[2]), torch.isinf(ref[2]))
    rest = torch.ones(m, dtype=torch.bool, device=gpu)
    rest[1:3] = False
    assert (y[rest].double() - ref[rest]).abs().max() < 2e-4


@pytest.mark.parametrize("m", [16, 30, 48, 64])
def test_infinite_values_meet_scales_of_the_long_expansion(gpu, m):
    """a group whose scales are beyond the short expansion's range: an infinite value times its weights is infinite, not NaN"""
    from uniql_amd import ops
    k, n = 1536, 128
    gen, b, s = _layer(gpu, k, n, 6)
    s[0, 9], s[5] = 0.5, 0.25
    x = torch.randn((m, k), device=gpu, generator=gen).half()
    x[2, 7], x[3, 5 * 128 + 70], x[m - 1, 11 * 128] = float("inf"), float("-inf"), float("inf")
    w = ops.w4a16_dequant(b, s, n, k)
    for scale, weight in ((s, w), (s[5:6].clone(), ops.w4a16_dequant(b, s[5:6].clone(), n, k))):
        y = ops.w4a16_gemm_ex(x, b, scale, workspace_for(n, gpu), m, n, k, out_f32=True, flags=_flags(2))
        ref = x.double() @ weight.double()
        assert torch.isinf(ref[2]).any() and torch.isinf(ref[3]).any()
        assert torch.equal(torch.isnan(y), torch.isnan(ref))
        assert torch.equal(torch.where(torch.isinf(y), y, 0.0).double(), torch.where(torch.isinf(ref), ref, 0.0))
        finite = torch.isfinite(ref)
        # fp32 sums of 1536 products, |x w| < 5 x 4: far less than 1536 2^-24 times their absolute sum
        bound = 1536 * 2.0 ** -24 * (torch.nan_to_num(x.double(), posinf=0.0, neginf=0.0).abs() @ weight.double().abs())
        assert torch.all(((y.double() - ref).abs() <= bound + 1e-6)[finite])


# sizes of this kernel: one and several groups a wave, K split into 2 to 9 and not at all, each row class; the last two where its
# fastest plan would add longer chains than the tiled kernel's
@pytest.mark.parametrize("m,k,n", [(15, 4480, 512), (12, 1920, 1024), (16, 8192, 4096), (13, 512, 13056), (9, 14336, 4096), (10, 6144, 512),
                                   (29, 4864, 7168), (23, 12800, 1536), (17, 3328, 8704), (40, 4096, 28672), (48, 4096, 4096), (35, 12288, 1280), (40, 9216, 3072),
                                   (56, 6784, 2048), (53, 6400, 256), (56, 8192, 512)])
def test_sums_are_as_exact_as_the_other_kernels(gpu, m, k, n):
    """distance from float64 in front of the fp16 rounding against that of the kernel which took such calls before: the
    streaming kernel, whose partial sums meet as integers, up to 16 rows, the tiled kernel above.  Both round fp32
    sums of the same exact products; with a few thousand outputs the two distances are known to about 1 %."""
    from uniql_amd import ops
    gen, b, s = _layer(gpu, k, n, 77)
    x = torch.randn((m, k), device=gpu, generator=gen)
    x[:, torch.randint(0, k, (max(1, k // 512),), device=gpu, generator=gen)] *= 16.0   # a few much larger channels
    x = x.half()
    ref = x.double() @ ops.w4a16_dequant(b, s, n, k).double()
    ws = workspace_for(n, gpu)

    def distance(flags):
        return float((ops.w4a16_gemm_ex(x, b, s, ws, m, n, k, out_f32=True, flags=flags).double() - ref).norm() / ref.norm())

    assert distance(0) <= 1.03 * distance(F_FORCE_SKINNY if m <= 16 else F_FORCE_TILED)


def test_calls_take_it_and_replay(gpu):
    """the calls that the library hands to it by itself, recorded once and replayed between eager calls that share
    nothing with the graph but the stream's buffers; every replay and every eager repeat gives the same bits"""
    from uniql_amd import ops
    layers = [(16, 4096, 4096), (24, 4096, 6144), (48, 14336, 4096), (40, 4000, 4096)]
    prepared = []
    for i, (m, k, n) in enumerate(layers):
        kp = (k + 127) // 128 * 128
        gen, b, s = _layer(gpu, kp, n, i)
        x = torch.randn((m, k), device=gpu, generator=gen).half()
        prepared.append((x, b, s, workspace_for(n, gpu), n, kp))

    def step():
        return [ops.w4a16_linear(*p) for p in prepared]

    want = step()
    for (x, b, s, ws, n, kp), y, (m, k, _) in zip(prepared, want, layers):
        ref = x.double() @ ops.w4a16_dequant(b, s, n, kp)[:k].double()
        check_layer_output_torch(y, ref)
        assert torch.equal(y, ops.w4a16_linear(x, b, s, ws, n, kp, flags=_flags(0)))   # its own plan: the same kernel
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(4):
        for y in out:
            y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
        assert all(torch.equal(a, b) for a, b in zip(step(), want))
