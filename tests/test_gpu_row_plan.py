"""96-row tiles of the 128-column kernel, and prefill calls whose rows run as two launches."""
import numpy as np
import pytest
import torch

from tests.helpers import check_layer_output_torch, make_linear_problem, reference_product, to_gpu, workspace_for

pytestmark = pytest.mark.gpu

F_FORCE_TILED, TILE96 = 1 << 2, 3 << 16


@pytest.mark.parametrize("m,k,n,splits", [(1, 128, 128, 0), (33, 384, 128, 1), (95, 256, 256, 0), (96, 640, 384, 2),
                                          (97, 512, 256, 1), (200, 1024, 128, 3), (333, 896, 384, 0)])
def test_96_row_tiles(gpu, m, k, n, splits):
    """the edges of the tile (one row, a row less and more than a tile, empty M tiles inside the last one), the
    shortest K, K splits of unequal length; the fp32 value is held to the bound of the other tile heights"""
    from uniql_amd import ops
    p = make_linear_problem(m, k, n, seed=m + k + n)
    x, b, s = to_gpu(p, gpu)
    flags = F_FORCE_TILED | TILE96 | (splits << 8)
    y32 = ops.w4a16_gemm_ex(x, b, s, workspace_for(n, gpu), m, n, k, out_f32=True, flags=flags)
    assert np.abs(y32.cpu().numpy() - reference_product(p, exact=True)).max() < 2e-4
    y16 = ops.w4a16_gemm_ex(x, b, s, workspace_for(n, gpu), m, n, k, flags=flags)
    assert torch.equal(y16, y32.half())


def _layer(gpu, k, n, seed):
    gen = torch.Generator(device=gpu).manual_seed(seed)
    b = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 16, 2 * n), dtype=torch.int32, device=gpu, generator=gen)
    s = (0.004 + 0.016 * torch.rand((k // 128, n), device=gpu, generator=gen)).half()
    return gen, b, s


@pytest.mark.parametrize("m,k,n,head", [(1100, 4096, 28672, 1024), (1100, 14336, 4096, 1024), (1057, 11008, 4096, 1024)])
def test_rows_in_two_launches(gpu, m, k, n, head):
    """The rows behind `head` are a launch of their own: every epilogue's pointers move with them, and the
    values are those of a call on these rows alone (the same plan, so the same bits)."""
    from uniql_amd import ops
    gen, b, s = _layer(gpu, k, n, m + k)
    ws = workspace_for(n, gpu)
    x = torch.randn((m, k + 8), device=gpu, generator=gen).half()[:, :k]     # strided rows
    bias = torch.randn(n, device=gpu, generator=gen).half()
    n_out = n - 40
    y = ops.w4a16_linear(x, b, s, ws, n, k)
    assert torch.equal(y[head:], ops.w4a16_linear(x[head:], b, s, ws, n, k))
    ref = torch.cat([part.double() @ ops.w4a16_dequant(b, s, n, k).double() for part in x.split(256)])
    check_layer_output_torch(y, ref)
    # output cut, bias, residual overwritten in place, rows of a wider buffer
    wide = torch.randn((m, n_out + 16), device=gpu, generator=gen).half()
    stream = wide[:, 8:8 + n_out]
    want = (stream.float() + (y[:, :n_out].float() + bias[:n_out].float()).half().float()).half()
    got = ops.w4a16_linear(x, b, s, ws, n, k, out_features=n_out, bias=bias[:n_out].clone(), residual=stream, out=stream)
    assert got.data_ptr() == stream.data_ptr() and torch.equal(got, want)
    # transposed, fp32, squared ReLU
    t = ops.w4a16_gemm_ex(x, b, s, ws, m, n, k, transpose_out=True)
    assert torch.equal(t[:, :m].t(), y)
    y32 = ops.w4a16_linear(x, b, s, ws, n, k, out_f32=True)
    assert torch.equal(y32.half(), y)
    r = torch.relu(y.float())
    assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, relu2=True), (r * r).half())
    # behind a rotation the copy of the activations and the partial tiles share the temporary area
    block = 256
    rotated = ops.hadamard_blockwise(x.contiguous(), block ** -0.5, block)
    assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k, had_block=block, had_scale=block ** -0.5),
                       ops.w4a16_linear(rotated, b, s, ws, n, k))


def test_two_launches_of_a_gated_pair(gpu):
    from uniql_amd import ops
    m, k, n = 1100, 4096, 28672
    gen, b, s = _layer(gpu, k, n, 3)
    ws = workspace_for(n, gpu)
    x = torch.randn((m, k), device=gpu, generator=gen).half()
    y = ops.w4a16_linear(x, b, s, ws, n, k, silu_mul=True)
    assert torch.equal(y[1024:], ops.w4a16_linear(x[1024:], b, s, ws, n, k, silu_mul=True))
    assert torch.equal(y[:1024], ops.w4a16_linear(x[:1024], b, s, ws, n, k, silu_mul=True))


def test_two_launches_replayed(gpu):
    """a graph's replays give the eager result, with eager calls on the same stream's accumulator in between"""
    from uniql_amd import ops
    m, k, n = 1030, 11008, 4096
    gen, b, s = _layer(gpu, k, n, 7)
    ws = workspace_for(n, gpu)
    x = torch.randn((m, k), device=gpu, generator=gen).half()
    want = ops.w4a16_linear(x, b, s, ws, n, k)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.w4a16_linear(x, b, s, ws, n, k)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.w4a16_linear(x, b, s, ws, n, k)
    for _ in range(4):
        out.zero_()
        graph.replay()
        assert torch.equal(out, want)
        assert torch.equal(ops.w4a16_linear(x, b, s, ws, n, k), want)
