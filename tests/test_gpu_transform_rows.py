"""Transforms: workgroups that take several rows of a composite or power-of-two width one after the other, rows that hold
infinities or NaN, and every tile width of the column transform."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# widths of one, two, four and eight chunks of 128 values; more rows than the chip holds workgroups, an odd number of them
@pytest.mark.parametrize("dim,base,rows", [(1536, 12, 3001), (3072, 12, 1401), (3584, 28, 1501), (5120, 40, 1157), (10240, 20, 781),
                                           (14336, 28, 1103), (28672, 28, 523), (20480, 40, 517)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_rows_behind_the_first(gpu, dim, base, rows, dtype):
    """a row's result does not depend on how many rows the call has or which comes before it"""
    from uniql_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(dim)
    x = torch.randn((rows, dim), device=gpu, generator=gen).to(dtype)
    y = ops.hadamard_composite(x, dim ** -0.5, base)
    for first in (0, 250, rows - 200):
        assert torch.equal(y[first:first + 200], ops.hadamard_composite(x[first:first + 200].clone(), dim ** -0.5, base))
    # rows that are not on the 16-byte grid take the kernel that moves single values
    odd = torch.empty(64 * dim + 1, dtype=dtype, device=gpu)[1:].view(64, dim)
    odd.copy_(x[rows - 64:])
    assert torch.equal(ops.hadamard_composite(odd, dim ** -0.5, base), y[rows - 64:])


# one to sixteen waves' worth of blocks; more rows than the chip holds workgroups, an odd number of them
@pytest.mark.parametrize("dim,rows", [(1024, 4397), (2048, 2301), (4096, 2305), (8192, 1101), (16384, 577), (32768, 301)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_power_of_two_rows(gpu, dim, rows, dtype):
    """a row's result does not depend on how many rows the call has, which comes before it, or whether it
    starts on the 16-byte grid; an infinity stays in its row"""
    from uniql_amd import ops
    gen = torch.Generator(device=gpu).manual_seed(dim)
    x = torch.randn((rows, dim), device=gpu, generator=gen).to(dtype)
    y = ops.hadamard_blockwise(x, dim ** -0.5, dim)
    for first in (0, 250, rows - 50):
        assert torch.equal(y[first:first + 50], ops.hadamard_blockwise(x[first:first + 50].clone(), dim ** -0.5, dim))
    odd = torch.empty(40 * dim + 1, dtype=dtype, device=gpu)[1:].view(40, dim)
    odd.copy_(x[rows - 40:])
    assert torch.equal(ops.hadamard_blockwise(odd, dim ** -0.5, dim), y[rows - 40:])
    x[rows - 2, dim - 1] = float("inf")
    again = ops.hadamard_blockwise(x, dim ** -0.5, dim)
    assert not torch.isfinite(again[rows - 2]).any()
    assert torch.equal(again[:rows - 2], y[:rows - 2]) and torch.equal(again[rows - 1], y[rows - 1])


@pytest.mark.parametrize("dim,base", [(3584, 28), (5120, 40)])
def test_infinities_and_nan_stay_in_their_row(gpu, dim, base):
    from uniql_amd import ops
    x = torch.randn((1200, dim), device=gpu, generator=torch.Generator(device=gpu).manual_seed(1)).half()
    clean = ops.hadamard_composite(x, dim ** -0.5, base)
    x[1, 3], x[600, 7], x[1199, dim - 1] = float("nan"), float("inf"), float("-inf")
    y = ops.hadamard_composite(x, dim ** -0.5, base)
    hit = torch.zeros(1200, dtype=torch.bool, device=gpu)
    hit[[1, 600, 1199]] = True
    assert torch.isnan(y[1]).all() and not torch.isfinite(y[600]).any() and not torch.isfinite(y[1199]).any()
    assert torch.equal(y[~hit], clean[~hit])


# every tile width: four, eight and sixteen waves, at the edges of the rules that choose them; a last tile that is cut
@pytest.mark.parametrize("rows,cols,dtype", [(1024, 4096, torch.float16), (1024, 8184, torch.float16), (1024, 8200, torch.bfloat16),
                                             (2048, 4104, torch.float16), (4096, 4088, torch.float32), (4096, 4104, torch.float32),
                                             (4096, 264, torch.float32), (2048, 8, torch.float32),
                                             (4096, 2552, torch.float16), (4096, 2560, torch.float16), (4096, 2568, torch.bfloat16),
                                             (4096, 4352, torch.float16), (4096, 4360, torch.float16), (4096, 6152, torch.bfloat16),
                                             (4096, 8200, torch.float16)])
def test_column_tiles(gpu, rows, cols, dtype):
    """bit for bit the row transform between two transposed copies; an infinity stays in its column"""
    from uniql_amd import ops
    x = torch.randn((rows, cols), device=gpu, generator=torch.Generator(device=gpu).manual_seed(cols)).to(dtype)
    x[5, cols - 3] = float("inf")
    y = ops.hadamard_columns(x, rows ** -0.5)
    want = ops.hadamard_blockwise(x.t().contiguous(), rows ** -0.5, rows).t()
    clean = torch.arange(cols, device=gpu) != cols - 3
    assert torch.equal(y[:, clean], want[:, clean])
    assert not torch.isfinite(y[:, cols - 3]).any()
