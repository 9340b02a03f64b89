"""The tiled kernel's exchange of K splits requests the partial tiles in batches of 2, 4 or 8, depending on the tile height
and on the splits that are left: every batch size, whole and with a remainder, plain and as gated pairs."""
import numpy as np
import pytest
import torch

from tests.helpers import make_linear_problem, reference_product, to_gpu, workspace_for

pytestmark = pytest.mark.gpu
F_TILED = 4


@pytest.mark.parametrize("mt,quartets", [(1, 1), (1, 2), (2, 1), (2, 2), (3, 1), (4, 1)])
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 8, 9, 18])
def test_every_batch_of_partial_tiles(gpu, mt, quartets, splits):
    from uniql_amd import ops
    m, k, n = 131, 36 * 128, 256   # the last M tile is ragged for every height
    p = make_linear_problem(m, k, n, seed=splits)
    x, b, s = to_gpu(p, gpu)
    ws = workspace_for(n, gpu)
    flags = F_TILED | (splits << 8) | (mt << 16) | (quartets << 20)
    ref = reference_product(p, exact=True)
    y32 = ops.w4a16_gemm_ex(x, b, s, ws, m, n, k, out_f32=True, flags=flags).cpu().numpy()
    assert np.abs(y32 - ref).max() < 3e-4   # as the other K split tests: fp32 sums over K = 4608
    # the pairs' sums are the plain call's: gate and up are columns c and c + 64 of a strip
    pair = ops.w4a16_linear(x, b, s, ws, n, k, out_features=n // 2, silu_mul=True, out_f32=True, flags=flags).cpu().double()
    y = torch.from_numpy(y32).double().reshape(m, n // 128, 2, 64)
    want = torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]
    # silu and the product in fp32: a few roundings of values up to |gate up|
    assert float((pair.reshape_as(want) - want).abs().max()) < 1e-6 * float(want.abs().max()) + 1e-6
    assert all(int(buf.count_nonzero()) == 0 for buf in ops._accum_cache.values())
