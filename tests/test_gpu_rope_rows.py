"""Rotary kernels at the edges of their rules: the kernel that gathers per pair up to 191 tokens, tables in LDS from 128 or 192 on,
a token's heads in one workgroup or in several, heads of one pair (quotients by division), one table row for all sequences."""
import numpy as np
import pytest
import torch

from oracle import uniql_oracle as O
from tests.test_gpu_rope_embedding import pruned_indices
from tests.test_oracle_fused_rope import rope_tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hk,s,d,D", [(1, 16, 2, 191, 96, 256), (1, 16, 2, 192, 96, 256), (2, 32, 32, 140, 64, 128),
                                           (3, 6, 2, 100, 14, 32), (1, 28, 4, 300, 6, 128), (260, 4, 2, 1, 8, 16), (70, 8, 1, 1, 20, 32),
                                           (1, 5, 5, 7, 2, 16), (1, 6, 3, 290, 2, 16), (3, 40, 8, 20, 108, 128), (1, 96, 3, 2, 250, 256),
                                           (1, 32, 32, 127, 108, 128), (1, 32, 32, 128, 108, 128), (2, 64, 64, 97, 90, 128),
                                           (1, 48, 12, 333, 112, 128), (1, 24, 24, 200, 128, 128), (1, 8, 1, 1024, 64, 64),
                                           (1, 8, 4, 1025, 20, 32), (1, 40, 4, 1024, 16, 32), (1, 14, 14, 130, 6, 16)])
@pytest.mark.parametrize("index_dtype", [torch.uint8, torch.int64, torch.int32])
def test_rows_and_heads(gpu, b, hq, hk, s, d, D, index_dtype):
    from uniql_amd import ops
    rng = np.random.default_rng(b + s + d)
    q = rng.standard_normal((b, s, hq, d)).astype(np.float16)
    k = rng.standard_normal((b, s, hk, d)).astype(np.float16)
    cos, sin, _ = rope_tables(s, D, batch=b if b == 2 else 1)
    idx = pruned_indices(hk, d, D, seed=d)
    want_q, want_k = O.rope_indices(q.transpose(0, 2, 1, 3), k.transpose(0, 2, 1, 3), cos, sin, idx)
    qt, kt = torch.from_numpy(q).to(gpu), torch.from_numpy(k).to(gpu)
    ops.rope_indices_(qt, kt, torch.from_numpy(cos).to(gpu), torch.from_numpy(sin).to(gpu),
                      torch.from_numpy(idx).to(index_dtype).to(gpu))
    assert np.array_equal(qt.cpu().numpy().view(np.uint16), want_q.transpose(0, 2, 1, 3).view(np.uint16))
    assert np.array_equal(kt.cpu().numpy().view(np.uint16), want_k.transpose(0, 2, 1, 3).view(np.uint16))


# halves of a workgroup's heads that are just enough for a workgroup of their own, and just not: 128 work items; 768 entries beyond 1024 tokens
@pytest.mark.parametrize("b,hq,hk,s,d,D", [(1, 32, 32, 1030, 48, 64), (1, 32, 32, 1030, 46, 64), (1, 32, 32, 1024, 64, 128), (1, 30, 30, 200, 64, 128),
                                           (1, 40, 40, 300, 64, 128), (1, 40, 10, 1025, 128, 128), (3, 48, 12, 343, 128, 128)])
def test_halves_that_are_enough_for_a_workgroup(gpu, b, hq, hk, s, d, D):
    test_rows_and_heads(gpu, b, hq, hk, s, d, D, torch.uint8)
