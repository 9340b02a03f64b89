"""The kernels that produce a 4-bit model's tensors, where their paths change: scales and weights outside of what the
quantiser's three-instruction quotient covers, the transforms' types and widths, the column transform, the cuts of packed
matrices."""
import numpy as np
import pytest
import torch

from oracle import uniql_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("given", [False, True])
def test_quantize_outside_the_fast_quotient(gpu, given):
    """Columns with zero, negative, subnormal, tiny or huge scales, infinite weights and quotients at both ends of fp16,
    ties included, beside ordinary ones: bit for bit the oracle's arithmetic."""
    from uniql_amd import ops
    g = torch.Generator().manual_seed(17)
    n, k = 192, 392
    w = (torch.randn(n, k, generator=g) * 0.05).half()
    w[5, 130:250] = 0
    w[6] = 0
    w[7] *= 2.0 ** -20
    w[8, 3] = float("inf")
    w[9] = (torch.arange(k) % 31 - 15).half() * 0.25          # quotients on the halves
    w[10] = 60000.0
    scales = None
    if given:
        scales = (torch.rand(4, n, generator=g) * 0.02 + 0.004).half()
        scales[1, 5] = 0
        scales[:, 9] = 0.5
        scales[0, 11], scales[1, 11], scales[2, 11], scales[3, 11] = -0.01, 2.0 ** -24, 2.0 ** -14, 1000.0
        scales[:, 10] = torch.tensor([1.0, 1.5, 0.5, 1.9]).half()   # quotients 60000, 40000, overflow, 31578
        w[12] = 30000.0
        scales[:, 12] = torch.tensor([0.9, 0.92, 0.5, 0.45]).half()
    _, o_packed, o_scale = O.w4a16_quantize(w.t().contiguous(), 128, scales, 64)
    packed, scale = ops.w4a16_quantize(w.to(gpu), None if scales is None else scales.to(gpu), pad_out=64)
    assert torch.equal(packed.cpu(), o_packed)
    assert np.array_equal(scale.cpu().numpy().view(np.uint16), o_scale.numpy().view(np.uint16))


@pytest.mark.parametrize("view", ["offset", "odd_stride"])
def test_quantize_rows_that_are_not_16_byte_aligned(gpu, view):
    from uniql_amd import ops
    g = torch.Generator().manual_seed(3)
    big = (torch.randn(128, 517, generator=g) * 0.1).half().to(gpu)
    w = big[:, 3:387] if view == "offset" else big[:, :384]
    got, want = ops.w4a16_quantize(w), ops.w4a16_quantize(w.contiguous())
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("given", [False, True])
def test_quantize_into_buffers_off_the_16_byte_grid(gpu, given):
    """the C entry asks for 4-byte words and 2-byte scales only"""
    from uniql_amd import _capi, ops
    g = torch.Generator().manual_seed(4)
    n, k = 192, 392
    w = (torch.randn(n, k, generator=g) * 0.1).half().to(gpu)
    scales = (torch.rand(4, n, generator=g) * 0.02 + 0.004).half().to(gpu) if given else None
    packed, scale = ops.w4a16_quantize(w, scales, pad_out=64)
    words = torch.full((packed.numel() + 2,), 7, dtype=torch.int32, device=gpu)
    halves = torch.full((scale.numel() + 2,), 7, dtype=torch.float16, device=gpu)
    code = _capi.load().uniql_w4a16_quantize(w.data_ptr(), k, scales.data_ptr() if given else None, words[1:].data_ptr(),
                                             halves[1:].data_ptr(), n, k, 256, 512, torch.cuda.current_stream().cuda_stream)
    assert code == 0
    assert torch.equal(words[1:-1], packed.flatten()) and torch.equal(halves[1:-1], scale.flatten())
    assert words[0] == words[-1] == 7 and halves[0] == halves[-1] == 7


def _as(t, dtype):
    """numpy float32 of what the kernel's rounding to `dtype` gives for a float32 tensor"""
    return t.to(dtype).float().numpy()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("block", [64, 128, 256, 2048, 4096, 8192, 16384, 32768])
def test_transform_in_every_type_and_width(gpu, dtype, block):
    from uniql_amd import ops
    x = torch.randn(3, 2 * block if block <= 4096 else block, generator=torch.Generator().manual_seed(block)).to(dtype)
    y = ops.hadamard_blockwise(x.to(gpu), block ** -0.5, block)
    want = torch.from_numpy(O.fwht(x.float().numpy(), 1.0, block=block)) * torch.tensor(block ** -0.5, dtype=torch.float32)
    assert np.array_equal(y.float().cpu().numpy(), _as(want, dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(1024, 8), (1024, 264), (2048, 8), (2048, 1048), (4096, 8), (4096, 136)])
def test_column_transform(gpu, dtype, rows, cols):
    """One tile and less, tiles that do not divide the width, more tiles than XCDs: the row transform of the transpose."""
    from uniql_amd import ops
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows + cols)).to(dtype).to(gpu)
    y = ops.hadamard_columns(x, rows ** -0.5)
    assert torch.equal(y, ops.fast_hadamard_transform(x.t().contiguous(), rows ** -0.5).t())
    assert ops.hadamard_columns(x[:, :4].contiguous(), 1.0) is None and ops.hadamard_columns(x[:512].contiguous(), 1.0) is None


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim", [12 * 128, 12 * 2048, 20 * 64, 20 * 1024, 28 * 128, 28 * 1024, 40 * 512, 40 * 1024])
def test_composite_transform_widths(gpu, dtype, dim):
    """The smallest and largest width of the vector kernel for each base, and one of the kernel it leaves the rest to."""
    from uniql_amd import ops
    base, scale = O.had_variant(dim)
    x = torch.randn(5, dim, generator=torch.Generator().manual_seed(dim)).to(dtype)
    y = ops.hadamard_composite(x.to(gpu), scale, base)
    want = torch.from_numpy(O.fwht_composite(x.float().numpy(), 1.0, base)) * torch.tensor(scale, dtype=torch.float32)
    assert np.array_equal(y.float().cpu().numpy(), _as(want, dtype))


def test_hadlinear_leaves_the_layer_it_is_made_from_alone(gpu):
    from uniql_amd.quantize.quant_linear_layers import HadLinear
    g = torch.Generator().manual_seed(2)
    lin = torch.nn.Linear(256, 1024, bias=False).half().to(gpu)
    lin.weight.data = torch.randn(1024, 256, generator=g).half().to(gpu)
    before = lin.weight.data.clone()
    fused = HadLinear(lin, input_transform=True, output_transform=True, fuse_had=True)
    want = O.hadlinear_fused_weight(before.cpu().numpy(), True, True)
    assert np.array_equal(fused.weight.data.cpu().numpy().view(np.uint16), want.view(np.uint16))
    plain = HadLinear(lin, input_transform=False, output_transform=False, fuse_had=True)
    assert torch.equal(plain.weight.data, before) and plain.weight.data_ptr() != lin.weight.data_ptr()
    assert torch.equal(lin.weight.data, before)


def _packed_layer(gpu, k, n, g):
    from uniql_amd import ops
    codes = torch.randint(0, 16, (k, n), generator=g).to(torch.uint8).to(gpu)
    scales = (torch.rand(k // 128, n, generator=g) * 0.02 + 0.004).half().to(gpu)
    scales[:, 3] = 0
    return ops.w4a16_pack(codes, scales), codes, scales


@pytest.mark.parametrize("k,k_real", [(128, 128), (256, 250), (1408, 1399)])
@pytest.mark.parametrize("runs,n_scaled,pad", [
    ([(0, 1, 256, 256, 256, 0)], 200, 0),                          # a prefix: whole chunks
    ([(64, 1, 320, 320, 320, 0)], 320, 64),                        # whole chunks from the second one on
    ([(0, 3, 100, 38, 19, 31)], 114, 14),                          # two pieces of every head
    ([(0, 2, 33, 17, 17, 0), (5, 0, 9, 3, 3, 0), (66, 4, 40, 40, 20, 0), (511, 1, 1, 1, 1, 0), (300, 1, 11, 6, 2, -3)], 201, 55),
])
def test_cut_columns(gpu, k, k_real, runs, n_scaled, pad):
    """Rows that do not end with a group, runs inside and across chunks, padding: packing the indexed codes."""
    from uniql_amd import ops
    (w, s), codes, scales = _packed_layer(gpu, k, 512, torch.Generator().manual_seed(k))
    cols = [base + u * full + i + (skip if i >= split else 0)
            for base, units, full, kept, split, skip in runs for u in range(units) for i in range(kept)]
    kept_codes, kept_scales = codes[:, cols], scales[:, cols]
    kept_codes[k_real:] = 0
    kept_scales[:, n_scaled:] = 0
    want = ops.w4a16_pack(kept_codes, kept_scales, pad_out=pad)
    got = ops.w4a16_cut_columns(w, s, 512, k, runs, k_real=k_real, n_scaled=n_scaled, pad_out=pad)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    with pytest.raises(RuntimeError):
        ops.w4a16_cut_columns(w, s, 512, k, [(1, 1, 512, 512, 512, 0)])


def test_cut_columns_many_groups_per_workgroup(gpu):
    from uniql_amd import ops
    k, n = 128 * 131, 4096
    (w, s), codes, scales = _packed_layer(gpu, k, n, torch.Generator().manual_seed(5))
    runs = [(0, 32, 128, 126, 63, 1)]
    cols = torch.tensor([128 * u + i + (i >= 63) for u in range(32) for i in range(126)], device=gpu)
    want = ops.w4a16_pack(codes[:, cols], scales[:, cols], pad_out=64)
    got = ops.w4a16_cut_columns(w, s, n, k, runs, pad_out=64)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_cuts_and_quantising_refuse_what_no_call_can_take(gpu):
    """runs that are not six values each, widths that 32 bits do not hold: an error with its reason, nothing allocated or launched"""
    from uniql_amd import ops
    (w, s), _, _ = _packed_layer(gpu, 256, 512, torch.Generator().manual_seed(1))
    x = torch.zeros((512, 256), dtype=torch.float16, device=gpu)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    with pytest.raises(RuntimeError, match="six values"):
        ops.w4a16_cut_columns(w, s, 512, 256, [(0, 1, 512, 512, 512)])
    for width in (1 << 31, -(1 << 32)):
        with pytest.raises(RuntimeError, match="kept width"):
            ops.w4a16_cut_columns(w, s, 512, 256, [(0, 1, 512, 512, 512, 0)], pad_out=width)
        with pytest.raises(RuntimeError, match="kept sizes"):
            ops.w4a16_cut_rows(w, s, 512, 256, 1, 256, 256, 512, pad_out=width)
        with pytest.raises(RuntimeError, match="larger than a call can take"):
            ops.w4a16_quantize(x, None, pad_out=width)
    assert torch.cuda.max_memory_allocated() == before


@pytest.mark.parametrize("n,n_real,pad", [(128, 128, 0), (256, 200, 56), (256, 130, 126), (256, 60, 324)])
@pytest.mark.parametrize("k,units,full,kept", [(256, 1, 0, 129), (512, 4, 128, 108), (1280, 10, 128, 77), (1280, 37, 33, 31)])
@pytest.mark.parametrize("per_column", [False, True])
def test_cut_rows(gpu, n, n_real, pad, k, units, full, kept, per_column):
    """Kept rows over group and word boundaries, odd widths: quantising the gathered dequantised rows."""
    from uniql_amd import ops
    (w, s), _, _ = _packed_layer(gpu, k, n, torch.Generator().manual_seed(n + k))
    if per_column:
        s = s[:1].contiguous()
    rows = torch.tensor([u * full + i for u in range(units) for i in range(kept)], device=gpu)
    want = ops.w4a16_quantize(ops.w4a16_dequant(w, s, n, k)[rows][:, :n_real].t().contiguous(), None, pad_out=pad)
    got = ops.w4a16_cut_rows(w, s, n, k, units, full, kept, n_real, pad_out=pad)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    with pytest.raises(RuntimeError):
        ops.w4a16_cut_rows(w, s, n, k, 2, k, 100, n_real, pad_out=pad)


# a run of single columns (whose inverse does not fit 32 bits), pairs, odd lengths, a prefix, padding columns inside a chunk
@pytest.mark.parametrize("runs", [[(0, 100, 5, 1, 1, 0)], [(3, 90, 4, 2, 1, 1)], [(0, 7, 71, 67, 30, 4), (500, 1, 12, 11, 11, 0)], [(64, 1, 448, 448, 448, 0)]])
def test_cut_columns_quotients(gpu, runs):
    from uniql_amd import ops
    k, n = 384, 512
    (w, s), codes, scales = _packed_layer(gpu, k, n, torch.Generator().manual_seed(9))
    cols = torch.tensor([base + u * full + i + (skip if i >= split else 0) for base, units, full, kept, split, skip in runs
                         for u in range(units) for i in range(kept)], device=gpu)
    pad = -len(cols) % 256
    want = ops.w4a16_pack(codes[:, cols], scales[:, cols], pad_out=pad)
    got = ops.w4a16_cut_columns(w, s, n, k, runs, pad_out=pad)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


# even runs an even distance apart, whose rows are expanded two at a time: single pairs, runs that overlap or follow each other,
# runs off the words' and groups' grids, one long run
@pytest.mark.parametrize("k,units,full,kept", [(1024, 255, 4, 2), (512, 100, 2, 4), (2048, 93, 22, 10), (4096, 32, 128, 108),
                                               (4096, 1, 0, 4094), (640, 5, 128, 128)])
@pytest.mark.parametrize("n,n_real,pad", [(256, 200, 56), (128, 128, 0)])
def test_cut_rows_in_pairs(gpu, k, units, full, kept, n, n_real, pad):
    """the same bits for scales on the 16-byte grid, off it, and as quantising the gathered dequantised rows, groups of zeros,
    subnormal and large scales among them"""
    from uniql_amd import ops
    (w, s), _, _ = _packed_layer(gpu, k, n, torch.Generator().manual_seed(k + kept))
    s = s.clone()
    s[0, 3:70], s[1, ::2], s[2, 5], s[3, 9] = 0.0, 6e-8, 300.0, -0.01
    rows = torch.tensor([u * full + i for u in range(units) for i in range(kept)], device=gpu)
    want = ops.w4a16_quantize(ops.w4a16_dequant(w, s, n, k)[rows][:, :n_real].t().contiguous(), None, pad_out=pad)
    off = torch.empty(s.numel() + 1, dtype=s.dtype, device=gpu)[1:].view_as(s)
    off.copy_(s)
    for scales in (s, off):
        got = ops.w4a16_cut_rows(w, scales, n, k, units, full, kept, n_real, pad_out=pad)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim", [128, 256, 4096, 32768, 20 * 128, 28 * 512])
def test_transform_of_rows_off_the_16_byte_grid(gpu, dtype, dim):
    """a contiguous view with an offset: the same bits as its aligned copy"""
    from uniql_amd import ops
    g = torch.Generator().manual_seed(dim)
    flat = torch.randn(3 * dim + 1, generator=g).to(dtype).to(gpu)
    x = flat[1:].view(3, dim)
    base = {2560: 20, 14336: 28}.get(dim)
    go = (lambda t: ops.hadamard_blockwise(t, 0.125)) if base is None else (lambda t: ops.hadamard_composite(t, 0.125, base))
    if dim == 128 and dtype == torch.float16:   # refused, as ever
        with pytest.raises(RuntimeError):
            go(x)
        return
    assert torch.equal(go(x), go(x.clone()))


@pytest.mark.parametrize("where", ["cpu", "cuda"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_scales_of_a_quantised_weight_stay_on_the_device(gpu, where, dtype):
    """the same layer wherever the scales are, and no wait for the device where they are beside the weight"""
    from uniql_amd import layout
    from uniql_amd.quantize.quant_linear_layers import W4A16B16O16Linear
    lin = torch.nn.Linear(384, 200, bias=False, device=gpu, dtype=torch.float16)
    lin.apply_gptq, lin.bits, lin.group_size = True, 4, 128
    lin.group_scale = (0.006 + 0.004 * torch.rand((3, 200), generator=torch.Generator().manual_seed(3))).to(dtype).to(where)
    torch.cuda.set_sync_debug_mode("error" if where == "cuda" else "default")
    try:
        q = W4A16B16O16Linear.from_fp16(lin)
    finally:
        torch.cuda.set_sync_debug_mode("default")
    _, packed, scale = layout.quantize_and_pack(lin.weight.detach().cpu().t().contiguous(), 128, lin.group_scale.half().cpu(), pad_out=56)
    assert torch.equal(q.weight.cpu(), packed) and torch.equal(q.scale.cpu(), scale)
