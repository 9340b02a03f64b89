"""What is timed when this package's speed is looked at, and how exact it has to stay.

A case is a dict of plain values whose "kind" names one piece of work that a program using the package
has it do, through the public modules and functions:

    decode    one decoder layer's quantised modules for a batch of sequences that advance by one token
              each, captured once in a HIP graph and replayed, as a serving loop runs it
    prefill   the same modules, called eagerly, on the tokens of one prompt
    linear    one W4A16B16O16Linear.forward, eager, few rows: the smallest call there is
    mamba     a Mamba2 block's two projections, the second behind its online rotation
    embed     the 4-bit embedding lookup of a prompt's or a batch's token ids
    hadamard  the online rotation module on activations
    quantize  from_fp16 of a linear layer or of an embedding table (producing the 4-bit model)
    rotate    HadLinear with fuse_had=True (the offline rotation in front of the quantiser)
    slice     cutting one block's packed tensors to a pruned size while a checkpoint is loaded

listed() holds the sizes looked at first, draw() gives others of the same ranges.  The widths are those of
Llama-3.1-8B, Llama-2-7B and Mamba2-8B, whole and pruned, that bench.py and the tests use.
"""
from __future__ import annotations

import math

import torch

HIDDEN = 4096          # hidden size of all three models
FULL_HEAD_DIM = 128    # rotary tables and checkpoints are kept at this head width
MAMBA_GROUPS, MAMBA_STATE, MAMBA_HEADS, MAMBA_INNER = 8, 128, 128, 8192
GRAPH_TOKENS = 128     # up to this many rows a step is launch-bound enough to be worth a graph
DEVICE = "cuda:0"


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # one user, one token: the latency of every step of a chat
        dict(name="decode_1_token", kind="decode", tokens=1, kv_heads=8, head_dim=128, inter=14336),
        # a small batch on a structured-pruned model (widths padded to 256, short rows, fewer columns stored)
        dict(name="decode_8_tokens_pruned", kind="decode", tokens=8, kv_heads=8, head_dim=108, inter=12160),
        # continuous batching: dozens of sequences advance together
        dict(name="decode_48_tokens", kind="decode", tokens=48, kv_heads=8, head_dim=128, inter=14336),
        # a short prompt of odd length on a pruned model: time to first token
        dict(name="prefill_333_pruned", kind="prefill", tokens=333, kv_heads=8, head_dim=108, inter=12160),
        # a long prompt: the largest call
        dict(name="prefill_4096", kind="prefill", tokens=4096, kv_heads=8, head_dim=128, inter=14336),
        # a single small projection called eagerly (key projection with a bias): host path and launch latency
        dict(name="linear_1_token", kind="linear", tokens=1, in_features=4096, out_features=1024, extra="bias"),
        # Mamba2 prompt: in_proj, whole-row rotation, out_proj
        dict(name="mamba_1024_tokens", kind="mamba", tokens=1024, inner=8192, had_block=8192),
        # the embedding lookup of a prompt against the largest vocabulary
        dict(name="embed_2048_ids", kind="embed", tokens=2048, vocab=256000, dim=4096),
        # the rotation module on a prompt's MLP activations, width 28 * 512
        dict(name="hadamard_1024x14336", kind="hadamard", tokens=1024, dim=14336, dtype="float16"),
        # producing the model: an MLP projection
        dict(name="quantize_linear", kind="quantize", what="linear", rows=14336, cols=4096),
        # rotating a projection's weight on both sides before it is quantised
        dict(name="rotate_weight", kind="rotate", in_features=14336, out_features=4096, sides="both", dtype="float16"),
        # loading a pruned model from the full checkpoint: one decoder layer
        dict(name="slice_layer", kind="slice", block="llama", kv_heads=8, head_dim=108, inter=12160),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _model(rng):
    """(kv heads, kept head width, MLP width): whole models or pruned by up to about a third."""
    kv_heads, inter = rng.choice([(8, 14336), (32, 11008)])
    head_dim = FULL_HEAD_DIM
    if rng.random() < 0.6:
        head_dim = 2 * rng.randint(42, 63)
        inter = 8 * rng.randint(int(0.66 * inter) // 8, inter // 8)
    return dict(kv_heads=kv_heads, head_dim=head_dim, inter=inter)


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "linear", "mamba", "embed", "hadamard", "quantize",
                       "rotate", "slice"])
    if kind == "decode":
        return dict(kind=kind, tokens=_log_int(rng, 1, GRAPH_TOKENS), **_model(rng))
    if kind == "prefill":
        return dict(kind=kind, tokens=_log_int(rng, GRAPH_TOKENS + 1, 4096), **_model(rng))
    if kind == "linear":
        return dict(kind=kind, tokens=_log_int(rng, 1, 64), in_features=8 * _log_int(rng, 32, 1792),
                    out_features=_log_int(rng, 256, 14336), extra=rng.choice(["none", "bias", "residual", "relu2"]))
    if kind == "mamba":
        had_block = rng.choice([MAMBA_INNER, 128])
        inner = MAMBA_INNER if had_block == MAMBA_INNER else MAMBA_HEADS * rng.randint(44, 64)
        return dict(kind=kind, tokens=_log_int(rng, 1, 4096), inner=inner, had_block=had_block)
    if kind == "embed":
        return dict(kind=kind, tokens=_log_int(rng, 1, 16384), vocab=rng.choice([32000, 128256, 256000]),
                    dim=rng.choice([2048, 4096, 5120, 8192]))
    if kind == "hadamard":
        return dict(kind=kind, tokens=_log_int(rng, 1, 4096), dim=rng.choice([128, 1024, 3584, 4096, 5120, 8192, 14336]),
                    dtype=rng.choice(["float16", "float16", "bfloat16", "float32"]))
    if kind == "quantize":
        if rng.random() < 0.3:
            return dict(kind=kind, what="embedding", rows=rng.randint(16000, 128256), cols=rng.choice([2048, 4096, 5120]))
        return dict(kind=kind, what=rng.choice(["linear", "gptq"]), rows=_log_int(rng, 256, 14336), cols=8 * _log_int(rng, 32, 1792))
    if kind == "rotate":
        return dict(kind=kind, in_features=rng.choice([1024, 3584, 4096, 5120, 8192, 14336]),
                    out_features=rng.choice([1024, 2048, 4096]), sides=rng.choice(["in", "out", "both"]),
                    dtype=rng.choice(["float16", "float16", "bfloat16", "float32"]))
    if rng.random() < 0.3:
        return dict(kind=kind, block="mamba", inner=MAMBA_HEADS * 2 * rng.randint(21, 31), state=8 * rng.randint(10, 15))
    m = _model(rng)
    if m["head_dim"] == FULL_HEAD_DIM:
        m["head_dim"] = 2 * rng.randint(42, 63)
    return dict(kind=kind, block="llama", **m)


# ---------------------------------------------------------------------------------------------
# what a program has in hand before the call
# ---------------------------------------------------------------------------------------------
def _normal(gen, *shape, std=1.0, dtype=torch.float16):
    return (torch.randn(shape, device=DEVICE, generator=gen) * std).to(dtype)


def _activations(gen, *shape):
    """Normal values with a few much larger channels, as hidden states have."""
    x = torch.randn(shape, device=DEVICE, generator=gen)
    loud = torch.randint(0, shape[-1], (max(1, shape[-1] // 512),), device=DEVICE, generator=gen)
    x[..., loud] *= 16.0
    return x.to(torch.float16)


def _fp16_linear(gen, out_features, in_features, bias=False):
    lin = torch.nn.Linear(1, 1, bias=False, device=DEVICE, dtype=torch.float16)
    lin.in_features, lin.out_features = in_features, out_features
    lin.weight.data = _normal(gen, out_features, in_features, std=0.02)
    if bias:
        lin.bias = torch.nn.Parameter(_normal(gen, out_features, std=0.1))
    return lin


def _quantised(gen, out_features, in_features, bias=False):
    from uniql_amd.quantize.quant_linear_layers import W4A16B16O16Linear
    return W4A16B16O16Linear.from_fp16(_fp16_linear(gen, out_features, in_features, bias))


def _heads(case):
    return (HIDDEN // FULL_HEAD_DIM), case["kv_heads"], case["head_dim"]


def _prepare_layer(case, gen):
    from uniql_amd.quantize.fused_layers import W4A16FusedLinear, W4A16GateUpSiLU
    nq, nkv, d = _heads(case)
    m = case["tokens"]
    st = dict(case=case)
    st["qkv"] = W4A16FusedLinear.from_linears([_quantised(gen, nq * d, HIDDEN), _quantised(gen, nkv * d, HIDDEN),
                                               _quantised(gen, nkv * d, HIDDEN)])
    st["o"] = _quantised(gen, HIDDEN, nq * d)
    st["gate_up"] = W4A16GateUpSiLU.from_linears(_quantised(gen, case["inter"], HIDDEN), _quantised(gen, case["inter"], HIDDEN))
    st["down"] = _quantised(gen, HIDDEN, case["inter"])
    st["x"] = _activations(gen, 1, m, HIDDEN)
    st["attn"] = _normal(gen, 1, m, nq * d)
    # decode: one new token for each of `tokens` sequences, every one at a position of its own; prefill: one sequence
    pos = torch.randint(0, 4096, (1, m), device=DEVICE, generator=gen) if case["kind"] == "decode" else torch.arange(m, device=DEVICE)[None]
    inv = 500000.0 ** (-torch.arange(0, FULL_HEAD_DIM, 2, device=DEVICE) / FULL_HEAD_DIM)
    angle = pos[..., None] * torch.cat([inv, inv])
    st["cos"], st["sin"] = angle.cos().to(torch.float16), angle.sin().to(torch.float16)
    # every key/value head keeps the same number of columns of each rotary half, its own choice of them
    order = torch.rand((nkv, FULL_HEAD_DIM // 2), device=DEVICE, generator=gen).argsort(dim=1)[:, :d // 2].sort(dim=1).values
    st["indices"] = torch.cat([order, order + FULL_HEAD_DIM // 2], dim=1).to(torch.uint8)
    return st


def _run_layer(st):
    from uniql_amd import ops
    nq, nkv, d = _heads(st["case"])
    q, k, v = st["qkv"](st["x"])
    ops.rope_indices_(q.unflatten(-1, (nq, d)), k.unflatten(-1, (nkv, d)), st["cos"], st["sin"], st["indices"])
    h = st["o"](st["attn"], residual=st["x"])
    a = st["gate_up"](h)
    return q, k, v, h, a, st["down"](a, residual=h)


def _prepare_mamba(case, gen):
    inner, m = case["inner"], case["tokens"]
    st = dict(case=case)
    st["in_proj"] = _quantised(gen, 2 * inner + 2 * MAMBA_GROUPS * MAMBA_STATE + MAMBA_HEADS, HIDDEN)
    st["out_proj"] = _quantised(gen, HIDDEN, inner).set_online_hadamard(case["had_block"])
    st["x"] = _activations(gen, 1, m, HIDDEN)
    st["y"] = _activations(gen, 1, m, inner)     # what the scan and the gated norm hand over
    return st


def _run_mamba(st):
    return st["in_proj"](st["x"]), st["out_proj"](st["y"])


def _captured(st, step):
    """Records `step` once, as a serving loop does before its first token; run() replays it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(st)
    torch.cuda.current_stream().wait_stream(side)
    st["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(st["graph"]):
        st["out"] = step(st)
    return st


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    if kind == "decode":
        return _captured(_prepare_layer(case, gen), _run_layer)
    if kind == "prefill":
        return _prepare_layer(case, gen)
    if kind == "mamba":
        st = _prepare_mamba(case, gen)
        return _captured(st, _run_mamba) if case["tokens"] <= GRAPH_TOKENS else st
    st = dict(case=case)
    if kind == "linear":
        st["layer"] = _quantised(gen, case["out_features"], case["in_features"], case["extra"] == "bias")
        st["x"] = _activations(gen, 1, case["tokens"], case["in_features"])
        st["residual"] = _activations(gen, 1, case["tokens"], case["out_features"]) if case["extra"] == "residual" else None
    elif kind == "embed":
        from uniql_amd.quantize.quant_embedding_layers import W4O16Embedding
        table = W4O16Embedding(case["vocab"], case["dim"], device=DEVICE)
        # random words are random codes; the scales those of rows of N(0, 0.02)
        table.weight.data.random_(-2 ** 31, 2 ** 31 - 1, generator=gen)
        table.scales.copy_(0.008 + 0.004 * torch.rand(case["vocab"], device=DEVICE, generator=gen))
        st["table"] = table
        st["ids"] = torch.randint(0, case["vocab"], (1, case["tokens"]), device=DEVICE, generator=gen)
    elif kind == "hadamard":
        from uniql_amd.quantize.quant_hadamard_layers import Hadamard
        st["rotation"] = Hadamard(case["dim"])
        st["x"] = _activations(gen, 1, case["tokens"], case["dim"]).to(getattr(torch, case["dtype"]))
    elif kind == "quantize":
        if case["what"] == "embedding":
            st["layer"] = torch.nn.Embedding(1, 1, device=DEVICE, dtype=torch.float16)
            st["layer"].num_embeddings, st["layer"].embedding_dim = case["rows"], case["cols"]
            st["layer"].weight.data = _normal(gen, case["rows"], case["cols"], std=0.02)
        else:
            st["layer"] = _fp16_linear(gen, case["rows"], case["cols"])
            if case["what"] == "gptq":  # weights a GPTQ pass has left, with the group scales it chose
                groups = -(-case["cols"] // 128)
                st["layer"].apply_gptq, st["layer"].bits, st["layer"].group_size = True, 4, 128
                st["layer"].group_scale = 0.006 + 0.004 * torch.rand((groups, case["rows"]), device=DEVICE, generator=gen)
    elif kind == "rotate":
        st["layer"] = _fp16_linear(gen, case["out_features"], case["in_features"])
        st["layer"].weight.data = st["layer"].weight.data.to(getattr(torch, case["dtype"]))
    elif kind == "slice":
        names = _slice_sizes(case)
        st["packed"] = {name: _quantised(gen, n, k) for name, (n, k) in names.items()}
    else:
        raise ValueError(kind)
    return st


def _slice_sizes(case):
    """name -> (output columns, input rows) of the full-size projections"""
    if case["block"] == "mamba":
        return dict(in_proj=(2 * MAMBA_INNER + 2 * MAMBA_GROUPS * MAMBA_STATE + MAMBA_HEADS, HIDDEN), out_proj=(HIDDEN, MAMBA_INNER))
    nq, nkv, full = HIDDEN // FULL_HEAD_DIM, case["kv_heads"], 14336 if case["kv_heads"] == 8 else 11008
    return dict(q=(nq * FULL_HEAD_DIM, HIDDEN), k=(nkv * FULL_HEAD_DIM, HIDDEN), v=(nkv * FULL_HEAD_DIM, HIDDEN),
                o=(HIDDEN, nq * FULL_HEAD_DIM), gate=(full, HIDDEN), up=(full, HIDDEN), down=(HIDDEN, full))


def _run_slice(st):
    from uniql_amd import slicing as S
    case, packed = st["case"], st["packed"]

    def tensors(name):
        layer = packed[name]
        return layer.weight, layer.scale, layer.workspace

    def shape(name):
        return packed[name].weight.shape

    if case["block"] == "mamba":
        return (S.slice_w4a16_in_proj(*tensors("in_proj"), HIDDEN, MAMBA_GROUPS, MAMBA_HEADS, MAMBA_INNER, MAMBA_STATE,
                                      case["inner"], case["state"], shape("in_proj")),
                S.slice_w4a16_out_proj(*tensors("out_proj"), HIDDEN, MAMBA_GROUPS, MAMBA_HEADS, MAMBA_INNER, case["inner"],
                                       shape("out_proj")))
    nq, nkv, d = _heads(case)
    full = _slice_sizes(case)["up"][0]
    out = []
    for name, heads in (("q", nq), ("k", nkv)):
        w, s, ws = tensors(name)
        out.append(S.slice_w4a16_qk_proj(w, None, s, ws, HIDDEN, heads, FULL_HEAD_DIM, d, shape(name)))
    out.append(S.slice_w4a16_v_proj(*tensors("v"), HIDDEN, nkv, FULL_HEAD_DIM, d, shape("v")))
    out.append(S.slice_w4a16_o_proj(*tensors("o"), HIDDEN, nq, FULL_HEAD_DIM, d, shape("o")))
    for name in ("gate", "up"):
        out.append(S.slice_w4a16_up_gate_proj(*tensors(name), HIDDEN, full, case["inter"], shape(name)))
    out.append(S.slice_w4a16_down_proj(*tensors("down"), HIDDEN, full, case["inter"], shape("down")))
    return out


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    case = state["case"]
    kind = case["kind"]
    if kind == "prefill":
        return _run_layer(state)
    if kind == "mamba":
        return _run_mamba(state)
    if kind == "linear":
        return state["layer"](state["x"], residual=state["residual"], activation="relu2" if case["extra"] == "relu2" else None)
    if kind == "embed":
        return state["table"](state["ids"])
    if kind == "hadamard":
        return state["rotation"](state["x"])
    if kind == "quantize":
        if case["what"] == "embedding":
            from uniql_amd.quantize.quant_embedding_layers import W4O16Embedding
            q = W4O16Embedding.from_fp16(state["layer"])
            return q.weight.data, q.scales
        from uniql_amd.quantize.quant_linear_layers import W4A16B16O16Linear
        q = W4A16B16O16Linear.from_fp16(state["layer"])
        return q.weight, q.scale
    if kind == "rotate":
        from uniql_amd.quantize.quant_linear_layers import HadLinear
        rotated = HadLinear(state["layer"], input_transform=case["sides"] != "out", output_transform=case["sides"] != "in",
                            fuse_had=True)
        return rotated.weight.data
    return _run_slice(state)


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------------------------
def _linear_work(m, n, k, n_out=None):
    """codes, scales, input rows, output rows; multiply-adds"""
    n_out = n if n_out is None else n_out
    return n * k / 2 + n * k / 64 + 2 * m * k + 2 * m * n_out, 2.0 * m * n * k


def _packed_bytes(n, k):
    return n * k / 2 + n * k / 64


def work(case):
    kind, m = case["kind"], case.get("tokens", 0)
    flops = 0.0
    if kind in ("decode", "prefill"):
        nq, nkv, d = _heads(case)
        parts = [_linear_work(m, (nq + 2 * nkv) * d, HIDDEN), _linear_work(m, HIDDEN, nq * d),
                 _linear_work(m, 2 * case["inter"], HIDDEN, case["inter"]), _linear_work(m, HIDDEN, case["inter"])]
        bytes_ = sum(p[0] for p in parts)
        flops = sum(p[1] for p in parts)
        bytes_ += 4 * m * (nq + nkv) * d + 2 * 2 * m * FULL_HEAD_DIM   # rotary: q, k in place, the tables
        bytes_ += 2 * 2 * m * HIDDEN                                    # the two residual inputs
    elif kind == "linear":
        bytes_, flops = _linear_work(m, case["out_features"], case["in_features"])
        bytes_ += {"bias": 2 * case["out_features"], "residual": 2 * m * case["out_features"]}.get(case["extra"], 0)
    elif kind == "mamba":
        inner = case["inner"]
        a = _linear_work(m, 2 * inner + 2 * MAMBA_GROUPS * MAMBA_STATE + MAMBA_HEADS, HIDDEN)
        b = _linear_work(m, HIDDEN, inner)
        bytes_, flops = a[0] + b[0], a[1] + b[1]
    elif kind == "embed":
        bytes_ = m * (8 + 2 + case["dim"] / 2 + 2 * case["dim"])
    elif kind == "hadamard":
        bytes_ = 2 * m * case["dim"] * torch.empty(0, dtype=getattr(torch, case["dtype"])).element_size()
    elif kind == "quantize":
        n, k = case["rows"], case["cols"]
        bytes_ = 2 * n * k + (n * k / 2 + 2 * n if case["what"] == "embedding" else _packed_bytes(n, k))
        bytes_ += 4 * n * k / 128 if case["what"] == "gptq" else 0
    elif kind == "rotate":
        bytes_ = 2 * case["in_features"] * case["out_features"] * torch.empty(0, dtype=getattr(torch, case["dtype"])).element_size()
    else:
        if case["block"] == "mamba":
            kept = [(2 * case["inner"] + 2 * MAMBA_GROUPS * case["state"] + MAMBA_HEADS, HIDDEN), (HIDDEN, case["inner"])]
        else:
            nq, nkv, d = _heads(case)
            kept = [(nq * d, HIDDEN), (nkv * d, HIDDEN), (nkv * d, HIDDEN), (HIDDEN, nq * d)] + \
                [(case["inter"], HIDDEN)] * 2 + [(HIDDEN, case["inter"])]
        bytes_ = sum(2 * _packed_bytes(n, k) for n, k in kept)
    return {"bytes": float(bytes_), "flops": float(flops)}


def tolerance(case):
    # The products add fp32 terms in an order that is the kernel's own and round to fp16 where the layers do.
    # Four times the distance of the outputs from the same sequence in float64 (layer: 6.4e-4 on the last
    # output, 5.7e-3 its largest; single products: 2.9e-4 and 1.3e-3; a squared output doubles it).
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 2.5e-3, "max": 2.5e-2}
    if case["kind"] in ("linear", "mamba"):
        twice = 2 if case.get("extra") == "relu2" else 1
        return {"rel": twice * 1.2e-3, "max": twice * 5e-3}
    # The rotation fixes the order of its fp32 additions, the quantisers their roundings, the lookup and
    # the cuts move codes: nothing may differ.
    return "exact"
