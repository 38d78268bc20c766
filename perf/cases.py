"""The work a user of the engine has it do, as cases that can be timed and compared.

A case is one pass through the modules a model is built from: ``PackedLinear``,
``PackedSwiGLU``, ``PackedEmbedding`` (gather and tied head), a weight load, and
a decode step of whole layers replayed from a HIP graph. Shapes are those of
``ternel_amd.layout.MODEL_LINEAR_SHAPES``, of ``bench.py`` and of the tests;
``draw`` spreads the same paths over smaller, larger and odd sizes.
"""

import math

import torch

from ternel_amd.layout import PackedTensorLayout
from ternel_amd.kernels import pack_weights
from ternel_amd.modules import PackedEmbedding, PackedLinear, PackedSwiGLU

GROUP = 128
BLOCK = 28
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
BYTES = {"f16": 2, "bf16": 2, "f32": 4}

# One layer's projections of the 27B census, as (output, input) widths: three
# layers in four carry linear attention, the fourth full attention.
LINEAR_ATTENTION = (("qkv", 2.0, 1.0), ("z", 1.2, 1.0), ("out", 1.0, 1.2))
FULL_ATTENTION = (("q", 2.4, 1.0), ("k", 0.2, 1.0), ("v", 0.2, 1.0), ("o", 1.0, 1.2))
MLP_RATIO = 3.4


def listed():
    return [
        # A single sequence's projection called by itself: one launch and the call around it.
        {"name": "linear-4096-m1", "kind": "linear", "rows": 4096, "columns": 4096, "batch": 1, "dtype": "f16"},
        # One decoded token through four layers of the 27B census (three linear-attention
        # layers, one full-attention layer, gate/up/down in each), captured once as a HIP
        # graph and replayed, as a decode loop does.
        {"name": "decode-4-layers", "kind": "decode", "hidden": 5120, "layers": 4, "dtype": "f16"},
        # Continuous batching: a few sequences decoded together, through one MLP.
        {"name": "mlp-m8", "kind": "mlp", "hidden": 17408, "columns": 5120, "batch": 8, "dtype": "bf16"},
        # A fuller decode batch through the attention input projection.
        {"name": "qkv-m32", "kind": "linear", "rows": 8192, "columns": 5120, "batch": 32, "dtype": "f16"},
        # The largest decode batches, and speculative windows, through one MLP.
        {"name": "mlp-m64", "kind": "mlp", "hidden": 17408, "columns": 5120, "batch": 64, "dtype": "bf16"},
        # The logits of a few sequences: the tied head of the 27B vocabulary.
        {"name": "head-m4", "kind": "head", "rows": 248320, "columns": 5120, "batch": 4, "dtype": "bf16"},
        # fp32 activations (a model run in its highest precision), a short batch.
        {"name": "qkv-m24-f32", "kind": "linear", "rows": 8192, "columns": 5120, "batch": 24, "dtype": "f32"},
        # A short prompt of odd length, or the ragged last chunk of a long one.
        {"name": "out-m203", "kind": "linear", "rows": 5120, "columns": 6144, "batch": 203, "dtype": "f16"},
        # The usual prefill chunk through one MLP.
        {"name": "mlp-m512", "kind": "mlp", "hidden": 17408, "columns": 5120, "batch": 512, "dtype": "bf16"},
        # A long prefill chunk through one MLP.
        {"name": "mlp-m2048", "kind": "mlp", "hidden": 17408, "columns": 5120, "batch": 2048, "dtype": "f16"},
        # The token embeddings of a long prompt.
        {"name": "embed-8192", "kind": "embed", "rows": 151936, "columns": 5120, "batch": 8192, "dtype": "f16"},
        # Loading a weight: the scan of every byte and the permutation into the kernels' layout.
        {"name": "load-gate", "kind": "load", "rows": 17408, "columns": 5120},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49)))))


def _log_width(rng, low, high):
    return GROUP * max(1, _log_int(rng, low // GROUP, high // GROUP))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "mlp", "mlp", "mlp", "decode", "head", "embed", "load"])
    dtype = rng.choice(["f16", "f16", "bf16", "bf16", "f32"]) if kind == "linear" else rng.choice(["f16", "bf16"])
    if kind == "linear":
        return {"kind": kind, "rows": _log_int(rng, 48, 24576), "columns": _log_width(rng, 1024, 17408),
                "batch": _log_int(rng, 1, 64 if dtype == "f32" else 1024), "dtype": dtype}
    if kind == "mlp":
        return {"kind": kind, "hidden": _log_width(rng, 2048, 17408), "columns": _log_width(rng, 1024, 5120),
                "batch": _log_int(rng, 1, 2048), "dtype": dtype}
    if kind == "decode":
        return {"kind": kind, "hidden": 640 * rng.randint(3, 8), "layers": rng.randint(1, 4), "dtype": dtype}
    if kind == "head":
        return {"kind": kind, "rows": _log_int(rng, 32000, 248320), "columns": _log_width(rng, 2048, 5120),
                "batch": _log_int(rng, 1, 16), "dtype": dtype}
    if kind == "embed":
        return {"kind": kind, "rows": _log_int(rng, 32000, 248320), "columns": _log_width(rng, 1024, 5120),
                "batch": _log_int(rng, 1, 8192), "dtype": dtype}
    return {"kind": "load", "rows": _log_int(rng, 1024, 24576), "columns": _log_width(rng, 1024, 17408)}


# -- shapes -------------------------------------------------------------------
def _width(ratio, hidden):
    return int(round(ratio * hidden / GROUP)) * GROUP


def _decode_shapes(case):
    """(name, rows, columns) of every projection of the step, in order."""
    hidden = case["hidden"]
    shapes = []
    for layer in range(case["layers"]):
        full = layer % 4 == 3
        for name, out, inp in FULL_ATTENTION if full else LINEAR_ATTENTION:
            shapes.append((f"{layer}.{name}", _width(out, hidden), _width(inp, hidden)))
            if name == "z":  # the two 48-row gates of linear attention
                shapes.append((f"{layer}.a", 48, hidden))
                shapes.append((f"{layer}.b", 48, hidden))
        middle = _width(MLP_RATIO, hidden)
        shapes.append((f"{layer}.gate", middle, hidden))
        shapes.append((f"{layer}.up", middle, hidden))
        shapes.append((f"{layer}.down", hidden, middle))
    return shapes


# -- inputs, from the seed alone ----------------------------------------------
def _generator(seed, k=0):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + k)
    return gen


def _blocks(rows, columns, gen):
    """Canonical blocks ``(rows, columns / 128, 28)``: trits -1/0/+1 with
    probabilities 0.3/0.4/0.3 and fp16 scales around 0.016."""
    count = rows * (columns // GROUP)
    out = torch.empty((count, BLOCK), dtype=torch.uint8, device="cuda")
    step = 1 << 20
    for at in range(0, count, step):
        n = min(step, count - at)
        scale = (torch.randn(n, generator=gen, device="cuda") * 0.02).abs_() + 1e-4
        out[at:at + n, :2] = scale.half().view(torch.uint8).reshape(n, 2)
        ten = torch.randint(0, 10, (n, 26, 5), generator=gen, device="cuda", dtype=torch.uint8)
        trits = (ten > 2).to(torch.uint8) + (ten > 6).to(torch.uint8)
        trits[:, 25, 3:] = 0
        for i, power in enumerate((1, 3, 9, 27, 81)):
            trits[:, :, i] *= power
        out[at:at + n, 2:] = trits.sum(dim=2, dtype=torch.int32).to(torch.uint8)
    return out.reshape(rows, columns // GROUP, BLOCK)


def _activations(batch, columns, dtype, gen):
    """Normal values under channel gains that spread as a hidden state's do."""
    gain = torch.exp(0.5 * torch.randn(columns, generator=gen, device="cuda"))
    return (torch.randn((batch, columns), generator=gen, device="cuda") * gain).to(DTYPES[dtype])


def _linear(rows, columns, gen):
    layout = PackedTensorLayout.for_tensor(rows, columns)
    layer = PackedLinear(layout)
    layer.packed = pack_weights(_blocks(rows, columns, gen), layout=layout)
    return layer


def prepare(case, seed):
    kind = case["kind"]
    gen = _generator(seed)
    if kind == "load":
        layout = PackedTensorLayout.for_tensor(case["rows"], case["columns"])
        return {"kind": kind, "layer": PackedLinear(layout), "blocks": _blocks(case["rows"], case["columns"], gen)}
    if kind == "embed":
        layout = PackedTensorLayout.for_tensor(case["rows"], case["columns"])
        layer = PackedEmbedding(layout, dtype=DTYPES[case["dtype"]])
        layer.packed = pack_weights(_blocks(case["rows"], case["columns"], gen), layout=layout)
        ids = torch.randint(0, case["rows"], (case["batch"],), generator=gen, device="cuda")
        return {"kind": kind, "layer": layer, "ids": ids}
    if kind == "head":
        layout = PackedTensorLayout.for_tensor(case["rows"], case["columns"])
        layer = PackedEmbedding(layout, dtype=DTYPES[case["dtype"]])
        layer.packed = pack_weights(_blocks(case["rows"], case["columns"], gen), layout=layout)
        return {"kind": kind, "layer": layer, "x": _activations(case["batch"], case["columns"], case["dtype"], gen)}
    if kind == "linear":
        layer = _linear(case["rows"], case["columns"], gen)
        return {"kind": kind, "layer": layer, "x": _activations(case["batch"], case["columns"], case["dtype"], gen)}
    if kind == "mlp":
        # alternating gate and up rows: the fused layer's one weight
        glu = PackedSwiGLU(case["hidden"], case["columns"])
        glu.packed = pack_weights(_blocks(2 * case["hidden"], case["columns"], gen), layout=glu.layout)
        down = _linear(case["columns"], case["hidden"], gen)
        x = _activations(case["batch"], case["columns"], case["dtype"], gen) * 0.1
        return {"kind": kind, "glu": glu, "down": down, "x": x}
    # decode: eager once, so that workspaces exist, then captured
    layers, inputs = [], []
    for k, (_, rows, columns) in enumerate(_decode_shapes(case)):
        gen = _generator(seed, k + 1)
        layers.append(_linear(rows, columns, gen))
        inputs.append(_activations(1, columns, case["dtype"], gen))
    for layer, x in zip(layers, inputs):
        layer(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = [layer(x) for layer, x in zip(layers, inputs)]
    return {"kind": kind, "graph": graph, "outputs": outputs, "layers": layers, "inputs": inputs}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "mlp":
        middle = state["glu"](state["x"])
        return middle, state["down"](middle)
    if kind == "decode":
        state["graph"].replay()
        return state["outputs"]
    if kind == "head":
        return state["layer"].as_linear(state["x"])
    if kind == "embed":
        return state["layer"](state["ids"])
    state["layer"].load_blocks(state["blocks"])
    return state["layer"].packed


# -- what a pass cannot do without --------------------------------------------
def _product(rows, columns, batch, size):
    """Bytes and operations of one packed product: every block, x and y once."""
    return (BLOCK * rows * (columns // GROUP) + batch * (rows + columns) * size, 2 * batch * rows * columns)


def work(case):
    kind = case["kind"]
    if kind == "load":  # read the blocks, write the words (rows padded to 64)
        groups = case["columns"] // GROUP
        return {"bytes": BLOCK * groups * (case["rows"] + -(-case["rows"] // 64) * 64), "flops": 0}
    size = BYTES[case["dtype"]]
    if kind == "embed":  # a row's blocks and its id read, its values written
        return {"bytes": case["batch"] * (BLOCK * (case["columns"] // GROUP) + 8 + case["columns"] * size), "flops": 0}
    if kind == "mlp":
        up = _product(2 * case["hidden"], case["columns"], case["batch"], size)
        down = _product(case["columns"], case["hidden"], case["batch"], size)
        # the fused layer writes hidden values a row, not 2 * hidden
        return {"bytes": up[0] - case["batch"] * case["hidden"] * size + down[0], "flops": up[1] + down[1]}
    if kind == "decode":
        products = [_product(rows, columns, 1, size) for _, rows, columns in _decode_shapes(case)]
        return {"bytes": sum(p[0] for p in products), "flops": sum(p[1] for p in products)}
    total = _product(case["rows"], case["columns"], case["batch"], size)
    return {"bytes": total[0], "flops": total[1]}


def tolerance(case):
    """About four times the distance of the path's outputs from 64-bit ones: one
    rounding to the output type for a product, three on the way through an MLP."""
    if case["kind"] in ("embed", "load"):
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 2e-6}
    if case["kind"] == "mlp":
        return {"rel": 1.2e-2 if case["dtype"] == "bf16" else 1.5e-3}
    return {"rel": 7e-3 if case["dtype"] == "bf16" else 9e-4}


# -- the same in 64 bits, from the canonical blocks ---------------------------
def _dense(blocks):
    """Blocks ``(rows, G, 28)`` -> weights ``(rows, G * 128)`` in float64."""
    rows, groups, _ = blocks.shape
    scale = blocks[:, :, :2].contiguous().view(torch.float16).double()
    codes = blocks[:, :, 2:].to(torch.int16)
    digits = [(codes // power) % 3 for power in (1, 3, 9, 27, 81)]
    trits = torch.stack(digits, dim=3).reshape(rows, groups, 130)[:, :, :GROUP]
    return ((trits - 1).double() * scale).reshape(rows, groups * GROUP)


def _product64(blocks, x):
    x64 = x.double().t().contiguous()
    parts = [_dense(blocks[at:at + 4096]) @ x64 for at in range(0, blocks.shape[0], 4096)]
    return torch.cat(parts).t().contiguous()


def exact(case, seed):
    kind = case["kind"]
    gen = _generator(seed)
    if kind == "load":
        return None
    if kind == "embed":
        blocks = _blocks(case["rows"], case["columns"], gen)
        ids = torch.randint(0, case["rows"], (case["batch"],), generator=gen, device="cuda")
        return _dense(blocks[ids])
    if kind in ("linear", "head"):
        blocks = _blocks(case["rows"], case["columns"], gen)
        return _product64(blocks, _activations(case["batch"], case["columns"], case["dtype"], gen))
    if kind == "mlp":
        glu = _blocks(2 * case["hidden"], case["columns"], gen)
        down = _blocks(case["columns"], case["hidden"], gen)
        x = _activations(case["batch"], case["columns"], case["dtype"], gen) * 0.1
        both = _product64(glu, x)
        gate, up = both[:, 0::2], both[:, 1::2]
        middle = gate * torch.sigmoid(gate) * up
        return middle, _product64(down, middle)
    outputs = []
    for k, (_, rows, columns) in enumerate(_decode_shapes(case)):
        gen = _generator(seed, k + 1)
        blocks = _blocks(rows, columns, gen)
        outputs.append(_product64(blocks, _activations(1, columns, case["dtype"], gen)))
    return outputs
