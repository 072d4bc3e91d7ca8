"""The calls whose time is measured: fused op descriptions compiled once and launched on device tensors, as a program
that runs a network with this backend does it.

`listed()` names one size of every kind, `draw(rng)` gives another size of the same kinds, `prepare` builds what such a
program holds before the call (compiled kernel, inputs, output tensors), `run` is one launch. `work` counts every input
read once and every output written once, and the multiplications and additions of a contraction.
"""
import json
import math

import torch

from akg_amd import driver, op_desc

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
SIZES = {"bfloat16": 2, "float16": 2, "float32": 4}
HEADS = 12


def listed():
    return [
        # a small tail of a graph (a gate, a scalar head): the time is that of the call and of one launch
        {"name": "elementwise_small", "kind": "elementwise", "rows": 37, "cols": 130},
        # attention weights of an encoder whose sequence length changes from batch to batch, through the calling form for
        # dynamic shapes; rows that the vector width does not divide
        {"name": "softmax_dynamic", "kind": "masked_softmax", "batch": 32, "q": 333, "k": 333},
        # the end of a transformer block, training or prefill: 16384 tokens
        {"name": "layernorm_residual", "kind": "layernorm", "rows": 16384, "cols": 4096, "dtype": "bfloat16"},
        # per-token quantisation in front of an int8 projection: the largest tensors
        {"name": "quant_int8", "kind": "quant", "rows": 32768, "cols": 8192, "dtype": "bfloat16"},
        # backward: gradients of a scale and a bias over the tokens of an ordinary batch
        {"name": "scale_bias_grad", "kind": "bias_grad", "rows": 4100, "cols": 3000, "dtype": "bfloat16"},
        # forward of a training batch norm, a middle stage of a convolutional network
        {"name": "batchnorm_train", "kind": "batchnorm", "n": 64, "c": 128, "h": 28, "w": 28, "dtype": "bfloat16"},
        # aggregation over the edges of a graph (three coordinates per atom pair), the backward of a gather
        {"name": "segment_sum", "kind": "segment_sum", "positions": 4954 * 4953, "width": 3, "segments": 4954, "skew": False},
        # attention probabilities of one layer in one description: scores, scale, mask and softmax
        {"name": "attention_probs", "kind": "attention", "batch": 192, "m": 512, "k": 64, "n": 512, "dtype": "bfloat16"},
        # a projection in a decoding step: 16 sequences, the weight in a dense layer's [out, in] layout
        {"name": "matmul_decode", "kind": "matmul", "m": 16, "k": 8192, "n": 8192, "dtype": "bfloat16", "act": "none", "tb": True},
        # a projection in a short prefill or a small training batch: few rows and a width the tiles do not divide
        {"name": "matmul_short", "kind": "matmul", "m": 300, "k": 4096, "n": 11000, "dtype": "bfloat16", "act": "gelu", "tb": False},
        # a projection in training or a long prefill
        {"name": "matmul_long", "kind": "matmul", "m": 4096, "k": 8192, "n": 8192, "dtype": "bfloat16", "act": "gelu", "tb": False},
        # its quantised form: int8 operands, dequantisation, bias and activation
        {"name": "matmul_int8", "kind": "matmul_int8", "m": 4096, "k": 8192, "n": 8192, "tb": False},
    ]


def _between(rng, low, high, step=1):
    """A multiple of `step` in [low, high], spread over the logarithm; half of those with step 1 are multiples of 8."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    if step == 1 and value >= 64 and rng.random() < 0.5:
        step = 8
    return int(min(max(round(value / step), -(-low // step)), high // step)) * step


def draw(rng):
    kind = rng.choice(["elementwise", "masked_softmax", "layernorm", "quant", "bias_grad", "batchnorm", "segment_sum",
                       "attention", "matmul", "matmul", "matmul", "matmul_int8"])
    half = rng.choice(["bfloat16", "bfloat16", "float16"])
    any_float = rng.choice([half, half, "float32"])
    if kind == "elementwise":
        case = {"rows": _between(rng, 1, 8192), "cols": _between(rng, 16, 8192)}
    elif kind == "masked_softmax":
        case = {"batch": _between(rng, 1, 32), "q": _between(rng, 1, 512), "k": _between(rng, 8, 512)}
    elif kind == "layernorm" or kind == "quant":
        case = {"rows": _between(rng, 16, 16384), "cols": _between(rng, 256, 8192), "dtype": any_float if kind == "layernorm" else half}
    elif kind == "bias_grad":
        case = {"rows": _between(rng, 64, 16384), "cols": _between(rng, 64, 8192), "dtype": any_float}
    elif kind == "batchnorm":
        side = _between(rng, 7, 112)
        c = _between(rng, 16, 1024, 8)
        case = {"n": _between(rng, 4, max(4, min(128, 60_000_000 // (c * side * side)))), "c": c, "h": side, "w": side, "dtype": any_float}
    elif kind == "segment_sum":
        if rng.random() < 0.5:   # edges of a graph or a mesh: a few numbers each
            case = {"positions": _between(rng, 10_000, 20_000_000), "width": rng.choice([1, 2, 3, 3, 4]), "segments": _between(rng, 300, 16384), "skew": False}
        else:                    # tokens of a batch: the gradient of an embedding table
            case = {"positions": _between(rng, 512, 32768), "width": _between(rng, 128, 2048, 8), "segments": _between(rng, 1000, 32768), "skew": True}
    elif kind == "attention":
        n = _between(rng, 32, 2048, 8)
        m = rng.choice([n, n, _between(rng, 1, 512)])
        case = {"batch": _between(rng, 1, max(1, min(384, 100_000_000 // (m * n)))), "m": m, "k": rng.choice([64, 64, 128]), "n": n, "dtype": half}
    else:
        k, n = _between(rng, 512, 8192, 64), _between(rng, 512, 12288, 8)
        case = {"m": _between(rng, 1, min(4096, 137_000_000_000 // (k * n))), "k": k, "n": n, "tb": rng.random() < 0.5}
        if kind == "matmul":
            case.update(dtype=half, act=rng.choice(["none", "relu", "gelu"]))
    return dict(case, kind=kind)


def _masked_softmax(batch, q, k):
    """softmax(x * 0.125 + (1 - mask) * -10000) over the last axis; x [batch, HEADS, q, k], mask [batch, 1, q, k], float32."""
    b = op_desc.DescBuilder("Fused_Sub_Mul_Mul_Add_Softmax_dynamic")
    mask = b.input([batch, 1, q, k], "float32")
    x = b.input([batch, HEADS, q, k], "float32")
    hide = b.mul(b.sub(b.const(1.0, "float32"), mask), b.const(-10000.0, "float32"))
    s = b.add(hide, b.mul(b.const(0.125, "float32"), x))
    e = b.unary("Exp", b.sub(s, b.reduce("ReduceMax", s, [3], True)))
    return b.dumps([b.div(e, b.reduce("ReduceSum", e, [3], True))])


def _opened(text, extents):
    """The description with these extents left open (-1)."""
    document = json.loads(text)

    def walk(node):
        if isinstance(node, dict):
            if "shape" in node:
                node["shape"] = [-1 if n in extents else n for n in node["shape"]]
            node = list(node.values())
        if isinstance(node, list):
            for child in node:
                walk(child)
    walk(document)
    return json.dumps(document)


def _describe(c):
    kind = c["kind"]
    if kind == "elementwise":
        return op_desc.elementwise_tanh_add_mul(c["rows"], c["cols"])
    if kind == "layernorm":
        return op_desc.layernorm_residual(c["rows"], c["cols"], c["dtype"])
    if kind == "quant":
        return op_desc.quant_int8_residual(c["rows"], c["cols"], c["dtype"])
    if kind == "bias_grad":
        return op_desc.bias_grad(c["rows"], c["cols"], c["dtype"])
    if kind == "batchnorm":
        return op_desc.batchnorm_train_forward(c["n"], c["c"], c["h"], c["w"], c["dtype"])
    if kind == "segment_sum":
        return op_desc.unsorted_segment_sum([c["positions"]], [c["width"]], c["segments"])
    if kind == "attention":
        return op_desc.attention_probabilities(c["batch"], c["m"], c["k"], c["n"], c["dtype"])
    if kind == "matmul":
        return op_desc.gemm_bias_act(c["m"], c["k"], c["n"], c["dtype"], c["act"], transpose_b=c["tb"])
    return op_desc.gemm_int8_dequant_bias_gelu(c["m"], c["k"], c["n"], transpose_b=c["tb"])


def _inputs(c, g):
    """The inputs of a case, in the order of its description, from the generator `g`."""
    kind, dev = c["kind"], torch.device("cuda")
    dtype = DTYPES[c.get("dtype", "float32")]

    def normal(*shape, sigma=1.0, dt=dtype):
        return (torch.randn(shape, generator=g, device=dev) * sigma).to(dt)

    if kind == "elementwise":
        return [normal(c["rows"], c["cols"]) for _ in range(3)]
    if kind == "masked_softmax":
        length = torch.randint(max(1, c["k"] // 2), c["k"] + 1, (c["batch"], 1, 1, 1), generator=g, device=dev)
        mask = (torch.arange(c["k"], device=dev) < length).float().expand(c["batch"], 1, c["q"], c["k"]).contiguous()
        return [mask, normal(c["batch"], HEADS, c["q"], c["k"], sigma=16.0)]
    if kind == "layernorm":
        x, gamma, beta, r = (normal(*s) for s in ((c["rows"], c["cols"]), (c["cols"],), (c["cols"],), (c["rows"], c["cols"])))
        return [x, 1 + gamma * 0.1, beta * 0.1, r]
    if kind == "quant":
        x, r = normal(c["rows"], c["cols"]), normal(c["rows"], c["cols"])
        x[:, torch.randint(0, c["cols"], (1 + c["cols"] // 1000,), generator=g, device=dev)] *= 25   # outlier channels
        return [x, r]
    if kind == "bias_grad":
        return [normal(c["rows"], c["cols"], sigma=0.1), normal(c["rows"], c["cols"])]
    if kind == "batchnorm":
        shape = (1, c["c"], 1, 1)
        offset = normal(*shape, dt=torch.float32)
        x = (torch.randn((c["n"], c["c"], c["h"], c["w"]), generator=g, device=dev) + offset).to(dtype)
        return [x, 1 + 0.1 * normal(*shape, dt=torch.float32), 0.1 * normal(*shape, dt=torch.float32)]
    if kind == "segment_sum":
        u = torch.rand((c["positions"],), generator=g, device=dev)
        if c["skew"]:   # tokens: the frequency of a word falls with its rank
            ids = (torch.exp(u * math.log(c["segments"])) - 1).to(torch.int32)
        else:
            ids = (u * c["segments"]).to(torch.int32)
        return [normal(c["positions"], c["width"]), ids.clamp_(0, c["segments"] - 1)]
    if kind == "attention":
        q, k = normal(c["batch"], c["m"], c["k"]), normal(c["batch"], c["n"], c["k"])
        causal = torch.arange(c["n"], device=dev)[None, :] > torch.arange(c["m"], device=dev)[:, None] + (c["n"] - c["m"] if c["n"] > c["m"] else 0)
        mask = torch.where(causal, -10000.0, 0.0).float().expand(c["batch"], c["m"], c["n"]).contiguous()
        return [q, k, mask]
    weight = (c["n"], c["k"]) if c["tb"] else (c["k"], c["n"])
    if kind == "matmul":
        return [normal(c["m"], c["k"]), normal(*weight, sigma=c["k"] ** -0.5), normal(c["n"], sigma=0.1)]

    def int8(*shape):
        return (torch.randn(shape, generator=g, device=dev) * 40).round().clamp_(-127, 127).to(torch.int8)

    scale = torch.rand((c["m"], 1), generator=g, device=dev) * 0.02 + 0.01
    return [int8(c["m"], c["k"]), scale, int8(*weight), torch.rand((c["n"],), generator=g, device=dev) * 1e-3 + 5e-4,
            normal(c["n"], sigma=0.1, dt=torch.bfloat16)]


def prepare(case, seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    inputs = _inputs(case, generator)
    if case["kind"] == "masked_softmax":
        kernel = driver.HipDynamicKernel(_opened(_masked_softmax(7777, 7778, 7779), (7777, 7778, 7779)))
        kernel.specialize([list(t.shape) for t in inputs]).prepare()
        outputs = [torch.empty_like(inputs[1])]
    else:
        kernel = driver.HipKernel(_describe(case))
        kernel.prepare()
        types = dict(DTYPES, int8=torch.int8)
        outputs = [torch.empty(t.shape, dtype=types[t.dtype], device="cuda") for t in kernel.outputs]
    return {"kernel": kernel, "inputs": inputs, "outputs": outputs}


def run(state):
    kernel, tensors = state["kernel"], state["inputs"] + state["outputs"]
    if isinstance(kernel, driver.HipDynamicKernel):
        kernel.launch_packed([t.data_ptr() for t in tensors], [t.shape for t in tensors], torch.cuda.current_stream().cuda_stream)
    else:
        kernel.launch(tensors)
    return state["outputs"]


def work(case):
    c, kind = case, case["kind"]
    e = SIZES[c.get("dtype", "float32")]
    if kind == "elementwise":
        return {"bytes": 16 * c["rows"] * c["cols"]}
    if kind == "masked_softmax":
        return {"bytes": 4 * c["batch"] * c["q"] * c["k"] * (2 * HEADS + 1)}
    if kind == "layernorm":
        return {"bytes": e * c["cols"] * (3 * c["rows"] + 2)}
    if kind == "quant":
        return {"bytes": c["rows"] * (c["cols"] * (2 * e + 1) + 4)}
    if kind == "bias_grad":
        return {"bytes": c["cols"] * (2 * e * c["rows"] + 8)}
    if kind == "batchnorm":
        return {"bytes": c["c"] * (2 * e * c["n"] * c["h"] * c["w"] + 16)}
    if kind == "segment_sum":
        return {"bytes": 4 * (c["positions"] * (c["width"] + 1) + c["segments"] * c["width"])}
    m, k, n = c["m"], c["k"], c["n"]
    if kind == "attention":
        return {"bytes": c["batch"] * (e * (m * k + n * k + m * n) + 4 * m * n), "flops": 2 * c["batch"] * m * k * n}
    if kind == "matmul":
        return {"bytes": e * (m * k + k * n + n + m * n), "flops": 2 * m * k * n}
    return {"bytes": m * k + k * n + 4 * (m + n) + 2 * n + 2 * m * n, "flops": 2 * m * k * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant", "segment_sum"):
        return "exact"    # integers and their scales; float32 sums that keep the order of the positions
    # Four times the distance from the same result in float64, which is the rounding of the result itself: 1.7e-3 of the
    # norm and one half unit (3.9e-3) at most for bfloat16, 2.1e-4 and 4.9e-4 for float16; float32 results (sums over up to
    # 50000 values, exponentials, tanh) were within 1.2e-7 and 3.5e-7.
    dtype = case.get("dtype", "bfloat16" if kind == "matmul_int8" else "float32")
    return {"bfloat16": {"rel": 7e-3, "max": 1.6e-2}, "float16": {"rel": 9e-4, "max": 2e-3}, "float32": {"rel": 1e-6, "max": 4e-6}}[dtype]


def exact(case, seed):
    """The outputs of `run` for these inputs by plain torch in float64; None for integers made by rounding."""
    c, kind = case, case["kind"]
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    inputs = _inputs(c, generator)

    def const(value):   # constants of a description are float32
        return torch.tensor(value, dtype=torch.float32, device="cuda").double()

    if kind == "segment_sum":
        data, ids = inputs
        return [torch.zeros(c["segments"], c["width"], dtype=torch.float64, device="cuda").index_add_(0, ids.long(), data.double())]
    d = [t.double() for t in inputs]
    del inputs
    if kind == "elementwise":
        return [torch.tanh((d[0] + d[1]) * d[2])]
    if kind == "masked_softmax":
        return [torch.softmax((1 - d[0]) * -10000.0 + 0.125 * d[1], -1)]
    if kind == "attention":
        return [torch.softmax(torch.bmm(d[0], d[1].transpose(1, 2).contiguous()) * const(c["k"] ** -0.5) + d[2], -1)]
    if kind == "quant":
        return [None, (d[0] + d[1]).abs().amax(1) / 127]
    if kind == "bias_grad":
        return [(d[0] * d[1]).sum(0), d[0].sum(0)]
    if kind == "layernorm" or kind == "batchnorm":
        axes = (1,) if kind == "layernorm" else (0, 2, 3)
        mean = d[0].mean(axes, keepdim=True)
        centred = d[0] - mean
        variance = (centred * centred).mean(axes, keepdim=True)
        y = centred * torch.rsqrt(variance + const(1e-5)) * d[1] + d[2]
        return [y + d[3]] if kind == "layernorm" else [y, mean, variance]
    if kind == "matmul":
        y = d[0] @ (d[1].t() if c["tb"] else d[1]) + d[2]
        if c["act"] == "relu":
            return [y.clamp_(min=0)]
    else:
        y = d[0] @ (d[2].t() if c["tb"] else d[2]) * d[1] * d[3] + d[4]
    if kind == "matmul_int8" or c["act"] == "gelu":
        y = y * (torch.tanh((y + y * y * y * const(0.044715)) * const(0.7978845608028654)) + 1) * 0.5
    return [y]
