"""The work a program gives this package, as timed cases.

A case is a plain dict. "kind" names the public entry point it goes through:

    layer    BinaryLinear_2_4(x): the linear layer on activations (tokens, k), the package's main use
    group    forward_grouped(layers, x): several projections of the same activations in one call
    product  PreparedWeight.matmul(b, c, alpha, beta): D = alpha A B + beta C on a weight reordered once
    onecall  cuda_binary_mul(A, B, meta): the stored operands straight into an fp32 product, nothing kept
    pack     BinaryLinear_2_4.pack(weight) and PreparedWeight(...): a dense weight into the stored format and on
             into the kernels' operand, as when a model's layers are converted

Weights are one-bit 2:4 sparse (m x k): signs uniform, one of the six two-of-four patterns per group of four,
uniformly. Activations and C are N(0, 1); the dense weights that pack() converts are N(0, 0.02), in the range of a
trained layer's. The unpacking functions (dequant_desparse_tile, py_binary_gemm) are host checks of the format and are
not timed.
"""
import math

import torch

from onebitsparsemul_amd import BinaryLinear_2_4, PreparedWeight, cuda_binary_mul, forward_grouped
from onebitsparsemul_amd import synthetic

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}


def listed():
    return [
        # one token through a square projection: the smallest call there is, latency and launches decide
        dict(name="layer_1_token", kind="layer", m=4096, k=4096, tokens=1, dtype="fp16", bias=False),
        # decoding sixteen sequences at once in a bf16 model, up projection
        dict(name="layer_16_tokens_bf16", kind="layer", m=11008, k=4096, tokens=16, dtype="bf16", bias=False),
        # q, k and v of one decoder layer for eight sequences
        dict(name="group_qkv_8_tokens", kind="group", rows="4096,4096,4096", k=4096, tokens=8, dtype="fp16"),
        # small batch through the down projection with the activations stored column by column
        dict(name="product_n4", kind="product", m=4096, k=11008, n=4, out="fp16", c="none", alpha=1.0, beta=0.0),
        # batched decoding on a large layer that has a bias
        dict(name="layer_48_tokens_bias", kind="layer", m=28672, k=8192, tokens=48, dtype="fp16", bias=True),
        # a prompt of no particular length in a bf16 model, down projection
        dict(name="layer_500_tokens_bf16", kind="layer", m=4096, k=11008, tokens=500, dtype="bf16", bias=False),
        # prefill with the residual added in the epilogue
        dict(name="product_prefill_c", kind="product", m=4096, k=4096, n=2048, out="fp16", c="fp16", alpha=0.5, beta=1.0),
        # a number of columns that no vector width divides
        dict(name="product_ragged_1001", kind="product", m=11008, k=4096, n=1001, out="fp16", c="none", alpha=1.0, beta=0.0),
        # the reference package's own call: stored operands in, fp32 out, the weight not prepared beforehand
        dict(name="onecall_256", kind="onecall", m=11008, k=4096, n=256),
        # the square product the throughput figure is quoted on
        dict(name="square_8192", kind="product", m=8192, k=8192, n=8192, out="fp16", c="none", alpha=1.0, beta=0.0),
        # the largest size of the reference's benchmark, with its flags: fp32 C and D, alpha = beta = 1
        dict(name="square_12800_fp32_c", kind="product", m=12800, k=12800, n=12800, out="fp32", c="fp32", alpha=1.0,
             beta=1.0),
        # converting one layer of a model
        dict(name="pack_fp16", kind="pack", m=11008, k=4096, dtype="fp16"),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _weight_shape(rng, most=28672 * 8192):
    """m a multiple of 64, k of 32 (what the stored format admits), each from 512 to 28672."""
    while True:
        m = int(_log_uniform(rng, 512, 28672)) // 64 * 64
        k = int(_log_uniform(rng, 512, 28672)) // 32 * 32
        if m * k <= most:
            return m, k


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "group", "product", "product", "product", "onecall", "pack"])
    m, k = _weight_shape(rng)
    if kind == "layer":
        # one to 64 tokens (decoding) as often as longer inputs (prompts)
        tokens = int(_log_uniform(rng, 1, 65) if rng.random() < 0.5 else _log_uniform(rng, 65, 4097))
        return dict(kind=kind, m=m, k=k, tokens=tokens, dtype=rng.choice(["fp16", "fp16", "bf16", "bf16", "fp32"]),
                    bias=rng.random() < 0.3)
    if kind == "group":
        m, k = _weight_shape(rng, 11008 * 4096)
        rows = [m, m] if rng.random() < 0.5 else [m, max(64, m // 4 // 64 * 64), max(64, m // 4 // 64 * 64)]
        return dict(kind=kind, rows=",".join(str(r) for r in rows), k=k, tokens=int(_log_uniform(rng, 1, 65)),
                    dtype=rng.choice(["fp16", "bf16"]))
    if kind == "product":
        most = 2 * 12800**3 / (2.0 * m * k)
        c = rng.choice(["none", "none", "fp16", "fp32"])
        return dict(kind=kind, m=m, k=k, n=int(min(_log_uniform(rng, 1, 8193), most)), out=rng.choice(["fp16", "fp16", "fp32"]),
                    c=c, alpha=rng.choice([1.0, 0.5]), beta=0.0 if c == "none" else rng.choice([1.0, 0.25]))
    if kind == "onecall":
        return dict(kind=kind, m=m, k=k, n=int(_log_uniform(rng, 1, 2049)))
    m, k = _weight_shape(rng, 11008 * 4096)
    return dict(kind=kind, m=m, k=k, dtype=rng.choice(["fp16", "fp16", "bf16"]))


def _layer(m, k, seed, bias=False):
    layer = BinaryLinear_2_4(k, m).to("cuda")
    a, meta = synthetic.make_weight(m, k, seed, device="cuda")
    layer.load_state_dict({"packed_binary_sparse": a, "meta": meta})
    if bias:
        layer.bias = synthetic.make_c(1, m, seed + 7, device="cuda").reshape(m)
    return layer


def _normal(rows, cols, seed, dtype, std=1.0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return (torch.randn((rows, cols), generator=g, device="cuda", dtype=torch.float32) * std).to(DTYPES[dtype])


def _rows(case):
    return [int(r) for r in case["rows"].split(",")]


def prepare(case, seed):
    """Layers and prepared weights are what a program keeps between calls; activations are there in its own dtype."""
    kind, k = case["kind"], case["k"]
    seed = 16 * seed  # sixteen seeds for one state's tensors
    if kind == "layer":
        return dict(kind=kind, layer=_layer(case["m"], k, seed, case["bias"]),
                    x=_normal(case["tokens"], k, seed + 8, case["dtype"]))
    if kind == "group":
        return dict(kind=kind, layers=[_layer(m, k, seed + i) for i, m in enumerate(_rows(case))],
                    x=_normal(case["tokens"], k, seed + 8, case["dtype"]))
    m = case["m"]
    if kind == "pack":
        return dict(kind=kind, layer=BinaryLinear_2_4(k, m).to("cuda"), weight=_normal(m, k, seed + 8, case["dtype"], 0.02))
    a, meta = synthetic.make_weight(m, k, seed, device="cuda")
    b = synthetic.make_b(k, case["n"], seed + 8, device="cuda")
    if kind == "onecall":
        return dict(kind=kind, a=a, meta=meta, b=b)
    c = None if case["c"] == "none" else synthetic.make_c(m, case["n"], seed + 8, dtype=DTYPES[case["c"]], device="cuda")
    return dict(kind=kind, weight=PreparedWeight(a, meta), b=b, c=c, alpha=case["alpha"], beta=case["beta"],
                out_dtype=DTYPES[case["out"]])


def run(state):
    kind = state["kind"]
    if kind == "layer":
        return state["layer"](state["x"])
    if kind == "group":
        return forward_grouped(state["layers"], state["x"])
    if kind == "product":
        return state["weight"].matmul(state["b"], c=state["c"], alpha=state["alpha"], beta=state["beta"],
                                      out_dtype=state["out_dtype"])
    if kind == "onecall":
        return cuda_binary_mul(state["a"], state["b"], state["meta"])
    layer = state["layer"]
    layer.pack(state["weight"])
    prepared = PreparedWeight(layer.packed_binary_sparse, layer.meta)
    return dict(packed=layer.packed_binary_sparse, meta=layer.meta, prepared=prepared.buffer)


def work(case):
    """Bytes: the weight at 1.5 bits (one sign bit per kept value, two position bits), activations, C and the result in
    their own types. flops: 2 m n k of the dense product (the reference's own count; half of the weight's entries are
    zeros)."""
    kind, k = case["kind"], case["k"]
    if kind in ("layer", "group"):
        rows = case["m"] if kind == "layer" else sum(_rows(case))
        t, size = case["tokens"], BYTES[case["dtype"]]
        bias = 2 * rows if case.get("bias") else 0
        return {"bytes": rows * k * 3 // 16 + size * t * (k + rows) + bias, "flops": 2.0 * rows * t * k}
    m = case["m"]
    if kind == "pack":  # dense weight in; stored operands and the kernels' operand out, both 1.5 bits per weight
        return {"bytes": m * k * BYTES[case["dtype"]] + 2 * (m * k * 3 // 16), "flops": 0}
    n = case["n"]
    out = 4 if kind == "onecall" else BYTES[case["out"]]
    c = 0 if kind == "onecall" or case["c"] == "none" else BYTES[case["c"]]
    return {"bytes": m * k * 3 // 16 + 2 * k * n + (out + c) * m * n, "flops": 2.0 * m * n * k}


def tolerance(case):
    """Packing and reordering are bit manipulations. Products accumulate in fp32 and round once to the result's type;
    fp32 activations are rounded to fp16 first. Measured against the same product in fp64 (rel, max): fp16 2.1e-4,
    4.9e-4; bf16 1.7e-3, 3.9e-3; fp32 results 7.2e-8, 4.1e-7 (K = 12800); the bounds are about four times that."""
    if case["kind"] == "pack":
        return "exact"
    if case.get("dtype") == "fp32":
        return {"rel": 8e-4, "max": 4e-3}
    out = "fp32" if case["kind"] == "onecall" else case.get("out") or case["dtype"]
    return {"fp16": {"rel": 8e-4, "max": 2e-3}, "bf16": {"rel": 6.6e-3, "max": 1.6e-2}, "fp32": {"rel": 5e-7, "max": 4e-6}}[out]
