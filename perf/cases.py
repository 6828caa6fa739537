"""The work that users of this package have it do, as timed cases with inputs, outputs and tolerances.

A case is a dict of plain values; `kind` says which public entry point it goes through:

- "mm": one `scaled_mm_hip` call, M activation rows by a prepacked fp8 weight;
- "decode": the feed-forward weights of `layers` decoder layers, one call each on the same few rows. The weights
  together are larger than the GPU's 256 MB last-level cache, as a decoder's are, so each call reads its own from HBM;
- "linear": inference through an `nn.Linear` relabelled by `to_scaled_mm_linear`;
- "train": forward and backward of such a layer under trainable adapters: gradients for the input and the bias;
- "quantize": quantizing and laying out such a layer's weight (after loading or changing it);
- "prepack": laying out an fp8 weight that was stored as a Linear's [N, K] ("nk": its transposed view is what
  `prepack_b_for_scaled_mm` gets) or as [K, N] ("kn").

Sizes are `m` rows, `n` output columns and `k` inputs. `a` is the activations' and the output's type, `w` the weight's;
`column` selects one scale per output column instead of one per tensor.
"""

import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "feather-ops_amd"))

import feather_ops  # noqa: E402
from feather_ops.scaled_mm import prepack_b_for_scaled_mm, scaled_mm_hip  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "e5m2": torch.float8_e5m2, "e4m3": torch.float8_e4m3fn}
FP8_MAX = {"e5m2": 57344.0, "e4m3": 448.0}
DEVICE = "cuda"


def listed():
    return [
        # The smallest call: one row (a modulation or time-step vector) through a small layer; launch latency.
        dict(name="row-1", kind="mm", m=1, n=1000, k=2560, a="bf16", w="e5m2", column=False, bias=False),
        # A decoding step of 16 sequences: up and down projections of four layers, weights from HBM.
        dict(name="decode-16", kind="decode", m=16, n=14336, k=4096, layers=4, a="fp16", w="e5m2", column=False),
        # The 77 text tokens of a prompt through a cross-attention projection.
        dict(name="text-77", kind="mm", m=77, n=5120, k=2560, a="bf16", w="e5m2", column=False, bias=True),
        # A prompt of 512 tokens through a text stream's MLP.
        dict(name="prompt-512", kind="mm", m=512, n=13824, k=5120, a="fp16", w="e4m3", column=True, bias=False),
        # The attention projection of a diffusion transformer at 4096 image tokens.
        dict(name="attn-4096", kind="mm", m=4096, n=3072, k=3072, a="bf16", w="e5m2", column=False, bias=False),
        # Its MLP's up projection, the headline configuration.
        dict(name="mlp-4096", kind="mm", m=4096, n=12288, k=3072, a="fp16", w="e5m2", column=False, bias=False),
        # Image tokens plus one: no dimension's last tile is full.
        dict(name="ragged-4097", kind="mm", m=4097, n=5120, k=2560, a="bf16", w="e5m2", column=False, bias=True),
        # A whole layer of a model as its user has it: 4096 image and 16 text tokens through an MLP's down projection.
        dict(name="linear-4112", kind="linear", m=4112, n=4096, k=12288, a="bf16", w="e4m3", column=True, bias=True),
        # Training adapters on a frozen quantized model: the MLP's up projection, forward and backward.
        dict(name="train-4096", kind="train", m=4096, n=12288, k=3072, a="bf16", w="e5m2", column=False, bias=True),
        # The same on a smaller layer and a ragged batch, with the weight quantized by column.
        dict(name="train-1000", kind="train", m=1000, n=5120, k=2560, a="fp16", w="e4m3", column=True, bias=True),
        # Loading a layer: its bf16 weight is quantized and laid out.
        dict(name="quantize", kind="quantize", n=12288, k=3072, a="bf16", w="e4m3", column=True, bias=False),
        # Loading an fp8 checkpoint's weight, stored [N, K] as Linear weights are.
        dict(name="prepack", kind="prepack", n=14336, k=4096, w="e5m2", order="nk"),
    ]


# The largest listed products: no drawn case costs more.
MAX_MNK = 4096 * 12288 * 3072
MAX_DECODE_WEIGHT = 14336 * 4096
MAX_LOAD_WEIGHT = 12288 * 3072


def draw(rng):
    def size(low, high, step=1):
        """A multiple of `step`, evenly spread over the logarithm."""
        value = low * (high / low) ** rng.random()
        return min(high, max(low, round(value / step) * step))

    kind = rng.choice(["mm", "mm", "mm", "mm", "decode", "linear", "train", "train", "quantize", "prepack"])
    a, w = rng.choice(["fp16", "bf16"]), rng.choice(["e5m2", "e4m3"])
    column, bias = rng.random() < 0.5, rng.random() < 0.5
    while True:
        n, k = size(1000, 16384, 8), size(1024, 16384, 16)
        if kind in ("quantize", "prepack"):
            if n * k > MAX_LOAD_WEIGHT:
                continue
            if kind == "quantize":
                return dict(kind=kind, n=n, k=k, a=a, w=w, column=column, bias=False)
            return dict(kind=kind, n=n, k=k, w=w, order=rng.choice(["nk", "nk", "kn"]))
        if kind == "decode":
            if not 0.5 * MAX_DECODE_WEIGHT < n * k <= MAX_DECODE_WEIGHT or n % 16:  # n is the down projection's depth
                continue
            return dict(kind=kind, m=size(1, 64), n=n, k=k, layers=4, a=a, w=w, column=column)
        m = size(64, 4112) if kind == "train" else size(1, 9232)
        if m * n * k > MAX_MNK:
            continue
        return dict(kind=kind, m=m, n=n, k=k, a=a, w=w, column=column, bias=True if kind == "train" else bias)


def _weight(case, n, k, g):
    """An fp8 weight [n, k] with its scale, quantized as `to_scaled_mm_linear` does."""
    w = torch.randn((n, k), generator=g, device=DEVICE) * k**-0.5
    amax = w.abs().amax(dim=1, keepdim=True) if case["column"] else w.abs().max()
    scale = amax / FP8_MAX[case["w"]]
    return (w / scale).to(DTYPES[case["w"]]), scale.reshape(-1) if case["column"] else scale


def _rows(case, k, g):
    return torch.randn((case["m"], k), generator=g, device=DEVICE).to(DTYPES[case["a"]])


def _inputs(case, seed):
    """The raw inputs of a case, from the seed alone."""
    g = torch.Generator(DEVICE).manual_seed(seed)
    kind, n, k = case["kind"], case["n"], case["k"]
    if kind == "prepack":
        shape = (n, k) if case["order"] == "nk" else (k, n)
        return {"w": torch.randn(shape, generator=g, device=DEVICE).to(DTYPES[case["w"]])}
    if kind == "decode":
        return {"pairs": [(_rows(case, kk, g), *_weight(case, nn, kk, g))
                          for _ in range(case["layers"]) for nn, kk in ((n, k), (k, n))]}
    dtype = DTYPES[case["a"]]
    if kind == "mm":
        w, scale = _weight(case, n, k, g)
        return {"x": _rows(case, k, g), "w": w, "scale": scale,
                "bias": torch.randn(n, generator=g, device=DEVICE).to(dtype) if case["bias"] else None}
    got = {"weight": (torch.randn((n, k), generator=g, device=DEVICE) * k**-0.5).to(dtype)}
    if case["bias"]:
        got["bias"] = torch.randn(n, generator=g, device=DEVICE).to(dtype)
    if kind in ("linear", "train"):
        got["x"] = _rows(case, k, g)
    if kind == "train":  # gradients are small next to the activations, with a few larger ones
        grad = torch.randn((case["m"], n), generator=g, device=DEVICE)
        got["grad"] = (grad * grad.abs() * 1e-3).to(dtype)
    return got


def _linear(case, inputs):
    lin = torch.nn.Linear(case["k"], case["n"], bias=case["bias"], device="meta", dtype=DTYPES[case["a"]])
    lin.weight = torch.nn.Parameter(inputs["weight"], requires_grad=False)
    if case["bias"]:
        lin.bias = torch.nn.Parameter(inputs["bias"], requires_grad=case["kind"] == "train")
    feather_ops.to_scaled_mm_linear(lin, DTYPES[case["w"]], per_channel=case["column"])
    return lin


def prepare(case, seed):
    inputs = _inputs(case, seed)
    kind = case["kind"]
    if kind == "prepack":
        return {"kind": kind, "b": inputs["w"].t() if case["order"] == "nk" else inputs["w"]}
    if kind == "decode":
        return {"kind": kind, "dtype": DTYPES[case["a"]],
                "calls": [(x, prepack_b_for_scaled_mm(w.t()), scale) for x, w, scale in inputs["pairs"]]}
    if kind == "mm":
        return {"kind": kind, "dtype": DTYPES[case["a"]], "x": inputs["x"], "scale": inputs["scale"],
                "b": prepack_b_for_scaled_mm(inputs["w"].t()), "bias": inputs["bias"]}
    state = {"kind": kind, "lin": _linear(case, inputs)}
    if kind == "quantize":
        state["w"], state["column"] = DTYPES[case["w"]], case["column"]
    else:
        state["x"] = inputs["x"][None]  # [batch, tokens, inputs]
    if kind == "train":
        state["x"].requires_grad_()
        state["grad"] = inputs["grad"][None]
    return state


def run(state):
    kind = state["kind"]
    if kind == "mm":
        return scaled_mm_hip(state["x"], state["b"], state["scale"], state["bias"], state["dtype"])
    if kind == "decode":
        return [scaled_mm_hip(x, b, scale, None, state["dtype"]) for x, b, scale in state["calls"]]
    if kind == "prepack":
        return prepack_b_for_scaled_mm(state["b"])
    lin = state["lin"]
    if kind == "quantize":
        lin.quantize_weight_(state["w"], state["column"])
        return {"weight": lin.weight_fp8, "scale": lin.weight_scale}
    if kind == "linear":
        with torch.no_grad():
            return lin(state["x"])
    y = lin(state["x"])
    grad_x, grad_bias = torch.autograd.grad(y, (state["x"], lin.bias), state["grad"])
    return {"y": y.detach(), "grad_x": grad_x, "grad_bias": grad_bias}


def work(case):
    kind, n, k = case["kind"], case["n"], case["k"]
    k_pad = -(-k // 128) * 128
    if kind == "prepack":
        return {"bytes": n * k + n * k_pad, "flops": 0}
    scales = 4 * (n if case["column"] else 1)
    if kind == "quantize":
        return {"bytes": 2 * n * k + n * k_pad + scales, "flops": n * k}
    m = case["m"]
    if kind == "decode":
        one = n * k + 2 * m * (n + k)
        return {"bytes": 2 * case["layers"] * one, "flops": 4 * case["layers"] * m * n * k}
    bias = 2 * n if case["bias"] else 0
    forward = {"bytes": n * k + 2 * m * (n + k) + scales + bias, "flops": 2 * m * n * k}
    if kind != "train":
        return forward
    # backward: the gradient and the weight in, the input's and the bias's gradients out
    return {"bytes": forward["bytes"] + n * k + 2 * m * (n + k) + scales + bias, "flops": 2 * forward["flops"] + m * n}


def tolerance(case):
    """About four times what the path shows against `exact`: half a unit of the output's type per element, and the
    bias's addition once more in that type; layouts, scales and fp8 codes are the same bytes."""
    if case["kind"] in ("prepack", "quantize"):
        return "exact"
    return {"rel": 8e-3, "max": 2e-2} if case["a"] == "bf16" else {"rel": 1e-3, "max": 2.5e-3}


def _dequantized(w, scale):
    return w.double() * (scale.double()[:, None] if scale.dim() else scale.double())


def _quantized(case, weight):
    """The fp8 codes [n, k] and scale of a layer's weight: the scale is held in 32 bits, the quotient is not."""
    amax = weight.float().abs().amax(dim=1) if case["column"] else weight.float().abs().max()
    scale = amax / FP8_MAX[case["w"]]
    return (weight.double() / (scale.double()[:, None] if case["column"] else scale.double())).to(DTYPES[case["w"]]), scale


def _packed(w):
    """[n, k] -> [k_pad / 16, n, 16], zero-padded."""
    n, k = w.shape
    w = torch.nn.functional.pad(w, (0, -k % 128))
    return w.view(n, -1, 16).transpose(0, 1).contiguous()


def exact(case, seed):
    inputs = _inputs(case, seed)
    kind = case["kind"]
    if kind == "prepack":
        return _packed(inputs["w"].double() if case["order"] == "nk" else inputs["w"].double().t())
    if kind == "decode":
        return [x.double() @ _dequantized(w, scale).t() for x, w, scale in inputs["pairs"]]
    if kind == "mm":
        y = inputs["x"].double() @ _dequantized(inputs["w"], inputs["scale"]).t()
        return y if inputs["bias"] is None else y + inputs["bias"].double()
    w, scale = _quantized(case, inputs["weight"])
    if kind == "quantize":
        return {"weight": _packed(w.double()), "scale": scale.double()}
    w = _dequantized(w, scale)
    y = (inputs["x"].double() @ w.t())[None]
    if case["bias"]:
        y = y + inputs["bias"].double()
    if kind == "linear":
        return y
    grad = inputs["grad"].double()
    return {"y": y, "grad_x": (grad @ w)[None], "grad_bias": grad.sum(0)}
