"""The products that users of cmpext3 run, as cases that can be timed and checked.

Every case goes through the Python operators (`fp16_matmul`, `bf16_matmul`,
`fp32_matmul`, `linear`, `bmm`, `conv2d`) on operands already on the GPU, the way a
model's forward pass calls them.  The sizes are those of this repository's benchmark,
tests and measured tables, from a call that is all launch overhead to the MLP product
of the benchmark.
"""
import torch

import cmpext3

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
MATMUL = {"fp16": cmpext3.fp16_matmul, "bf16": cmpext3.bf16_matmul, "fp32": cmpext3.fp32_matmul}


def _linear(dtype, m, n, k, bias=True):
    return {"op": "linear", "dtype": dtype, "m": m, "n": n, "k": k, "bias": bias}


def _matmul(dtype, m, n, k):
    return {"op": "matmul", "dtype": dtype, "m": m, "n": n, "k": k}


def _attention(dtype, heads, seq, dim):
    return {"op": "attention", "dtype": dtype, "heads": heads, "seq": seq, "dim": dim}


def _conv(dtype, batch, c_in, side, c_out, nhwc=False):
    return {"op": "conv2d", "dtype": dtype, "batch": batch, "c_in": c_in, "side": side, "c_out": c_out, "nhwc": nhwc}


def listed():
    return [
        # a small layer (a gate, a time embedding, an adapter): launch overhead and latency
        dict(_linear("fp16", 128, 512, 512), name="linear_fp16_small"),
        # a decoder's up-projection while it generates for 16 sequences: W read once
        dict(_linear("bf16", 16, 14336, 4096, False), name="linear_bf16_decode16"),
        # the same phase with 64 sequences, where rereading x starts to count
        dict(_linear("bf16", 64, 11008, 4096, False), name="linear_bf16_decode64"),
        # a square projection over a prompt of 1024 tokens: one tile for each CU
        dict(_linear("bf16", 1024, 4096, 4096), name="linear_bf16_prefill"),
        # the benchmark's headline product
        dict(_matmul("fp16", 4096, 4096, 4096), name="matmul_fp16_square"),
        # the benchmark's MLP product, the largest
        dict(_matmul("bf16", 4096, 14336, 4096), name="matmul_bf16_mlp"),
        # the benchmark's skinny product: B as [K, N], bound by reading it
        dict(_matmul("fp16", 16, 8192, 8192), name="matmul_fp16_skinny"),
        # odd rows and columns (a cropped batch, a vocabulary with added tokens)
        dict(_matmul("bf16", 4095, 4097, 4096), name="matmul_bf16_odd"),
        # the benchmark's ragged fp32 product: no row is 16-byte aligned
        dict(_matmul("fp32", 4097, 3001, 2049), name="matmul_fp32_ragged"),
        # a layer kept in fp32
        dict(_linear("fp32", 512, 4096, 4096), name="linear_fp32"),
        # one attention layer's two batched products: Q K^T on the transposed keys, then P V
        dict(_attention("fp16", 32, 1024, 128), name="attention_fp16"),
        # a bottleneck's 1x1 convolution late in an image network: few pixels per image
        dict(_conv("fp16", 32, 1024, 14, 256), name="conv2d_fp16_14x14"),
    ]


def _size(rng, lo, hi, step=1):
    """A size from lo to hi, uniform over its logarithm, rounded to a multiple of step."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(v / step)) * step))


def _whole(rng, lo, hi):
    """A model's width: a multiple of 8, 64 or 128."""
    return _size(rng, lo, hi, rng.choice([8, 64, 64, 128, 128]))


def draw(rng):
    while True:
        kind = rng.choice(["small", "decode", "decode", "linear", "linear", "matmul", "matmul", "odd", "fp32", "fp32",
                           "attention", "conv2d", "conv2d"])
        half = rng.choice(["fp16", "bf16"])
        if kind == "small":  # layers that cost a launch
            case = _linear(half, _size(rng, 65, 256), _whole(rng, 256, 2048), _whole(rng, 256, 2048), rng.random() < 0.7)
        elif kind == "decode":  # 1 to 64 rows against a large weight, as W^T or as B
            m, n, k = _size(rng, 1, 64), _whole(rng, 2048, 28672), _whole(rng, 2048, 14336)
            case = _matmul(half, m, n, k) if rng.random() < 0.3 else _linear(half, m, n, k, rng.random() < 0.3)
        elif kind == "linear":  # prompts and batches of any length
            case = _linear(half, _size(rng, 65, 8192), _whole(rng, 256, 14336), _whole(rng, 256, 14336), rng.random() < 0.5)
        elif kind == "matmul":
            case = _matmul(half, _size(rng, 65, 8192), _whole(rng, 64, 14336), _whole(rng, 64, 14336))
        elif kind == "odd":  # no size a multiple of anything
            case = _matmul(half, _size(rng, 65, 4200) | 1, _size(rng, 65, 4200) | 1, _size(rng, 256, 4200) | rng.choice([0, 1]))
        elif kind == "fp32":
            m = _size(rng, 16, 4200)
            if rng.random() < 0.5:
                case = _linear("fp32", m, _whole(rng, 128, 4096), _whole(rng, 128, 8192))
            else:
                case = _matmul("fp32", m, _size(rng, 128, 4200), _size(rng, 128, 4200))
        elif kind == "attention":
            case = _attention(half, _size(rng, 8, 128), _size(rng, 128, 2048, rng.choice([1, 8, 64, 128])), rng.choice([64, 128]))
        else:  # image networks: many pixels and few channels, or few pixels and many channels
            side = rng.choice([7, 14, 28, 32, 56, 64, 128])
            case = _conv(half, _size(rng, 1, 64), _whole(rng, 32, 2048), side, _whole(rng, 32, 2048), rng.random() < 0.25)
        w = work(case)
        limit = 5e10 if case["dtype"] == "fp32" else 1.4e11 if kind == "odd" else 4.8e11
        if w["flops"] <= limit and 1e6 <= w["bytes"] <= 4.1e8:  # (below, nothing but the call itself is timed)
            return case


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=gen, device="cuda").mul_(scale).to(dt)

    state = {"case": case}
    if case["op"] == "linear":  # activations, and weights scaled as a trained layer's are
        state["x"] = normal(case["m"], case["k"])
        state["w"] = normal(case["n"], case["k"], scale=case["k"] ** -0.5)
        state["b"] = normal(case["n"], scale=0.1) if case["bias"] else None
    elif case["op"] == "matmul":
        state["a"] = normal(case["m"], case["k"])
        state["b"] = normal(case["k"], case["n"], scale=case["k"] ** -0.5)
    elif case["op"] == "attention":  # P is a softmax's output, as P V has it in a model
        h, s, d = case["heads"], case["seq"], case["dim"]
        state["q"], state["k"], state["v"] = normal(h, s, d, scale=d ** -0.5), normal(h, s, d), normal(h, s, d)
        state["p"] = torch.softmax(torch.randn((h, s, s), generator=gen, device="cuda"), -1).to(dt)
    else:
        b, s = case["batch"], case["side"]
        state["x"] = normal(b, case["c_in"], s, s)
        if case["nhwc"]:
            state["x"] = state["x"].contiguous(memory_format=torch.channels_last)
        state["w"] = normal(case["c_out"], case["c_in"], 1, 1, scale=case["c_in"] ** -0.5)
        state["b"] = normal(case["c_out"], scale=0.1)
    return state


def run(state):
    case = state["case"]
    if case["op"] == "linear":
        return cmpext3.linear(state["x"], state["w"], state["b"])
    if case["op"] == "matmul":
        return MATMUL[case["dtype"]](state["a"], state["b"])
    if case["op"] == "attention":
        return [cmpext3.bmm(state["q"], state["k"].transpose(1, 2)), cmpext3.bmm(state["p"], state["v"])]
    return cmpext3.conv2d(state["x"], state["w"], state["b"])


def exact(case, seed):
    state = {k: v.double() if isinstance(v, torch.Tensor) else v for k, v in prepare(case, seed).items()}
    if case["op"] == "linear":
        out = state["x"] @ state["w"].t()
        return out if state["b"] is None else out + state["b"]
    if case["op"] == "matmul":
        return state["a"] @ state["b"]
    if case["op"] == "attention":
        keys = state["k"].transpose(1, 2).contiguous()
        return [torch.bmm(state["q"], keys), torch.bmm(state["p"], state["v"])]
    w = state["w"].flatten(1)
    out = torch.stack([w @ image.contiguous().flatten(1) for image in state["x"]])
    return out.view(*out.shape[:2], case["side"], case["side"]) + state["b"].view(1, -1, 1, 1)


def work(case):
    size = DTYPES[case["dtype"]].itemsize
    if case["op"] in ("linear", "matmul"):
        m, n, k = case["m"], case["n"], case["k"]
        values, flops = m * k + k * n + m * n + (n if case.get("bias") else 0), 2 * m * n * k
    elif case["op"] == "attention":
        h, s, d = case["heads"], case["seq"], case["dim"]
        values, flops = h * (4 * s * d + 2 * s * s), 4 * h * s * s * d
    else:
        pixels = case["batch"] * case["side"] ** 2
        values = pixels * (case["c_in"] + case["c_out"]) + case["c_out"] * (case["c_in"] + 1)
        flops = 2 * pixels * case["c_in"] * case["c_out"]
    return {"bytes": size * values, "flops": flops}


def tolerance(case):
    # sums in 32 bits and one rounding to the output's type: about four times the measured
    # distance from the 64-bit product (fp16 2.1e-4, bf16 1.7e-3, fp32 8.1e-7), and
    # at most two units in the last place of a value
    if case["dtype"] == "fp32":
        return {"rel": 4e-6, "max": 4e-5}
    return {"rel": 8e-4, "max": 2e-3} if case["dtype"] == "fp16" else {"rel": 6e-3, "max": 1.6e-2}
