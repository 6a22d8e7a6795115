"""What a program that runs ternary models has this library do, as cases to be measured.

Four kinds of case, each through the package's public entry points:

* ``linear``: one ``TernaryLinear`` module called on ``tokens`` rows of activations in the caller's
  data type (float32, or the half types of a surrounding torch model), with or without a bias, at
  batch sizes from one decode token to a long prompt and at any width, tile-aligned or not;
* ``layer``: one decoder layer as a decoder launches it, on resident operands: RMSNorm + fused QKV,
  the split-softmax merge of the attention's partial results + output projection added to the
  residual, RMSNorm + gated MLP, down projection added to the residual (the token's GEMVs for one
  token, quantize + token GEMM for several);
* ``prefill``: ``StackDecoder.prefill`` of a whole prompt, ending with its last token's logits;
* ``generate``: a prompt and the tokens after it, greedy (``top_k`` 0) or drawn by the device sampler.

Sizes are the package's own workloads (1024 -> 4096, 4096 -> 14336, 8192 <-> 28672, the 24-layer
d=1024 stack with a vocabulary of 32000) or generic ones between and around them.  Weights are random
ternary codes with positive fp16 group scales, activations Gaussian with a few outlier channels or
heavy-tailed, as quantized transformers meet them.
"""

from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ivonar-inference_amd"))

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
GROUP = 128
HEAD_DIM = 64
EPS = 1e-6
MOST_LAYER_FLOPS = 2 * 2048 * 4096 * 14336  # a drawn linear or layer stays within the longest prompt listed,
MOST_STACK = {"bytes": 7.6e9, "flops": 4.0e11}  # a drawn prompt or answer within the listed ones


def listed():
    return [
        # one projection of a small model at one decode token: the smallest call there is
        {"name": "linear token 1024-4096", "kind": "linear", "tokens": 1, "k": 1024, "n": 4096, "dtype": "f32",
         "bias": False},
        # a half-precision model decoding eight sequences at once
        {"name": "linear batch 8 4096-14336", "kind": "linear", "tokens": 8, "k": 4096, "n": 14336, "dtype": "bf16",
         "bias": False},
        # a short prompt through a layer whose widths fit no tile, with a bias
        {"name": "linear 77 1100-3334 bias", "kind": "linear", "tokens": 77, "k": 1100, "n": 3334, "dtype": "f32",
         "bias": True},
        # a prompt through the down projection of a small model in half precision
        {"name": "linear 500 4096-1024", "kind": "linear", "tokens": 500, "k": 4096, "n": 1024, "dtype": "f16",
         "bias": False},
        # the longest prompt chunk through the widest projection of a mid-sized model
        {"name": "linear 2048 4096-14336", "kind": "linear", "tokens": 2048, "k": 4096, "n": 14336, "dtype": "f32",
         "bias": False},
        # one decode token through a layer of a large model: the weights are the work
        {"name": "layer token 8192/28672", "kind": "layer", "tokens": 1, "hidden": 8192, "dense": 28672, "splits": 4},
        # a dozen sequences decoding together through the same layer
        {"name": "layer batch 12 8192/28672", "kind": "layer", "tokens": 12, "hidden": 8192, "dense": 28672,
         "splits": 2},
        # a medium prompt through a layer of the small model
        {"name": "layer 300 1024/4096", "kind": "layer", "tokens": 300, "hidden": 1024, "dense": 4096, "splits": 1},
        # a prompt of odd length through a layer of a mid-sized model
        {"name": "layer 777 4096/11008", "kind": "layer", "tokens": 777, "hidden": 4096, "dense": 11008, "splits": 1},
        # reading a page of text with the 24-layer stack
        {"name": "prefill 500", "kind": "prefill", "prompt": 500, "layers": 24, "hidden": 1024, "dense": 4096,
         "vocab": 32000},
        # a short question and a greedy answer
        {"name": "generate 36+65 greedy", "kind": "generate", "prompt": 36, "count": 65, "top_k": 0, "layers": 24,
         "hidden": 1024, "dense": 4096, "vocab": 32000},
        # the same with the device sampler as a chat program sets it
        {"name": "generate 36+33 top-k 40", "kind": "generate", "prompt": 36, "count": 33, "top_k": 40, "layers": 24,
         "hidden": 1024, "dense": 4096, "vocab": 32000},
    ]


# ------------------------------------------------------------------ drawn cases


def _log_int(rng, low, high, step=1):
    """A multiple of step between low and high, spread over the logarithm."""
    value = math.exp(rng.uniform(math.log(low), math.log(high + 1)))
    return max(low, min(high, int(value) // step * step))


def _width(rng, low, high, finest):
    """A layer width: half of them multiples of 128, the others of 64, 4 or `finest`."""
    return _log_int(rng, low, high, rng.choice((128, 128, 128, 64, 4, finest)))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "layer", "layer", "prefill", "generate"))
    while True:
        if kind == "linear":
            case = {"kind": kind, "tokens": _log_int(rng, 1, 2048), "k": _width(rng, 256, 28672, 1),
                    "n": _width(rng, 256, 28672, 2), "dtype": rng.choice(("f32", "f32", "bf16", "f16")),
                    "bias": rng.random() < 0.25}
        elif kind == "layer":
            case = {"kind": kind, "tokens": _log_int(rng, 1, 2048), "hidden": _log_int(rng, 512, 8192, 64),
                    "dense": _log_int(rng, 1024, 28672, rng.choice((128, 128, 4))), "splits": rng.choice((1, 2, 4, 8))}
        else:
            case = {"kind": kind, "prompt": _log_int(rng, 1, 1024 if kind == "prefill" else 128)}
            if kind == "generate":
                case["count"] = _log_int(rng, 8, 96)
                case["top_k"] = 0 if rng.random() < 0.5 else _log_int(rng, 1, 256)
            case.update(layers=rng.randint(4, 24), hidden=_log_int(rng, 512, 2048, 64),
                        dense=_log_int(rng, 1024, 8192, 128), vocab=_log_int(rng, 1000, 64000))
        cost = work(case)
        most = {"flops": MOST_LAYER_FLOPS} if kind in ("linear", "layer") else MOST_STACK
        if all(cost[key] <= limit for key, limit in most.items()):
            return case


# ------------------------------------------------------------------ inputs


def _generator(seed, part=0):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + part)


def _nibbles(probabilities):
    """All 10000 bytes of four codes, as often as the probabilities (tenths) of codes 0, 1, 2 ask."""
    digit = np.repeat(np.arange(3), probabilities).astype(np.int64)
    index = np.arange(10000)
    value = sum(digit[index // 10 ** f % 10] << (2 * f) for f in range(4))
    return torch.from_numpy(value.astype(np.uint8)).cuda()


def _ternary(generator, rows, k, sigma=0.02, probabilities=(3, 4, 3)):
    """Packed codes uint8 [rows, ceil(k/4)] (codes past k are 1, the zero weight) and fp16 scales."""
    width = -(-k // 4)
    table = _nibbles(probabilities)
    packed = torch.empty((rows, width), dtype=torch.uint8, device="cuda")
    for start in range(0, rows, 4096):
        part = packed[start:start + 4096]
        part.copy_(table[torch.randint(0, 10000, part.shape, generator=generator, device="cuda", dtype=torch.int32)])
    if k % 4:
        keep = (1 << (2 * (k % 4))) - 1
        packed[:, -1] = (packed[:, -1] & keep) | (0x55 & ~keep)
    groups = -(-k // GROUP)
    scales = torch.randn((rows, groups), generator=generator, device="cuda").mul_(sigma).abs_().add_(1e-4).half()
    return packed, scales


def _activations(generator, tokens, k):
    """N(0, 1) with 1% of the channels twenty times as large."""
    x = torch.randn((tokens, k), generator=generator, device="cuda")
    channels = torch.randperm(k, generator=generator, device="cuda")[:max(1, k // 100)]
    x[:, channels] *= 20.0
    return x


def _norm_weight(generator, k):
    return 1.0 + 0.1 * torch.randn(k, generator=generator, device="cuda")


def _linear_inputs(case, seed):
    g = _generator(seed)
    tokens, k, n = case["tokens"], case["k"], case["n"]
    # weights of the wide projections are sparser and their activations heavy-tailed
    skewed = k >= 2048
    packed, scales = _ternary(g, n, k, probabilities=(2, 6, 2) if skewed else (3, 4, 3))
    bias = 0.02 * torch.randn(n, generator=g, device="cuda") if case["bias"] else None
    if skewed:
        normal = torch.randn((4, tokens, k), generator=g, device="cuda")
        x = normal[0] / (normal[1:].square().sum(0) / 3.0).sqrt()  # Student-t with three degrees of freedom
    else:
        x = _activations(g, tokens, k)
    return packed, scales, bias, x.to(DTYPES[case["dtype"]])


def _layer_inputs(case, seed):
    g = _generator(seed)
    tokens, hidden, dense, splits = case["tokens"], case["hidden"], case["dense"], case["splits"]
    weights = {"entry": _ternary(g, 3 * hidden, hidden), "out": _ternary(g, hidden, hidden),
               "gate": _ternary(g, dense, hidden), "up": _ternary(g, dense, hidden),
               "down": _ternary(g, hidden, dense)}
    norms = _norm_weight(g, hidden), _norm_weight(g, hidden)
    residual = _activations(g, tokens, hidden)
    heads = hidden // HEAD_DIM
    partials = torch.randn((tokens, heads, splits, HEAD_DIM + 2), generator=g, device="cuda")
    partials[..., 1] = partials[..., 1].abs() + 0.5  # each split's peak, its weight total, then its weighted values
    return weights, norms, residual, partials


def _stack_inputs(case, seed):
    """The decoder's weights on the host, as a loader hands them over, and the prompt's ids."""
    from ivonar_amd import synthetic

    g = _generator(seed)
    hidden, dense, vocab = case["hidden"], case["dense"], case["vocab"]
    config = synthetic.StackConfig(vocab=vocab, hidden=hidden, layers=case["layers"], dense=dense, eps=EPS)

    def layer(rows, k):
        packed, scales = _ternary(g, rows, k)
        return synthetic.Layer(packed.cpu().numpy(), scales.cpu().numpy(), k)

    def norm():
        return _norm_weight(g, hidden).cpu().numpy()

    token = layer(vocab, hidden)
    layers = [synthetic.StackLayer(qkv=layer(3 * hidden, hidden), out=layer(hidden, hidden),
                                   gate=layer(dense, hidden), up=layer(dense, hidden), down=layer(hidden, dense),
                                   mixer_norm=norm(), ffn_norm=norm()) for _ in range(case["layers"])]
    weights = synthetic.LinearStackWeights(config, token, layers, norm())
    ids = torch.randint(min(2, vocab - 1), vocab, (case["prompt"],), generator=g, device="cuda").tolist()
    return weights, ids


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        from ivonar_amd.quantization import TernaryLinear

        packed, scales, bias, x = _linear_inputs(case, seed)
        module = TernaryLinear(packed, scales, case["k"], bias)
        module.matrix()  # the layer's device operand, laid out once when a model is loaded
        return SimpleNamespace(kind=kind, module=module, x=x)
    if kind == "layer":
        return _prepare_layer(case, seed)

    from ivonar_amd.decoder import StackDecoder

    weights, ids = _stack_inputs(case, seed)
    top_k = case.get("top_k", 0)
    decoder = StackDecoder(weights, "cuda", sampling=top_k > 0)
    if top_k > 0:
        decoder.configure_sampling(0.8, top_k, 1.1)
    decoder.capture()
    return SimpleNamespace(kind=kind, decoder=decoder, ids=ids, count=case.get("count", 0), seed=int(seed))


def _prepare_layer(case, seed):
    from ivonar_amd import ops
    from ivonar_amd.matrix import Matrix
    from ivonar_amd.quantization import TernaryLinear

    weights, norms, residual, partials = _layer_inputs(case, seed)
    tokens, hidden, dense = case["tokens"], case["hidden"], case["dense"]
    device = residual.device

    def linear(name):
        return TernaryLinear(*weights[name], dense if name == "down" else hidden)

    state = SimpleNamespace(
        kind="layer", tokens=tokens, hidden=hidden, splits=case["splits"], norms=norms, residual=residual,
        partials=partials.reshape(tokens, -1),
        entry=Matrix([linear("entry")], device), out=Matrix([linear("out")], device),
        gate_up=Matrix([linear("gate"), linear("up")], device, interleave=True, max_lanes=16),
        down=Matrix([linear("down")], device),
        mixer_in=torch.empty((tokens, 3 * hidden), device=device), mid=torch.empty((tokens, dense), device=device),
    )
    if tokens > 1:
        state.wide = ops.activation_buffers(tokens, hidden, device)
        state.tall = ops.activation_buffers(tokens, dense, device)
    return state


# ------------------------------------------------------------------ one pass


def run(state):
    if state.kind == "linear":
        return state.module(state.x)
    if state.kind == "layer":
        return _run_token(state) if state.tokens == 1 else _run_tokens(state)
    decoder = state.decoder
    if state.kind == "prefill":
        return decoder.prefill(state.ids)
    if decoder.sampler is not None:
        torch.cuda.manual_seed(state.seed)  # a seeded answer, as a user asks for one
    decoder.reset()
    first = decoder.prefill(state.ids).clone()
    return {"first": first, "tokens": torch.tensor(decoder.advance_many(state.count)), "logits": decoder.logits}


def _run_token(s):
    from ivonar_amd import ops

    ops.gemv(s.entry, s.residual[0], out=s.mixer_in[0], mode="norm", aux=s.norms[0], eps=EPS)
    ops.gemv(s.out, s.partials[0], out=s.residual[0], mode="attn", epilogue="residual", splits=s.splits)
    ops.gemv(s.gate_up, s.residual[0], out=s.mid[0], mode="norm", epilogue="silu_pair", aux=s.norms[1], eps=EPS)
    ops.gemv(s.down, s.mid[0], out=s.residual[0], epilogue="residual")
    return {"mixer_in": s.mixer_in, "mid": s.mid, "residual": s.residual}


def _run_tokens(s):
    from ivonar_amd import ops

    ops.quantize_rows(s.residual, ops.MODE_NORM, s.norms[0], EPS, out=s.wide)
    ops.gemm(s.entry, *s.wide, out=s.mixer_in)
    ops.quantize_rows(s.partials, ops.MODE_ATTN, splits=s.splits, n=s.hidden, out=s.wide)
    ops.gemm(s.out, *s.wide, out=s.residual, epilogue="residual")
    ops.quantize_rows(s.residual, ops.MODE_NORM, s.norms[1], EPS, out=s.wide)
    ops.gemm(s.gate_up, *s.wide, out=s.mid, epilogue="silu_pair")
    ops.quantize_rows(s.mid, out=s.tall)
    ops.gemm(s.down, *s.tall, out=s.residual, epilogue="residual")
    return {"mixer_in": s.mixer_in, "mid": s.mid, "residual": s.residual}


# ------------------------------------------------------------------ what a pass cannot do without


def _matrix_bytes(n, k):
    return n * -(-k // 4) + 2 * n * -(-k // GROUP)


def _layer_shapes(hidden, dense):
    return (3 * hidden, hidden), (hidden, hidden), (2 * dense, hidden), (hidden, dense)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["tokens"], case["k"], case["n"]
        element = 4 if case["dtype"] == "f32" else 2
        return {"bytes": _matrix_bytes(n, k) + element * m * k + 4 * m * n + (4 * n if case["bias"] else 0),
                "flops": 2 * m * k * n}
    hidden, dense = case["hidden"], case["dense"]
    weights = sum(_matrix_bytes(n, k) for n, k in _layer_shapes(hidden, dense))
    products = sum(n * k for n, k in _layer_shapes(hidden, dense))
    if kind == "layer":
        m = case["tokens"]
        partials = hidden // HEAD_DIM * case["splits"] * (HEAD_DIM + 2)
        # in: residual, partials, norm weights; out: mixer input, MLP middle, residual
        return {"bytes": weights + 4 * m * (hidden + partials + 3 * hidden + dense + hidden) + 8 * hidden,
                "flops": 2 * m * products}
    vocab, count = case["vocab"], case.get("count", 0)
    stack = case["layers"] * (weights + 8 * hidden)
    head = _matrix_bytes(vocab, hidden) + 4 * hidden + 4 * vocab
    tokens = case["prompt"] + count
    # the stack's weights once for the prompt and once for every token after it, the head once for each choice
    return {"bytes": (1 + count) * (stack + head) + tokens * _matrix_bytes(1, hidden),
            "flops": 2 * (tokens * case["layers"] * products + (1 + count) * vocab * hidden)}


def tolerance(case):
    """Four times what the paths show against exact().

    The sums themselves are good to 1e-7.  What shows is a quotient next to a half that rounds to the
    other int8 value where its fp32 row came out an ulp apart: one such value in one token of a linear;
    in a layer also in the rows that follow from sums; and through a stack every such value moves the
    rows of the layers behind it, up to the size of the int8 rounding itself (0.01 to 0.04 of the
    logits)."""
    if case["kind"] == "linear":
        return {"rel": 2e-3, "max": 0.1}
    if case["kind"] == "layer":
        return {"rel": 3e-3, "max": 0.3}
    return {"rel": 0.1, "max": 0.5, "differ": 0.1}


# ------------------------------------------------------------------ the same in 64 bits


def _weights64(packed, scales, k):
    """code * scale in float64 [rows, k]."""
    fields = torch.stack([(packed >> (2 * f)) & 3 for f in range(4)], dim=-1).reshape(packed.shape[0], -1)[:, :k]
    return (fields.double() - 1.0).mul_(scales.double().repeat_interleave(GROUP, dim=1)[:, :k])


def _quantized64(v):
    """Per-token absmax int8 values of float64 rows, scaled back."""
    scale = (v.abs().amax(dim=-1, keepdim=True) / 127.0).clamp_min(1e-5)
    return torch.round(v / scale), scale


def _product64(v, packed, scales, k):
    q, scale = _quantized64(v)
    out = torch.empty((v.shape[0], packed.shape[0]), dtype=torch.float64, device=v.device)
    for start in range(0, packed.shape[0], 4096):
        rows = slice(start, start + 4096)
        out[:, rows] = q @ _weights64(packed[rows], scales[rows], k).t().contiguous()
    return out.mul_(scale)


def _rms64(v, weight):
    return (v * (v.square().mean(dim=-1, keepdim=True) + EPS).rsqrt()).clamp(-8.0, 8.0) * weight.double()


def _silu64(v):
    return v / (1.0 + torch.exp(-v))


def exact(case, seed):
    if case["kind"] == "linear":
        packed, scales, bias, x = _linear_inputs(case, seed)
        y = _product64(x.double(), packed, scales, case["k"])
        return y if bias is None else y + bias.double()
    if case["kind"] == "layer":
        weights, norms, residual, partials = _layer_inputs(case, seed)
        hidden, dense = case["hidden"], case["dense"]
        x = residual.double()
        mixer_in = _product64(_rms64(x, norms[0]), *weights["entry"], hidden)
        parts = partials.double()
        share = torch.exp(parts[..., 0] - parts[..., 0].amax(dim=-1, keepdim=True))
        merged = (share[..., None] * parts[..., 2:]).sum(-2) / (share * parts[..., 1]).sum(-1, keepdim=True)
        x = x + _product64(merged.reshape(x.shape), *weights["out"], hidden)
        normed = _rms64(x, norms[1])
        mid = _silu64(_product64(normed, *weights["gate"], hidden)) * _product64(normed, *weights["up"], hidden)
        x = x + _product64(mid, *weights["down"], dense)
        return {"mixer_in": mixer_in, "mid": mid, "residual": x}
    weights, ids = _stack_inputs(case, seed)
    first = _prompt64(case, weights, ids)
    if case["kind"] == "prefill":
        return first
    # the tokens after the first follow from choices between near values: they have no 64-bit answer
    return {"first": first, "tokens": None, "logits": None}


def _prompt64(case, weights, ids):
    def operand(layer):
        return torch.from_numpy(layer.packed).cuda(), torch.from_numpy(layer.scales).cuda(), layer.in_features

    def vector(values):
        return torch.from_numpy(values).cuda()

    hidden = case["hidden"]
    packed, scales, k = operand(weights.token)
    at = torch.tensor(ids, device="cuda")
    x = _weights64(packed[at], scales[at], k)
    for layer in weights.layers:
        mixed = _product64(_rms64(x, vector(layer.mixer_norm)), *operand(layer.qkv))[:, 2 * hidden:]
        x = x + _product64(mixed.contiguous(), *operand(layer.out))
        normed = _rms64(x, vector(layer.ffn_norm))
        mid = _silu64(_product64(normed, *operand(layer.gate))) * _product64(normed, *operand(layer.up))
        x = x + _product64(mid, *operand(layer.down))
    return _product64(_rms64(x[-1:], vector(weights.final_norm)), packed, scales, k)[0]
