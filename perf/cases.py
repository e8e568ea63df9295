"""The work a program built on this library has it do, as cases that can be timed and compared.

A case is a dict of plain values; its "family" says which pass it is:

    decode   one layer's MLP for a few tokens over GGUF weights (RMSNorm, three products, SwiGLU, residual), with
             the final norm and the vocabulary projection behind it where "vocab" is not 0
    prefill  the operators around the matrix products of a prompt: embedding Gather, RMSNorm, RoPE, SwiGLU, residual
    softmax  attention scores [heads, queries, keys] with or without a mask
    sample   from logits to tokens
    dequant  the weights of one MLP decoded from GGUF blocks to bf16, with their row sums of squares
    pool     LayerNorm, the mean over the tokens and the maximum of every row (an encoder's last step)
    layout   heads brought in front of the tokens, appended to a cache and widened

Every operator goes through `hyle_amd.torch_io.Bound`: prepared once, submitted on every pass.
"""
from __future__ import annotations

import math

import torch

from hyle_amd import compute as hc
from hyle_amd import torch_io as tio

DEVICE = "cuda:0"
TYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
HYLE = {"f32": hc.DataType.kFloat32, "bf16": hc.DataType.kBFloat16, "f16": hc.DataType.kFloat16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
GGUF = {"Q4_K": hc.GgufQuantizedType.kQ4K, "Q6_K": hc.GgufQuantizedType.kQ6K, "Q8_0": hc.GgufQuantizedType.kQ8_0}
# high bytes of a block's f16 scales, and the bits that leave its weights near 0.1
SCALE_BYTES = {"Q4_K": (1, 3), "Q6_K": (209,), "Q8_0": (1,)}
SCALE_RANGE = {"Q4_K": (0x08, 0x07), "Q6_K": (0x04, 0x03), "Q8_0": (0x10, 0x07)}
EMBEDDINGS = 151936  # rows of the embedding table


def listed():
    return [
        # one token through a layer, submitted operator by operator: what a chat with one user waits for
        {"name": "decode_one_token", "family": "decode", "tokens": 1, "hidden": 2048, "ffn": 6144, "up": "Q4_K", "down": "Q6_K",
         "vocab": 0, "head": "Q6_K", "dtype": "bf16", "replayed": False},
        # the same token with the vocabulary projection behind it, captured once and replayed: a serving loop
        {"name": "decode_token_to_logits_replayed", "family": "decode", "tokens": 1, "hidden": 2048, "ffn": 6144, "up": "Q4_K",
         "down": "Q4_K", "vocab": 151936, "head": "Q6_K", "dtype": "bf16", "replayed": True},
        # five streams at once through the widest layer the library's own tests use
        {"name": "decode_five_tokens_wide", "family": "decode", "tokens": 5, "hidden": 5120, "ffn": 17408, "up": "Q8_0",
         "down": "Q8_0", "vocab": 0, "head": "Q8_0", "dtype": "bf16", "replayed": False},
        # a long prompt at the benchmark's shapes
        {"name": "prefill_8192", "family": "prefill", "tokens": 8192, "hidden": 2048, "ffn": 6144, "heads": 16, "depth": 128,
         "rotary": 128, "half_split": True, "dtype": "bf16"},
        # a prompt of the length it happens to have, another model's sizes, another type, a partial rotation
        {"name": "prefill_ragged", "family": "prefill", "tokens": 1037, "hidden": 2560, "ffn": 9728, "heads": 20, "depth": 80,
         "rotary": 32, "half_split": True, "dtype": "f16"},
        # causal attention over 4096 positions: the largest tensor of the benchmark
        {"name": "softmax_causal", "family": "softmax", "heads": 32, "queries": 4096, "keys": 4096, "dtype": "f32", "mask": "boolean",
         "scale": 1.0},
        # the second chunk of a prompt: neither side a power of two, an additive mask
        {"name": "softmax_ragged", "family": "softmax", "heads": 24, "queries": 777, "keys": 1013, "dtype": "bf16", "mask": "additive",
         "scale": 0.088},
        # a batch whose rows are greedy or drawn: argmax and Categorical over all, then one pick per row
        {"name": "sample_batch", "family": "sample", "rows": 64, "vocab": 151936, "count": 0, "dtype": "f32"},
        # five rows drawn from their forty best
        {"name": "sample_top40", "family": "sample", "rows": 5, "vocab": 248320, "count": 40, "dtype": "bf16"},
        # the weights of one layer before a matrix product in bf16, a file of mixed formats
        {"name": "dequant_layer", "family": "dequant", "hidden": 2048, "ffn": 6144},
        # the last step of an encoder over a long document
        {"name": "pool_ragged", "family": "pool", "tokens": 5003, "hidden": 2560, "dtype": "f32"},
        # keys of a chunk to the cache's layout behind the 3072 positions it holds
        {"name": "layout_append", "family": "layout", "tokens": 1024, "cached": 3072, "heads": 16, "depth": 128, "dtype": "bf16"},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    family = rng.choice(["decode", "decode", "prefill", "prefill", "softmax", "softmax", "sample", "sample", "dequant", "pool", "layout"])
    dtype = rng.choice(["f32", "bf16", "f16"])
    if family == "decode":
        wide = rng.randint(4, 20)
        vocab = rng.choice([0, 0, _log(rng, 32000, 151936)]) if wide <= 12 else 0
        kinds = [rng.choice(["Q4_K", "Q6_K", "Q8_0"]) for _ in range(3)]
        return {"family": family, "tokens": rng.choice([1, 1, 2, 3, 4, 5, 6, 7, 8]), "hidden": 256 * wide,
                "ffn": 256 * _log(rng, 8, 68), "up": kinds[0], "down": kinds[1], "vocab": vocab, "head": kinds[2],
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "replayed": rng.random() < 0.5}
    if family == "prefill":
        depth = rng.choice([64, 80, 96, 128, 256])
        return {"family": family, "tokens": _log(rng, 1, 8192), "hidden": 64 * _log(rng, 8, 80), "ffn": 64 * _log(rng, 24, 200),
                "heads": rng.randint(4, 32), "depth": depth, "rotary": rng.choice([depth, depth, depth // 2]),
                "half_split": rng.random() < 0.75, "dtype": dtype}
    if family == "softmax":
        heads, keys = rng.randint(8, 64), _log(rng, 64, 8192)
        most = (1 << 29) * 9 // (10 * heads * keys)
        queries = max(1, min(_log(rng, 1, 4096), most))
        return {"family": family, "heads": heads, "queries": queries, "keys": keys, "dtype": dtype,
                "mask": rng.choice(["none", "boolean", "additive"]), "scale": rng.choice([1.0, 0.088])}
    if family == "sample":
        return {"family": family, "rows": _log(rng, 1, 64), "vocab": _log(rng, 32000, 248320),
                "count": rng.choice([0, 0, 20, 40, 64, 100]), "dtype": dtype}
    if family == "dequant":
        return {"family": family, "hidden": 256 * _log(rng, 2, 20), "ffn": 256 * _log(rng, 4, 68)}
    if family == "pool":
        return {"family": family, "tokens": _log(rng, 16, 8192), "hidden": 8 * _log(rng, 48, 640), "dtype": dtype}
    return {"family": family, "tokens": _log(rng, 1, 4096), "cached": _log(rng, 1, 8192), "heads": rng.randint(2, 32),
            "depth": rng.choice([64, 80, 96, 128, 256]), "dtype": dtype}


def _block(kind):
    return hc.GGUF_BLOCKS[GGUF[kind]]


def _weight_bytes(kind, k, n):
    per, size = _block(kind)
    return n * (k // per) * size


class _Make:
    """Inputs on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(seed)

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=TYPES[dtype], device=DEVICE).normal_(mean, std, generator=self.g)

    def whole(self, shape, low, high, dtype=torch.int32):
        return torch.randint(low, high, shape, dtype=dtype, device=DEVICE, generator=self.g)

    def weight(self, kind, k, n):
        """Rows of native blocks: random quants, block scales in a narrow band."""
        per, size = _block(kind)
        raw = torch.randint(0, 256, (n, k // per, size), dtype=torch.uint8, device=DEVICE, generator=self.g)
        low, keep = SCALE_RANGE[kind]
        for at in SCALE_BYTES[kind]:
            raw[:, :, at] &= keep
            raw[:, :, at] |= low
        return raw.view(n, -1)


class _Pass:
    """The operators of one pass in order, each bound to its inputs and outputs."""

    def __init__(self, context):
        self.context, self.steps, self.outputs, self.graph = context, [], [], None

    def add(self, operation, *inputs, descs=None):
        bound = tio.Bound(self.context, operation, descs or [tio.desc_of(t) for t in inputs])
        outputs = bound.outputs()
        self.steps.append((bound, list(inputs), outputs))
        return outputs[0] if len(outputs) == 1 else outputs

    def submit(self):
        for bound, inputs, outputs in self.steps:
            bound.submit(inputs, outputs)

    def capture(self):
        """The same launches as one HIP graph; the eager pass before it loads the kernels."""
        self.submit()
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.submit()


_CONTEXT = []


def _context():
    if not _CONTEXT:
        _CONTEXT.append(hc.Context.create(0))
    return _CONTEXT[0]


def prepare(case, seed):
    make, p = _Make(seed), _Pass(_context())
    family = case["family"]
    dtype = case.get("dtype", "bf16")
    if family == "decode":
        m, h, f = case["tokens"], case["hidden"], case["ffn"]

        def product(kind, k, n, x):
            return p.add(hc.GgufMatVec(hc.ActivationArithmetic.kGgmlQ8), make.weight(kind, k, n), x,
                         descs=[hc.TensorDesc.gguf_weight(GGUF[kind], HYLE[dtype], k, n), tio.desc_of(x)])

        x = make.normal((m, h), dtype)
        normed = p.add(hc.RmsNorm(1e-6), x, make.normal((h,), dtype, 0.1, 1.0))
        gate, up = product(case["up"], h, f, normed), product(case["up"], h, f, normed)
        act = p.add(hc.GatedActivation(hc.GatedActivationKind.kSilu, hc.GatedInputKind.kSeparate), gate, up)
        down = product(case["down"], f, h, act)
        y = p.add(hc.Binary(hc.BinaryKind.kAdd), x, down)
        p.outputs = [gate, up, act, down, y]
        if case["vocab"]:
            last = p.add(hc.RmsNorm(1e-6), y, make.normal((h,), dtype, 0.1, 1.0))
            p.outputs += [last, product(case["head"], h, case["vocab"], last)]
        if case["replayed"]:
            p.capture()
    elif family == "prefill":
        t, h, f = case["tokens"], case["hidden"], case["ffn"]
        ids = make.whole((t,), 0, EMBEDDINGS)
        rows = p.add(hc.Gather(0), make.normal((EMBEDDINGS, h), dtype), ids)
        normed = p.add(hc.RmsNorm(1e-6), rows, make.normal((h,), dtype, 0.1, 1.0))
        query = make.normal((1, t, case["heads"], case["depth"]), dtype)
        half = case["rotary"] // 2
        frequencies = (10000.0 ** (-torch.arange(half, dtype=torch.float64, device=DEVICE) / half)).to(torch.float32)
        layout = hc.RopeLayout.kHalfSplit if case["half_split"] else hc.RopeLayout.kInterleaved
        start = int(make.whole((1,), 0, 1024).item())
        turned = p.add(hc.RoPE(case["rotary"], 1, layout), query, torch.arange(start, start + t, dtype=torch.int32, device=DEVICE), frequencies)
        act = p.add(hc.GatedActivation(hc.GatedActivationKind.kSilu, hc.GatedInputKind.kSeparate), make.normal((t, f), dtype, 2.0),
                    make.normal((t, f), dtype, 2.0))
        p.outputs = [rows, normed, turned, act, p.add(hc.Binary(hc.BinaryKind.kAdd), rows, make.normal((t, h), dtype))]
    elif family == "softmax":
        h, q, k = case["heads"], case["queries"], case["keys"]
        scores = make.normal((h, q, k), dtype, 3.0 / case["scale"])
        kept = torch.ones((q, k), dtype=torch.bool, device=DEVICE).tril(max(0, k - q))
        inputs = [scores]
        if case["mask"] == "boolean":
            inputs.append(kept)
        elif case["mask"] == "additive":
            inputs.append(torch.zeros((q, k), dtype=TYPES[dtype], device=DEVICE).masked_fill_(~kept, float("-inf")))
        mask = {"none": hc.MaskKind.kNone, "boolean": hc.MaskKind.kBoolean, "additive": hc.MaskKind.kAdditive}[case["mask"]]
        p.outputs = [p.add(hc.Softmax(scale=case["scale"], mask=mask), *inputs)]
    elif family == "sample":
        rows, vocab = case["rows"], case["vocab"]
        logits = make.normal((rows, vocab), dtype, 4.0)
        identities = make.whole((rows, 4), -(1 << 31), 1 << 31).view(torch.uint32)
        if case["count"]:
            best, at = p.add(hc.TopK(count=case["count"]), logits)
            p.outputs = [best, at, p.add(hc.Categorical(), best, identities)]
        else:
            best, at = p.add(hc.TopK(), logits)
            drawn, score = p.add(hc.Categorical(True), logits, identities)
            flags = make.whole((rows,), 0, 2).to(torch.bool)
            p.outputs = [best, at, drawn, score, p.add(hc.Select(), flags, at.view(rows), drawn)]
    elif family == "dequant":
        h, f = case["hidden"], case["ffn"]
        p.outputs = []
        for kind, k, n in (("Q4_K", h, f), ("Q8_0", h, f), ("Q6_K", f, h)):
            p.outputs += p.add(hc.GgufDequantSumSquares(), make.weight(kind, k, n),
                               descs=[hc.TensorDesc.gguf_weight(GGUF[kind], hc.DataType.kBFloat16, k, n)])
    elif family == "pool":
        x = make.normal((case["tokens"], case["hidden"]), dtype)
        x *= torch.empty((case["tokens"], 1), dtype=TYPES[dtype], device=DEVICE).uniform_(0.1, 10.0, generator=make.g)
        normed = p.add(hc.LayerNorm(1e-5), x, make.normal((case["hidden"],), dtype, 0.1, 1.0), make.normal((case["hidden"],), dtype, 0.1))
        full = hc.DataType.kFloat32
        p.outputs = [normed, p.add(hc.Reduce(hc.ReductionKind.kMean, hc.Axes.from_([0]), accumulation_type=full), normed),
                     p.add(hc.Reduce(hc.ReductionKind.kMaximum, hc.Axes.from_([-1]), accumulation_type=full), normed)]
    else:
        t, c, h, d = case["tokens"], case["cached"], case["heads"], case["depth"]
        fresh = make.normal((t, h, d), dtype)
        moved = p.add(hc.Copy(), fresh.permute(1, 0, 2))
        joined = p.add(hc.Concat(1), make.normal((h, c, d), dtype), moved)
        p.outputs = [moved, joined, p.add(hc.Cast(hc.DataType.kFloat32 if dtype != "f32" else hc.DataType.kBFloat16), joined)]
    return p


def run(p):
    if p.graph is not None:
        p.graph.replay()
    else:
        p.submit()
    return p.outputs


def work(case):
    """Every operator's inputs once and its outputs once; the operators' results are results of the pass."""
    family, s = case["family"], SIZE[case.get("dtype", "bf16")]
    if family == "decode":
        m, h, f, v = case["tokens"], case["hidden"], case["ffn"], case["vocab"]
        weights = 2 * _weight_bytes(case["up"], h, f) + _weight_bytes(case["down"], f, h)
        values = 3 * h * f
        rows = s * m * ((2 * h) + 2 * (h + f) + 3 * f + (f + h) + 3 * h) + s * h
        if v:
            weights += _weight_bytes(case["head"], h, v)
            values += h * v
            rows += s * m * (2 * h + h + v) + s * h
        return {"bytes": weights + rows, "flops": 2 * m * values}
    if family == "prefill":
        t, h, f, q = case["tokens"], case["hidden"], case["ffn"], case["heads"] * case["depth"]
        return {"bytes": s * (t * (2 * h + 2 * h + 2 * q + 3 * f + 3 * h) + h) + 8 * t + 2 * case["rotary"],
                "flops": t * (4 * h + 3 * q + 5 * f + h)}
    if family == "softmax":
        n = case["heads"] * case["queries"] * case["keys"]
        mask = {"none": 0, "boolean": 1, "additive": s}[case["mask"]] * case["queries"] * case["keys"]
        return {"bytes": 2 * s * n + mask, "flops": 5 * n}
    if family == "sample":
        n, rows = case["rows"] * case["vocab"], case["rows"]
        if case["count"]:
            return {"bytes": s * n + rows * case["count"] * (2 * s + 4) + rows * 20, "flops": n}
        return {"bytes": 2 * s * n + rows * (s + 4 + 16 + 8 + 13), "flops": 4 * n}
    if family == "dequant":
        h, f = case["hidden"], case["ffn"]
        return {"bytes": _weight_bytes("Q4_K", h, f) + _weight_bytes("Q8_0", h, f) + _weight_bytes("Q6_K", f, h) + 6 * h * f + 4 * (2 * f + h),
                "flops": 3 * 4 * h * f}
    if family == "pool":
        t, h = case["tokens"], case["hidden"]
        return {"bytes": s * (4 * t * h + 3 * h + t), "flops": 9 * t * h}
    n, joined = case["tokens"] * case["heads"] * case["depth"], (case["tokens"] + case["cached"]) * case["heads"] * case["depth"]
    return {"bytes": s * (2 * n + 2 * joined + joined) + (4 if s == 2 else 2) * joined, "flops": joined}


def tolerance(case):
    """About four times what the operators differ from the same operators in 64 bits (rel: f32 6e-8 norms, 2.4e-7
    softmax, 4.2e-6 RoPE at positions above 1000; narrow types 1e-5 to 2e-4, where a value falls on the other side of a
    rounding), and in "max" two units in the last place."""
    family, dtype = case["family"], case.get("dtype", "bf16")
    unit = {"f32": 1e-5, "bf16": 1.6e-2, "f16": 2e-3}[dtype]
    if family == "layout":
        return "exact"
    if family == "dequant":  # the bf16 weights are exact, the sums are f32
        return {"rel": 2e-6}
    if family == "decode":  # 4.4e-4 with the norms in 64 bits: an 8-bit activation code changes by one here and there
        return {"rel": 2e-3, "max": 5e-2}
    if family == "prefill":
        return {"rel": {"f32": 2e-5, "bf16": 8e-4, "f16": 3e-4}[dtype], "max": max(unit, 1e-3)}
    if family == "sample":  # the scores are f32 logarithms; tokens and picked logits do not move
        return {"rel": 2e-6, "differ": 0.0}
    return {"rel": {"f32": 1e-6, "bf16": 1e-4, "f16": 4e-5}[dtype], "max": unit}
