"""The work that programs give this package, as cases that can be timed and
checked: the fused launches of a decoder layer, of attention blocks, of video
diffusion blocks, of an image encoder's block, and the decode of stored
weights for the matrix products. Everything goes through `HipOps`.

A case is a dict of plain values; `kind` names what it runs:

  layer            a dense decoder layer's launches between its matrix
                   products: embedding, RMSNorm, the per-head query/key norm
                   with RoPE and the paged cache write, the residual add with
                   its norm, SwiGLU
  attention        the same attention step as separate operations: RMSNorm of
                   every query and key head, RoPE, cache write
  gated_attention  attentionInputs: a gated query projection, partial rotary
                   with a position a section (text with images)
  dit_block        a diffusion block's stream: the latents' conversion, AdaLN,
                   the gated residual, AdaLN, GELU-tanh
  dit_attention    its queries and keys: full-width RMSNorm, then RoPE from
                   tables or 3-D RoPE on the grid
  dit_rows         the block of a model whose modulation differs by row:
                   modulateChunks, gatedAddChunk, the per-head gate
  encoder          an image encoder's block: LayerNorm with weight and bias,
                   RoPE over two axes, GELU
  weights          a layer's stored weights decoded for its matrix products
  rotated          the same for ConvRot's rotated weights
"""

import math

import numpy as np
import torch

from drift_amd import ops as d

TYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
PAGE = 16  # tokens a cache page


def listed():
    return [
        # one new token of a conversation: the smallest calls, all latency
        dict(name="decode_token", kind="layer", tokens=1, start=1027, hidden=4096, heads=32, kv_heads=8, dim=128,
             ffn=14336, vocabulary=151936, dtype="bf16"),
        # an ordinary prompt, in the F32 the runner's models hold
        dict(name="prompt_f32", kind="layer", tokens=509, start=0, hidden=2560, heads=32, kv_heads=8, dim=128,
             ffn=10240, vocabulary=151936, dtype="f32"),
        # a long prompt's chunk behind earlier ones
        dict(name="long_prompt", kind="layer", tokens=4093, start=77, hidden=4096, heads=32, kv_heads=8, dim=128,
             ffn=14336, vocabulary=151936, dtype="bf16"),
        # the dense decoder's attention step as the runner composes it
        dict(name="attention_steps", kind="attention", tokens=2039, start=5, heads=32, kv_heads=8, dim=128,
             rotary=128, sections="single", dtype="f32"),
        # a gated attention's inputs over a prompt with images: heads of 256,
        # 64 of their values turning, positions by section
        dict(name="gated_attention", kind="gated_attention", tokens=4096, start=30, heads=16, kv_heads=2, dim=256,
             rotary=64, sections="interleaved", dtype="bf16"),
        # a video block: two samples of 21 x 30 x 52 latents, the largest
        dict(name="dit_block", kind="dit_block", samples=2, tokens=32760, width=3072, dtype="bf16"),
        # a small video or an image, F32
        dict(name="dit_block_f32", kind="dit_block", samples=1, tokens=7800, width=3072, dtype="f32"),
        # queries and keys of a video block from the runner's angle tables
        dict(name="dit_attention", kind="dit_attention", frames=9, rows=30, cols=52, heads=24, dim=128,
             angles="table", dtype="bf16"),
        # image-to-video: every token has its own modulation
        dict(name="dit_rows", kind="dit_rows", tokens=14040, width=3072, chunks=6, heads=24, dtype="bf16"),
        # an image of 67 x 61 patches through an encoder's block
        dict(name="encoder", kind="encoder", rows=67, cols=61, heads=16, dim=72, ffn=4304, activation="GeluTanh",
             dtype="f32"),
        # a layer's gate and down weights as a 4-bit file stores them
        dict(name="weights", kind="weights", formats="Q4_K,Q6_K", rows=14336, width=4096, dtype="bf16"),
        # a rotated 8-bit linear of a diffusion model
        dict(name="rotated", kind="rotated", four_bit=False, group=0, rows=13824, width=5120),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "attention", "gated_attention", "dit_block", "dit_attention", "dit_rows",
                       "encoder", "weights", "rotated"])
    dtype = rng.choice(["bf16", "f32"])
    if kind == "layer":
        heads, kv = rng.choice([(32, 8), (16, 8), (16, 2), (28, 4), (40, 8)])
        hidden, ffn = rng.choice([(1024, 3072), (2048, 6144), (2560, 10240), (4096, 14336), (5120, 13824)])
        return dict(kind=kind, tokens=_log(rng, 1, 4096), start=_log(rng, 1, 4000) - 1, hidden=hidden, heads=heads,
                    kv_heads=kv, dim=rng.choice([64, 128, 128]), ffn=ffn, vocabulary=_log(rng, 30000, 151936),
                    dtype=dtype)
    if kind in ("attention", "gated_attention"):
        heads, kv, dim, rotary = rng.choice([(32, 8, 128, 128), (16, 2, 256, 64), (24, 4, 256, 64), (28, 4, 128, 128),
                                             (32, 2, 128, 64), (16, 4, 64, 64)])
        return dict(kind=kind, tokens=_log(rng, 1, 8192), start=_log(rng, 1, 4000) - 1, heads=heads, kv_heads=kv,
                    dim=dim, rotary=rotary, sections=rng.choice(["single", "contiguous", "interleaved"]),
                    dtype=dtype)
    if kind == "dit_block":
        return dict(kind=kind, samples=rng.choice([1, 1, 2, 3]), tokens=_log(rng, 64, 8190),
                    width=rng.choice([1536, 2048, 3072, 3840, 5120]), dtype=dtype)
    if kind == "dit_attention":
        return dict(kind=kind, frames=rng.choice([1, 3, 5, 9]), rows=rng.randint(8, 45), cols=rng.randint(8, 60),
                    heads=rng.choice([12, 24, 30, 40]), dim=128, angles=rng.choice(["table", "head_table", "grid"]),
                    dtype=dtype)
    if kind == "dit_rows":
        heads = rng.choice([12, 24, 32])
        return dict(kind=kind, tokens=_log(rng, 64, 8190), width=heads * 128, chunks=rng.choice([2, 6]), heads=heads,
                    dtype=dtype)
    if kind == "encoder":
        heads, dim, ffn = rng.choice([(16, 72, 4304), (16, 80, 5120), (12, 64, 3072), (16, 64, 4096)])
        return dict(kind=kind, rows=rng.randint(9, 96), cols=rng.randint(9, 96), heads=heads, dim=dim, ffn=ffn,
                    activation=rng.choice(["GeluTanh", "GeluErf", "Silu"]), dtype="f32")
    if kind == "weights":
        names = rng.sample(["Q8_0", "Q4_K", "Q5_K", "Q6_K", "Q4_0", "Q5_1", "IQ4_NL", "IQ4_XS", "Q4_0_ROCMFP4", "F16"],
                           rng.choice([1, 2]))
        return dict(kind=kind, formats=",".join(names), rows=_log(rng, 512, 14336) | 1,
                    width=256 * rng.choice([4, 10, 16, 19, 20]), dtype=rng.choice(["bf16", "f16"]))
    four_bit = rng.choice([False, True])
    return dict(kind=kind, four_bit=four_bit, group=rng.choice([64, 128]) if four_bit else 0,
                rows=_log(rng, 512, 13824) | 1, width=256 * rng.choice([6, 12, 16, 20]))


# ------------------------------------------------------------------ inputs

class _Inputs:
    """Tensors made on the GPU from a seed."""

    def __init__(self, case, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.type = TYPES[case.get("dtype", "bf16")]

    def normal(self, *shape, dtype=None, scale=1.0, mean=0.0):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        if scale != 1.0 or mean != 0.0:
            x.mul_(scale).add_(mean)
        return x.to(dtype or self.type)

    def vector(self, *shape, scale=0.1, mean=0.0):
        return self.normal(*shape, dtype=torch.float32, scale=scale, mean=mean)

    def bytes(self, *shape):
        n = math.prod(shape)
        words = torch.randint(-2 ** 63, 2 ** 63 - 1, ((n + 7) // 8,), generator=self.g, device="cuda")
        return words.view(torch.uint8)[:n].view(shape)

    def integers(self, low, high, *shape):
        return torch.randint(low, high, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def empty(self, *shape, dtype=None):
        return torch.empty(shape, dtype=dtype or self.type, device="cuda")


# where a block of each storage type holds its F16 scales
_HALVES = {"Q8_0": (0,), "Q4_K": (0, 2), "Q5_K": (0, 2), "Q6_K": (208,), "Q4_0": (0,), "Q5_1": (0, 2),
           "IQ4_NL": (0,), "IQ4_XS": (0,)}


def _stored(make, name, rows, cols):
    """A table of random blocks with scales of ordinary size."""
    t = d.STORAGE_TYPES[name]
    if name == "F16":
        data = make.normal(rows, cols, dtype=torch.float16).view(torch.uint8)
        return d.StoredTable(data, t, cols)
    blocks = make.bytes(rows, cols // t.values, t.bytes)
    for at in _HALVES.get(name, ()):
        scale = make.vector(rows, cols // t.values).abs_().mul_(0.05).add_(1e-3).to(torch.float16)
        blocks[..., at:at + 2] = scale.unsqueeze(-1).view(torch.uint8)
    if name == "Q4_0_ROCMFP4":  # two unsigned E4M3 scales a block
        blocks[..., 16:18] &= 0x3f
    return d.StoredTable(blocks.view(rows, -1), t, cols)


def _sections(case, pairs):
    a = 3 * pairs // 8
    return {"single": d.RopeSections.Single(), "contiguous": d.RopeSections.Contiguous(pairs - 2 * a, a, a),
            "interleaved": d.RopeSections.Interleaved(pairs - 2 * (pairs // 3), pairs // 3, pairs // 3)}[
                case["sections"]]


def _positions(case, sections):
    """Text positions, or with sections an image's (frame, row, column) from
    the first quarter of the prompt to its half, text around it."""
    n = case["tokens"]
    p = torch.arange(case["start"], case["start"] + n, dtype=torch.int32, device="cuda")
    if sections.positionsPerToken == 1:
        return p
    p = p.repeat(3, 1)
    a, b = n // 4, n // 2
    side = max(1, math.isqrt(max(0, b - a)))
    i = torch.arange(b - a, dtype=torch.int32, device="cuda")
    p[0, a:b] = case["start"] + a
    p[1, a:b] = case["start"] + a + i // side
    p[2, a:b] = case["start"] + a + i % side
    return p


def _cache(make, case):
    """A cache with the sequence's pages in no order among others."""
    used = -(-(case["start"] + case["tokens"]) // PAGE)
    cache = d.KvCache.allocate(used + 3, PAGE, case["kv_heads"], case["dim"])
    cache.keys.zero_()
    cache.values.zero_()
    order = torch.randperm(used + 3, generator=make.g, device="cuda")[:used].to(torch.int32)
    return cache, order


def prepare(case, seed):
    make, kind = _Inputs(case, seed), case["kind"]
    s = {"case": case, "hip": d.HipOps()}
    if kind == "layer":
        t, h, n, kv, dim = (case[k] for k in ("tokens", "hidden", "heads", "kv_heads", "dim"))
        s["table"] = _stored(make, "Q8_0", case["vocabulary"], h)
        s["ids"] = make.integers(0, case["vocabulary"], t)
        s["x"], s["y"] = make.empty(t, h), make.normal(t, h)
        s["w1"], s["w2"] = make.vector(h, mean=1.0), make.vector(h, mean=1.0)
        s["normed"] = make.empty(t, h)
        s["after"] = d.RowNorm(s["w2"], 1e-6, 0.0, make.empty(t, h))
        s["q"], s["k"], s["v"] = make.normal(t, n, dim), make.normal(t, kv, dim), make.normal(t, kv, dim)
        s["norms"] = d.QueryKeyNorms(make.vector(dim, mean=1.0), make.vector(dim, mean=1.0), 1e-6, 0.0,
                                     d.Rope(1e6, dim, d.RopeLayout.Neox))
        s["positions"] = _positions(case, s["norms"].rope.sections)
        s["cache"], s["pages"] = _cache(make, case)
        s["rq"] = make.empty(t, n, dim)
        s["gate"], s["up"], s["product"] = make.normal(t, case["ffn"]), make.normal(t, case["ffn"]), make.empty(t, case["ffn"])
    elif kind in ("attention", "gated_attention"):
        t, n, kv, dim = (case[k] for k in ("tokens", "heads", "kv_heads", "dim"))
        gated = kind == "gated_attention"
        s["q"] = make.normal(t, n, 2 * dim if gated else dim)
        s["k"], s["v"] = make.normal(t, kv, dim), make.normal(t, kv, dim)
        rope = d.Rope(1e6, case["rotary"], d.RopeLayout.Neox, _sections(case, case["rotary"] // 2))
        # the gated decoders store their norm weights less one
        s["norms"] = d.QueryKeyNorms(make.vector(dim, mean=0.0 if gated else 1.0),
                                     make.vector(dim, mean=0.0 if gated else 1.0), 1e-6, 1.0 if gated else 0.0, rope)
        s["positions"] = _positions(case, rope.sections)
        s["cache"], s["pages"] = _cache(make, case)
        s["rq"], s["rk"] = make.empty(t, n, dim), make.empty(t, kv, dim)
        if gated:
            s["queries"], s["gate"] = make.empty(t, n, dim), make.empty(t, n, dim)
    elif kind == "dit_block":
        rows, w = case["samples"] * case["tokens"], case["width"]
        # the latents arrive in the other float type
        s["latents"] = make.normal(rows, w, dtype=torch.float32 if make.type == torch.bfloat16 else torch.bfloat16)
        s["y"], s["f"] = make.normal(rows, w), make.normal(rows, w)
        s["x"], s["h1"], s["h2"], s["g"] = (make.empty(rows, w) for _ in range(4))
        s["table"] = [make.vector(case["samples"], w) for _ in range(4)]
        s["gates"] = make.vector(case["samples"], w, scale=0.5)
    elif kind == "dit_attention":
        t, n, dim = case["frames"] * case["rows"] * case["cols"], case["heads"], case["dim"]
        s["q"], s["k"] = make.normal(t, n * dim), make.normal(t, n * dim)
        s["qw"], s["kw"] = make.vector(n * dim, mean=1.0), make.vector(n * dim, mean=1.0)
        s["rq"], s["rk"] = make.empty(t, n * dim), make.empty(t, n * dim)
        if case["angles"] != "grid":
            angle = _grid_angles(case)
            if case["angles"] == "head_table":
                angle = angle[:, None, :].repeat(1, n, 1)
            s["cos"], s["sin"] = angle.cos().float().contiguous(), angle.sin().float().contiguous()
    elif kind == "dit_rows":
        t, w, n = case["tokens"], case["width"], case["heads"]
        s["x"], s["y"], s["z"] = (make.normal(t, w) for _ in range(3))
        s["table"] = make.vector(t, case["chunks"] * w)
        s["gates"] = make.vector(t * n, scale=0.5, mean=1.0)
        s["h"] = make.empty(t, w)
    elif kind == "encoder":
        t, n, dim = case["rows"] * case["cols"], case["heads"], case["dim"]
        s["x"], s["normed"] = make.normal(t, n * dim), make.empty(t, n * dim)
        s["w"], s["b"] = make.vector(n * dim, mean=1.0), make.vector(n * dim)
        s["q"], s["k"] = make.normal(t, n, dim), make.normal(t, n, dim)
        s["rope"] = d.Rope(1e4, dim, d.RopeLayout.Neox, d.RopeSections.Axes((dim // 4, dim // 4)))
        i = torch.arange(t, dtype=torch.int32, device="cuda")
        s["positions"] = torch.stack((i // case["cols"], i % case["cols"])).contiguous()
        s["rq"], s["rk"] = make.empty(t, n, dim), make.empty(t, n, dim)
        s["f"], s["g"] = make.normal(t, case["ffn"]), make.empty(t, case["ffn"])
    elif kind == "weights":
        s["tables"] = [_stored(make, name, case["rows"], case["width"]) for name in case["formats"].split(",")]
        s["out"] = [make.empty(case["rows"], case["width"]) for _ in s["tables"]]
    else:
        rows, w = case["rows"], case["width"]
        scales = make.vector(rows).abs_().mul_(0.05).add_(1e-4)
        levels = None
        if case["four_bit"]:
            relative = (make.bytes(rows, w // case["group"]) & 0x0f) + 0x30  # E4M3 from a half to two
            codebook = torch.linspace(-100, 115, 16, device="cuda") + make.vector(16)
            levels = d.ConvRotLevels(codebook, relative.contiguous(), case["group"])
        codes = make.bytes(rows, w // 2 if case["four_bit"] else w).view(torch.int8)
        s["weight"] = s["hip"].rotated(codes, d.ConvRotParts(scales, levels))
        s["out"] = make.empty(rows, w, dtype=torch.bfloat16)
    return s


# ------------------------------------------------------------------ a pass

def run(s):
    case, hip = s["case"], s["hip"]
    kind = case["kind"]
    if kind == "layer":
        hip.embedding(s["table"], s["ids"], s["x"])
        hip.rmsNorm(s["x"], s["w1"], 1e-6, 0.0, s["normed"])
        hip.queryKeyNormRopeCache(s["q"], s["k"], s["v"], s["norms"], s["positions"], s["cache"], s["pages"],
                                  case["start"], s["rq"])
        hip.addRmsNorm(s["x"], s["y"], s["after"])
        hip.gated(d.Activation.Silu, s["gate"], s["up"], s["product"])
        return {"x": s["x"], "normed": s["normed"], "queries": s["rq"], "keys": s["cache"].keys,
                "values": s["cache"].values, "after": s["after"].out, "product": s["product"]}
    if kind == "attention":
        n = s["norms"]
        hip.rmsNorm(s["q"], n.queryNorm, n.epsilon, n.weightOffset, s["rq"])
        hip.rmsNorm(s["k"], n.keyNorm, n.epsilon, n.weightOffset, s["rk"])
        hip.rope(s["rq"], s["positions"], n.rope, s["rq"])
        hip.rope(s["rk"], s["positions"], n.rope, s["rk"])
        hip.cacheWrite(s["rk"], s["v"], s["cache"], s["pages"], case["start"])
        return {"queries": s["rq"], "rotated": s["rk"], "keys": s["cache"].keys, "values": s["cache"].values}
    if kind == "gated_attention":
        hip.attentionInputs(s["q"], s["k"], s["v"], s["norms"], s["positions"], s["cache"], s["pages"], case["start"],
                            s["queries"], s["gate"], s["rk"], s["rq"])
        return {"queries": s["rq"], "gate": s["gate"], "keys": s["cache"].keys, "values": s["cache"].values}
    if kind == "dit_block":
        per = case["tokens"]
        shift1, scale1, shift2, scale2 = s["table"]
        hip.convert(s["latents"], s["x"])
        hip.layerNormModulate(s["x"], scale1, shift1, 1e-6, s["h1"], per)
        hip.gatedAdd(s["x"], s["y"], s["gates"], per)
        hip.layerNormModulate(s["x"], scale2, shift2, 1e-6, s["h2"], per)
        hip.activation(d.Activation.GeluTanh, s["f"], s["g"])
        return {"x": s["x"], "h1": s["h1"], "h2": s["h2"], "g": s["g"]}
    if kind == "dit_attention":
        shape = (-1, case["heads"], case["dim"])
        for x, w, out in ((s["q"], s["qw"], s["rq"]), (s["k"], s["kw"], s["rk"])):
            hip.rmsNorm(x, w, 1e-6, 0.0, out)
            heads = out.view(shape)
            if case["angles"] == "grid":
                hip.rope3d(heads, case["frames"], case["rows"], case["cols"], heads)
            else:
                hip.ropeTable(heads, s["cos"], s["sin"], heads)
        return {"queries": s["rq"], "keys": s["rk"]}
    if kind == "dit_rows":
        hip.modulateChunks(s["x"], s["table"], 0, 1, s["h"])
        hip.gatedAddChunk(s["h"], s["y"], s["table"], case["chunks"] - 1)
        heads = (-1, case["width"] // case["heads"])
        hip.rowGatedAdd(s["h"].view(heads), s["z"].view(heads), s["gates"])
        return {"h": s["h"]}
    if kind == "encoder":
        hip.layerNorm(s["x"], s["w"], s["b"], 1e-6, s["normed"])
        hip.rope(s["q"], s["positions"], s["rope"], s["rq"])
        hip.rope(s["k"], s["positions"], s["rope"], s["rk"])
        hip.activation(d.Activation[case["activation"]], s["f"], s["g"])
        return {"normed": s["normed"], "queries": s["rq"], "keys": s["rk"], "g": s["g"]}
    if kind == "weights":
        for table, out in zip(s["tables"], s["out"]):
            hip.dequantize(table, out)
        return s["out"]
    hip.dequantize(s["weight"], s["out"])
    return s["out"]


def work(case):
    """Bytes: each launch's inputs read once and its outputs written once.
    The arithmetic is a few vector operations a value and no product: 0."""
    kind, e = case["kind"], 4 if case.get("dtype") == "f32" else 2
    if kind == "layer":
        t, h = case["tokens"], case["hidden"]
        q, kv = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
        row = h // 32 * 34 + 4 + h * e  # the gather
        row += 2 * h * e  # the norm
        row += 2 * q * e + 2 * kv * e + 2 * kv * 2 + 4  # queries in and out, keys and values into the F16 cache
        row += 4 * h * e  # x, y in, x and its norm out
        row += 3 * case["ffn"] * e
        return {"bytes": t * row + 8 * h + 8 * case["dim"] + 4 * (case["start"] + t) // PAGE, "flops": 0}
    if kind in ("attention", "gated_attention"):
        t, q, kv = case["tokens"], case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
        if kind == "attention":
            row = 4 * (q + kv) * e + 2 * kv * e + 2 * kv * 2
        else:
            row = 4 * q * e + 2 * kv * e + 2 * kv * 2
        return {"bytes": t * (row + (4 if case["sections"] == "single" else 12)) + 8 * case["dim"], "flops": 0}
    if kind == "dit_block":
        n = case["samples"] * case["tokens"] * case["width"]
        return {"bytes": n * (6 + 4 * e + 3 * e + 2 * e) + 20 * case["samples"] * case["width"], "flops": 0}
    if kind == "dit_attention":
        t, w = case["frames"] * case["rows"] * case["cols"], case["heads"] * case["dim"]
        tables = {"grid": 0, "table": 8 * case["dim"] // 2, "head_table": 8 * w // 2}[case["angles"]]
        return {"bytes": 2 * (t * (4 * w * e + tables) + 4 * w), "flops": 0}
    if kind == "dit_rows":
        t, w = case["tokens"], case["width"]
        return {"bytes": t * w * (8 * e + 12) + 4 * t * case["heads"], "flops": 0}
    if kind == "encoder":
        t, w = case["rows"] * case["cols"], case["heads"] * case["dim"]
        return {"bytes": t * (6 * w + 2 * case["ffn"]) * e + 8 * w + 16 * t, "flops": 0}
    n = case["rows"] * case["width"]
    if kind == "weights":
        types = [d.STORAGE_TYPES[f] for f in case["formats"].split(",")]
        return {"bytes": sum(n // t.values * t.bytes + 2 * n for t in types), "flops": 0}
    codes = n // 2 + n // case["group"] if case["four_bit"] else n
    return {"bytes": codes + 2 * n + 4 * case["rows"], "flops": 0}


def tolerance(case):
    """Decodes are defined bit for bit. Elsewhere about four times what the
    outputs lie from their 64-bit values, which is their rounding: F32 sums
    and F32 exponentials, and half a BF16 or F16 step (a whole one where a
    result lies between two)."""
    if case["kind"] in ("weights", "rotated"):
        return "exact"
    if case["dtype"] == "bf16" or "kv_heads" in case:
        return {"rel": 8e-3, "max": 2e-2} if case["dtype"] == "bf16" else {"rel": 1e-3, "max": 2e-3}
    return {"rel": 1e-6, "max": 1e-5}


# ------------------------------------------------------------------ the same in 64 bits

def _grid_angles(case):
    """[tokens, dim / 2] angles in double: frame, row and column turn 22, 21
    and 21 of 64 pairs, each axis with its own frequencies."""
    side = 2 * (case["dim"] // 6)
    axes = ((case["dim"] - 2 * side) // 2, side // 2, side // 2)
    t = torch.arange(case["frames"] * case["rows"] * case["cols"], device="cuda")
    places = (t // (case["rows"] * case["cols"]), t // case["cols"] % case["rows"], t % case["cols"])
    return torch.cat([p.double()[:, None] / 1e4 ** (torch.arange(n, device="cuda").double() / n)
                      for p, n in zip(places, axes)], dim=1)


def _rms(x, w, offset=0.0):
    x = x.double()
    return x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * (w.double() + offset)


def _ln(x):
    x = x.double()
    return (x - x.mean(-1, keepdim=True)) / (x.var(-1, unbiased=False, keepdim=True) + 1e-6).sqrt()


def _angles(positions, rope):
    """[tokens, rotary / 2]: the angle is by definition the F32 product of
    the position and the F32 inverse frequency."""
    half, code, sizes = rope.rotaryDimensions // 2, rope.sections.code, rope.sections.sizes
    section, exponent = [], []
    for j in range(half):
        axis, e = 0, 2.0 * j / rope.rotaryDimensions
        if code == 1:
            axis = 0 if j < sizes[0] else 1 if j < sizes[0] + sizes[1] else 2
        elif code == 2:
            axis = 1 if j % 3 == 1 and j < 3 * sizes[1] else 2 if j % 3 == 2 and j < 3 * sizes[2] else 0
        elif code == 3:
            start = 0
            while j >= start + sizes[axis]:
                start += sizes[axis]
                axis += 1
            e = (j - start) / sizes[axis]
        section.append(axis)
        exponent.append(e)
    inverse = np.float32(1.0) / np.array([rope.theta ** e for e in exponent]).astype(np.float32)
    p = positions if positions.dim() == 2 else positions[None]
    by_pair = p[torch.tensor(section, device="cuda")].t().float()
    return (by_pair * torch.from_numpy(inverse).to("cuda")).double()


def _turn(x, rope, positions):
    """NeoX pairs of x [tokens, heads, dim] turned, the tail as it is."""
    a = _angles(positions, rope)[:, None, :]
    half = rope.rotaryDimensions // 2
    c, s = a.cos(), a.sin()
    lo, hi = x[..., :half], x[..., half:2 * half]
    return torch.cat((lo * c - hi * s, lo * s + hi * c, x[..., 2 * half:]), dim=-1)


def _cached(state, keys, values):
    """The zeroed cache with keys and values at the sequence's positions."""
    case, cache = state["case"], state["cache"]
    at = torch.arange(case["start"], case["start"] + case["tokens"], device="cuda")
    page, slot = state["pages"].long()[at // PAGE], at % PAGE
    ks = torch.zeros(cache.keys.shape, dtype=torch.float64, device="cuda")
    vs = torch.zeros(cache.values.shape, dtype=torch.float64, device="cuda")
    ks[page, slot] = keys
    vs[page, :, :, slot] = values.double()
    return ks, vs


def exact(case, seed):
    kind = case["kind"]
    if kind in ("weights", "rotated"):
        return None  # held bit for bit
    s = prepare(case, seed)
    if kind == "layer":
        raw = s["table"].data[s["ids"].long()].view(case["tokens"], -1, 34)
        scale = raw[..., :2].contiguous().view(torch.float16).double()
        x = (raw[..., 2:].contiguous().view(torch.int8).double() * scale).view(case["tokens"], -1)
        n = s["norms"]
        rq = _turn(_rms(s["q"], n.queryNorm), n.rope, s["positions"])
        keys, values = _cached(s, _turn(_rms(s["k"], n.keyNorm), n.rope, s["positions"]), s["v"])
        total = x + s["y"].double()
        gate = s["gate"].double()
        return {"x": total, "normed": _rms(x, s["w1"]), "queries": rq, "keys": keys, "values": values,
                "after": _rms(total, s["w2"]), "product": gate * gate.sigmoid() * s["up"].double()}
    if kind in ("attention", "gated_attention"):
        n, dim = s["norms"], case["dim"]
        rq = _turn(_rms(s["q"][..., :dim], n.queryNorm, n.weightOffset), n.rope, s["positions"])
        rk = _turn(_rms(s["k"], n.keyNorm, n.weightOffset), n.rope, s["positions"])
        keys, values = _cached(s, rk, s["v"])
        if kind == "attention":
            return {"queries": rq, "rotated": rk, "keys": keys, "values": values}
        return {"queries": rq, "gate": s["q"][..., dim:].double(), "keys": keys, "values": values}
    if kind == "dit_block":
        shape = (case["samples"], case["tokens"], case["width"])
        shift1, scale1, shift2, scale2 = (t.double()[:, None] for t in s["table"])
        x0 = s["latents"].double().view(shape)
        h1 = _ln(x0) * (1 + scale1) + shift1
        x1 = x0 + s["gates"].double()[:, None] * s["y"].double().view(shape)
        h2 = _ln(x1) * (1 + scale2) + shift2
        return {"x": x1.flatten(0, 1), "h1": h1.flatten(0, 1), "h2": h2.flatten(0, 1),
                "g": torch.nn.functional.gelu(s["f"].double(), approximate="tanh")}
    if kind == "dit_attention":
        if case["angles"] == "grid":
            angle = _grid_angles(case)
            c, sn = angle.cos()[:, None], angle.sin()[:, None]
        else:
            c, sn = s["cos"].double(), s["sin"].double()
            c, sn = (c, sn) if c.dim() == 3 else (c[:, None], sn[:, None])
        out = []
        for x, w in ((s["q"], s["qw"]), (s["k"], s["kw"])):
            v = _rms(x, w).view(x.shape[0], case["heads"], -1, 2)
            a, b = v[..., 0], v[..., 1]
            out.append(torch.stack((a * c - b * sn, a * sn + b * c), dim=-1).view(x.shape))
        return {"queries": out[0], "keys": out[1]}
    if kind == "dit_rows":
        table = s["table"].double().view(case["tokens"], case["chunks"], case["width"])
        h = s["x"].double() * (1 + table[:, 1]) + table[:, 0] + table[:, -1] * s["y"].double()
        gates = s["gates"].double().view(case["tokens"], -1).repeat_interleave(case["width"] // case["heads"], dim=1)
        return {"h": h + gates * s["z"].double()}
    f = s["f"].double()
    g = {"GeluTanh": lambda: torch.nn.functional.gelu(f, approximate="tanh"),
         "GeluErf": lambda: torch.nn.functional.gelu(f), "Silu": lambda: f * f.sigmoid()}[case["activation"]]()
    return {"normed": _ln(s["x"]) * s["w"].double() + s["b"].double(),
            "queries": _turn(s["q"].double(), s["rope"], s["positions"]),
            "keys": _turn(s["k"].double(), s["rope"], s["positions"]), "g": g}
