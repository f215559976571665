"""The work a program built on this framework gives it, as sized cases: what is timed, over which ranges, and how far
two correct implementations may differ.

Every case goes through the public entry points (`kq.*`, `kq.nn.*`).  The kinds:

  linear      one KQuantLinear call (a projection of a decode step, or of a prompt)
  layer       the seven projections of a dense transformer block, q / k / v / o / gate / up / down
  vocab       a tied embedding table: rows of the step's tokens looked up, then the logits over the vocabulary
  moe         router top-k, fused gate / up expert product, down product with the routing mix; a shared expert or none
  moe_bias    the block-scaled fp4 expert stacks with biases and the clamped SwiGLU
  lora        forward and activation gradient of a frozen quantized layer (an adapter trains upstream of it)
  mla         per-head absorbed projections, both orientations
  requantize  whole matrices decoded from one wire format and encoded into another

Sizes are those of the repository's benchmark and tests (4096 / 14336 / 128256, 8192 / 28672, 128 experts of
2048 <-> 768, 32 experts of 2880, 128 heads of 128 <-> 512) and generic ones between and beside them.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mlx-kquant_amd"))
import kq  # noqa: E402
import kq.nn  # noqa: E402
from kq.codec_geometry import CODEC_GEOMETRY, bytes_per_row  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
# codecs with an encoder that runs on the GPU; the others get structurally valid random wire
ENCODED = ("q8_0", "q4_0", "q4_1", "q5_0", "q5_1", "q2_k", "q3_k", "q4_k", "q5_k", "q6_k")
# (most matrices, the sensitive ones) of the mixes that quantized checkpoints come in
RECIPES = (("q4_k", "q6_k"), ("q5_k", "q6_k"), ("q3_k", "q4_k"), ("q8_0", "q8_0"), ("iq4_xs", "q6_k"),
           ("iq3_s", "iq4_xs"), ("iq2_xxs", "q2_k"), ("q4_0", "q4_0"), ("mxfp4", "q8_0"))
# 2 M N K of the largest call: the bound that drawn cases keep well below
LARGEST_FLOPS = 2.0 * 2048 * 28672 * 8192


def listed():
    return [
        # the smallest call: one square projection, one token, f16
        {"name": "linear_m1", "kind": "linear", "codec": "q4_k", "M": 1, "N": 4096, "K": 4096, "dtype": "f16"},
        # single-user decoding: the projections of one block (4-bit / 6-bit mix), one token
        {"name": "layer_m1", "kind": "layer", "codec": "q4_k", "codec2": "q6_k", "M": 1, "hidden": 4096, "kv": 1024,
         "ffn": 14336, "dtype": "bf16"},
        # batched serving: the same block, 32 sequences decoding together
        {"name": "layer_m32", "kind": "layer", "codec": "q4_k", "codec2": "q6_k", "M": 32, "hidden": 4096, "kv": 1024,
         "ffn": 14336, "dtype": "bf16"},
        # an ordinary prompt of ragged length on another mix
        {"name": "layer_m333", "kind": "layer", "codec": "iq4_xs", "codec2": "q6_k", "M": 333, "hidden": 4096,
         "kv": 1024, "ffn": 14336, "dtype": "bf16"},
        # the largest call: a long prompt on the widest matrix
        {"name": "linear_m2048", "kind": "linear", "codec": "q5_k", "M": 2048, "N": 28672, "K": 8192, "dtype": "bf16"},
        # first and last step of a decode iteration with a tied table, four sequences
        {"name": "vocab_m4", "kind": "vocab", "codec": "q6_k", "M": 4, "vocab": 128256, "hidden": 4096, "dtype": "bf16"},
        # mixture of experts, single-user decoding
        {"name": "moe_t1", "kind": "moe", "codec": "q4_k", "codec2": "q6_k", "T": 1, "E": 128, "R": 8, "hidden": 2048,
         "ffn": 768, "shared": False, "dtype": "bf16"},
        # the same stacks, a prompt of ragged length
        {"name": "moe_t1000", "kind": "moe", "codec": "q4_k", "codec2": "q6_k", "T": 1000, "E": 128, "R": 8,
         "hidden": 2048, "ffn": 768, "shared": False, "dtype": "bf16"},
        # fp4 expert stacks with biases, a batch of sequences decoding (or a short prompt)
        {"name": "moe_bias_t64", "kind": "moe_bias", "T": 64, "E": 32, "R": 4, "hidden": 2880, "ffn": 2880,
         "dtype": "bf16"},
        # fine-tuning above a frozen base: forward and backward of one projection
        {"name": "lora_m1024", "kind": "lora", "codec": "q4_k", "M": 1024, "N": 4096, "K": 4096, "dtype": "bf16"},
        # absorbed attention projections of four decoding sequences
        {"name": "mla_b4", "kind": "mla", "codec": "q8_0", "heads": 128, "B": 4, "L": 1, "dim": 128, "rank": 512,
         "dtype": "bf16"},
        # conversion of a checkpoint's matrix from one wire format to another
        {"name": "requantize", "kind": "requantize", "codec": "q8_0", "codec2": "q4_k", "N": 4096, "K": 4096,
         "imatrix": False, "dtype": "f32"},
    ]


# ------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, step):
    """Whole number of `step`s between lo and hi, spread over the logarithm."""
    return max(step, int(round(_log(rng, lo, hi) / step)) * step)


def _count(rng, lo, hi):
    return max(lo, min(hi, int(round(_log(rng, lo, hi)))))


def _outer(rng, lo, hi):
    """An output width: mostly a multiple of 64, sometimes whatever a vocabulary or a pruned layer leaves."""
    n = _size(rng, lo, hi, 64)
    return n if rng.random() < 0.7 else n - rng.randrange(1, 64)


def _inner(rng, codec, lo, hi):
    """A quantized row length: a multiple of 256, or for codecs of small blocks sometimes only of their block."""
    wpb = CODEC_GEOMETRY[codec][3]
    return _size(rng, lo, hi, wpb if wpb < 256 and rng.random() < 0.4 else 256)


def draw(rng):
    kind = rng.choice(("linear", "layer", "vocab", "moe", "moe_bias", "lora", "mla", "requantize"))
    dtype = rng.choice(("bf16", "bf16", "f16"))
    if kind == "linear":
        codec = rng.choice(sorted(CODEC_GEOMETRY))
        K, N = _inner(rng, codec, 1024, 14336), _outer(rng, 1024, 28672)
        M = _count(rng, 1, max(1, min(2048, int(0.2 * LARGEST_FLOPS / (2 * N * K)))))
        return {"kind": kind, "codec": codec, "M": M, "N": N, "K": K, "dtype": dtype}
    if kind == "layer":
        codec, codec2 = rng.choice(RECIPES)
        hidden = _size(rng, 1024, 8192, 256)
        ffn, kv = _size(rng, 2 * hidden, 4 * hidden, 256), hidden // rng.choice((1, 4, 8))
        weights = hidden * (2 * hidden + 2 * kv + 3 * ffn)
        M = _count(rng, 1, max(1, min(1024, int(0.2 * LARGEST_FLOPS / (2 * weights)))))
        return {"kind": kind, "codec": codec, "codec2": codec2, "M": M, "hidden": hidden, "kv": kv, "ffn": ffn,
                "dtype": dtype}
    if kind == "vocab":
        return {"kind": kind, "codec": rng.choice(("q6_k", "q8_0", "q4_k", "q5_k", "iq4_xs")), "M": _count(rng, 1, 16),
                "vocab": _outer(rng, 32000, 128256), "hidden": _size(rng, 1024, 4096, 256), "dtype": dtype}
    if kind == "moe":
        codec, codec2 = rng.choice(RECIPES)
        E, hidden, ffn = rng.choice((8, 32, 64, 128)), _size(rng, 1024, 4096, 256), _size(rng, 512, 4096, 256)
        while E * hidden * ffn > 128 * 2048 * 1024:
            hidden, ffn = max(1024, hidden - 256), max(512, ffn - 256)
        R = rng.randrange(1, 9)
        T = _count(rng, 1, max(1, min(1024, int(0.1 * LARGEST_FLOPS / (6 * R * hidden * ffn)))))
        return {"kind": kind, "codec": codec, "codec2": codec2, "T": T, "E": E, "R": min(R, E // 2), "hidden": hidden,
                "ffn": ffn, "shared": rng.random() < 0.3, "dtype": dtype}
    if kind == "moe_bias":
        E = rng.choice((8, 16, 32))
        return {"kind": kind, "T": _count(rng, 1, 256), "E": E, "R": rng.randrange(1, 5),
                "hidden": _size(rng, 1024, 3072, 32), "ffn": _size(rng, 1024, 3072, 32), "dtype": dtype}
    if kind == "lora":
        codec = rng.choice(("q4_k", "q5_k", "q6_k", "q8_0", "iq4_xs", "mxfp4", "q3_k", "q4_0"))
        K, N = _size(rng, 1024, 8192, 256), _size(rng, 1024, 8192, 64)
        M = _count(rng, 32, min(2048, int(0.07 * LARGEST_FLOPS / (2 * N * K))))
        return {"kind": kind, "codec": codec, "M": M, "N": N, "K": K, "dtype": dtype}
    if kind == "mla":
        return {"kind": kind, "codec": rng.choice(("q8_0", "q4_k", "q6_k", "q5_k", "iq4_xs")),
                "heads": rng.choice((16, 32, 64, 128)), "B": _count(rng, 1, 8), "L": _count(rng, 1, 32),
                "dim": rng.choice((64, 128, 192)), "rank": rng.choice((256, 512)), "dtype": dtype}
    codec2 = rng.choice(ENCODED)
    K = _size(rng, 1024, 8192, 256)
    return {"kind": "requantize", "codec": rng.choice(("q8_0", "q6_k", "q5_k", "iq4_xs", "mxfp4")), "codec2": codec2,
            "N": _count(rng, 128, (4096 * 4096) // K), "K": K,
            "imatrix": codec2 in kq.codec_geometry.IMATRIX_CODECS and rng.random() < 0.5,
            "dtype": rng.choice(("f32", "f16", "bf16"))}


# ------------------------------------------------------------------ inputs
class _Maker:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(shape, device="cuda", generator=self.gen) * scale).to(dtype)

    def ints(self, hi, *shape, lo=0):
        return torch.randint(lo, hi, shape, device="cuda", generator=self.gen)

    def wire(self, codec, rows, K):
        """Wire bytes of a [rows, K] matrix of N(0, 0.02) weights; at most 128 Mi of them are distinct, the
        rest repeats."""
        distinct = min(rows, max(64, (128 << 20) // K))
        if codec in ENCODED:
            w = self.normal(distinct, K, scale=0.02)
            wire = kq.quantize(w, codec, torch.ones(K, device="cuda") if codec in kq.codec_geometry.IMATRIX_CODECS else None)[0]
        else:
            wire = self._random_wire(codec, distinct, K)
        if distinct < rows:
            wire = wire.repeat(-(-rows // distinct), 1)[:rows].contiguous()
        return wire

    def _random_wire(self, codec, rows, K):
        """Random code bytes under block scales that give weights of about 0.02."""
        _, _, bpb, wpb = CODEC_GEOMETRY[codec]
        n = rows * (K // wpb)
        b = self.ints(256, n, bpb).to(torch.uint8)
        # a typical |weight| over the block's scale field
        unit = {"iq4_xs": 900.0, "iq4_nl": 60.0, "iq3_s": 110.0, "iq3_xxs": 110.0, "iq2_xxs": 90.0, "iq2_xs": 90.0,
                "iq2_s": 90.0, "iq1_s": 6.0, "iq1_m": 6.0}.get(codec, 1.0)
        if codec == "mxfp4":
            b[:, 0] = self.ints(122, n, lo=119).to(torch.uint8)
        elif codec == "nvfp4":
            b[:, 0:4] = self.ints(0x18, n, 4, lo=0x08).to(torch.uint8)
        else:
            d = (torch.rand(n, device="cuda", generator=self.gen) * 0.5 + 0.75) * (0.02 / unit)
            half = d.to(torch.float16).view(torch.uint8).reshape(n, 2)
            if codec == "iq1_m":  # the scale's four nibbles ride in the high nibbles of bytes 49, 51, 53, 55
                for i in range(4):
                    nib = (half[:, i // 2] >> (4 * (i % 2))) & 15
                    b[:, 49 + 2 * i] = (b[:, 49 + 2 * i] & 15) | (nib << 4)
            else:
                b[:, 0:2] = half
        return b.reshape(rows, K // wpb * bpb)

    def linear(self, codec, N, K):
        return kq.nn.KQuantLinear(K, N, False, codec, device="cuda").load_wire(self.wire(codec, N, K))


def prepare(case, seed):
    mk, dt, kind = _Maker(seed), DTYPES[case["dtype"]], case["kind"]
    s = {"kind": kind, "case": case}
    if kind in ("linear", "lora"):
        s["lin"] = mk.linear(case["codec"], case["N"], case["K"])
        s["x"] = mk.normal(case["M"], case["K"], dtype=dt)
        if kind == "lora":
            s["x"].requires_grad_(True)
            s["dy"] = mk.normal(case["M"], case["N"], scale=0.1, dtype=dt)
    elif kind == "layer":
        h, kv, f, c, c2 = case["hidden"], case["kv"], case["ffn"], case["codec"], case["codec2"]
        plan = (("q", c, h, h), ("k", c, kv, h), ("v", c2, kv, h), ("o", c, h, h), ("gate", c, f, h), ("up", c, f, h),
                ("down", c2, h, f))
        s["layers"] = {name: mk.linear(codec, n, k) for name, codec, n, k in plan}
        x = {"attn": mk.normal(case["M"], h, dtype=dt), "mixed": mk.normal(case["M"], h, scale=0.3, dtype=dt),
             "mlp": mk.normal(case["M"], h, dtype=dt), "act": mk.normal(case["M"], f, scale=0.3, dtype=dt)}
        s["x"] = {"q": x["attn"], "k": x["attn"], "v": x["attn"], "o": x["mixed"], "gate": x["mlp"], "up": x["mlp"],
                  "down": x["act"]}
    elif kind == "vocab":
        emb = kq.nn.KQuantEmbedding(case["vocab"], case["hidden"], case["codec"], out_dtype=dt, device="cuda")
        s["emb"] = emb.load_wire(mk.wire(case["codec"], case["vocab"], case["hidden"]))
        s["tokens"] = mk.ints(case["vocab"], case["M"])
        s["h"] = mk.normal(case["M"], case["hidden"], dtype=dt)
    elif kind == "moe":
        E, h, f, c, c2 = case["E"], case["hidden"], case["ffn"], case["codec"], case["codec2"]
        for name, codec, n, k in (("gate", c, f, h), ("up", c, f, h), ("down", c2, h, f)):
            s[name] = mk.wire(codec, E * n, k).reshape(E, n, bytes_per_row(codec, k))
            if case["shared"]:
                s["shared_" + name] = mk.wire(codec, n, k)
        s["x"] = mk.normal(case["T"], h, scale=0.5, dtype=dt)
        s["logits"] = mk.normal(case["T"], E + int(case["shared"]))
    elif kind == "moe_bias":
        E, h, f = case["E"], case["hidden"], case["ffn"]
        for name, n, k in (("gate", f, h), ("up", f, h), ("down", h, f)):
            s[name] = mk.wire("mxfp4", E * n, k).reshape(E, n, bytes_per_row("mxfp4", k))
            s[name + "_bias"] = mk.normal(E, n, scale=0.01)
        s["x"] = mk.normal(case["T"], h, scale=0.5, dtype=dt)
        s["idx"] = mk.normal(case["T"], E).topk(case["R"], dim=-1).indices.to(torch.int32)
    elif kind == "mla":
        nh, d, r, c = case["heads"], case["dim"], case["rank"], case["codec"]
        for name in ("embed", "unembed"):
            s[name] = kq.nn.KQuantMultiLinear(r, d, nh, c, device="cuda").load_wire(
                mk.wire(c, nh * d, r).reshape(nh, d, bytes_per_row(c, r)))
        s["q"] = mk.normal(case["B"], nh, case["L"], d, dtype=dt)
        s["latent"] = mk.normal(case["B"], nh, case["L"], r, scale=0.3, dtype=dt)
    else:
        s["wire"] = mk.wire(case["codec"], case["N"], case["K"])
        s["imatrix"] = mk.normal(case["K"]).square() + 0.05 if case["imatrix"] else None
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "linear":
        return s["lin"](s["x"])
    if kind == "lora":
        y = s["lin"](s["x"])
        return y.detach(), torch.autograd.grad(y, s["x"], s["dy"])[0]
    if kind == "layer":
        x = s["x"]
        return {name: lin(x[name]) for name, lin in s["layers"].items()}
    if kind == "vocab":
        return s["emb"](s["tokens"]), s["emb"].as_linear(s["h"])
    if kind == "moe":
        c, c2 = case["codec"], case["codec2"]
        idx, scores = kq.moe_router_topk(s["logits"], case["R"], True, shared_gate=case["shared"])
        if case["shared"]:
            h = kq.moe_glu_gather_shexp_kq(s["x"], s["gate"], s["up"], s["shared_gate"], s["shared_up"], c, idx)
            return kq.gather_qmv_mix_kq(h, s["down"], s["shared_down"], c2, idx, scores)
        h = kq.moe_glu_gather_kq(s["x"], s["gate"], s["up"], c, idx)
        return kq.gather_qmv_mix_ns_kq(h, s["down"], c2, idx, scores)
    if kind == "moe_bias":
        h = kq.moe_glu_gather_kq(s["x"], s["gate"], s["up"], "mxfp4", s["idx"], act="swiglu_clamp", limit=7.0,
                                 gate_bias=s["gate_bias"], up_bias=s["up_bias"], alpha=1.702)
        return kq.gather_qmv_kq(h, s["down"], "mxfp4", s["idx"], bias=s["down_bias"])
    if kind == "mla":
        return s["embed"](s["q"], transpose=False), s["unembed"](s["latent"])
    w = kq.dequantize(s["wire"], None, case["codec"], dtype=DTYPES[case["dtype"]])
    return w, kq.quantize(w, case["codec2"], s["imatrix"])[0]


# ------------------------------------------------------------------ what a pass cannot do without
def _touched(pairs, experts):
    """Distinct experts that uniformly routed pairs hit, on average."""
    return experts * (1.0 - (1.0 - 1.0 / experts) ** pairs)


def work(case):
    kind, c = case["kind"], case.get("codec")
    half = 2  # bytes of an activation
    if kind in ("linear", "lora"):
        M, N, K = case["M"], case["N"], case["K"]
        n = 2 if kind == "lora" else 1
        return {"bytes": N * bytes_per_row(c, K) + n * half * M * (N + K), "flops": n * 2.0 * M * N * K}
    if kind == "layer":
        M, h, kv, f, c2 = case["M"], case["hidden"], case["kv"], case["ffn"], case["codec2"]
        wire = (2 * h + kv + 2 * f) * bytes_per_row(c, h) + kv * bytes_per_row(c2, h) + h * bytes_per_row(c2, f)
        return {"bytes": wire + half * M * ((3 * h + f) + (3 * h + 2 * kv + 2 * f)),
                "flops": 2.0 * M * h * (2 * h + 2 * kv + 3 * f)}
    if kind == "vocab":
        M, v, h = case["M"], case["vocab"], case["hidden"]
        return {"bytes": (v + M) * bytes_per_row(c, h) + M * (8 + half * (2 * h + v)), "flops": 2.0 * M * v * h}
    if kind in ("moe", "moe_bias"):
        T, R, E, h, f = case["T"], case["R"], case["E"], case["hidden"], case["ffn"]
        c1, c2 = (c, case["codec2"]) if kind == "moe" else ("mxfp4", "mxfp4")
        one = 2 * f * bytes_per_row(c1, h) + h * bytes_per_row(c2, f) + (4 * (2 * f + h) if kind == "moe_bias" else 0)
        shared = int(case.get("shared", False))
        # the expert activations between the two products are written and read; each token's result written once
        io = half * T * h + 2 * half * T * (R + shared) * f + half * T * h * (R if kind == "moe_bias" else 1)
        router = 4 * T * (E + shared) if kind == "moe" else 4 * T * R
        return {"bytes": (_touched(T * R, E) + shared) * one + io + router, "flops": 6.0 * T * (R + shared) * h * f}
    if kind == "mla":
        nh, B, L, d, r = case["heads"], case["B"], case["L"], case["dim"], case["rank"]
        return {"bytes": 2 * nh * d * bytes_per_row(c, r) + 2 * half * B * nh * L * (d + r),
                "flops": 4.0 * B * nh * L * d * r}
    N, K = case["N"], case["K"]
    size = 4 if case["dtype"] == "f32" else 2
    # the decoded matrix is a result of its own and the encoder's input: written once, read once
    return {"bytes": N * (bytes_per_row(c, K) + bytes_per_row(case["codec2"], K)) + 2 * N * K * size, "flops": 0.0}


def tolerance(case):
    """Encoders and decoders are exact.  The products sum in f32 and round once to the activation type: against the
    same product in 64 bits that is 1.66e-3 for bf16 and 2.1e-4 for f16 over every kind and codec, 2.35e-3 and 3.0e-4
    where a rounded product feeds a second one (measured); four times that is stated."""
    if case["kind"] == "requantize":
        return "exact"
    two = case["kind"] in ("moe", "moe_bias")
    if case["dtype"] == "bf16":
        return {"rel": 9e-3 if two else 6.6e-3}
    return {"rel": 1.2e-3 if two else 8.4e-4}
