"""Performance cases of the SageAttention forward path: what they are, their inputs, one pass, its work and tolerance.

Every case is a call (or the documented pair of calls) of the package's public entry points on tensors that are already
on the GPU, the way a model's attention layer makes it.  ``kind`` names the entry points:

  "fixed"   sageattn on [B, H, L, D] or [B, L, H, D]: K mean, quantisers, V panels and attention in one call
  "packed"  sageattn_varlen on packed sequences of different lengths
  "steps"   k_mean, per_block_int8 and forward, called one after the other
"""
import math
import random

import torch

import baselinebenchmark_amd as sa

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}

# A plain call: what the other cases and the drawn ones change.
_BASE = dict(kind="fixed", B=1, Hq=8, Hkv=8, Sq=1024, Skv=1024, D=128, dtype="bfloat16", layout="HND", causal=False, pv="fp16",
             BLKQ=128, BLKK=64, k_interleave=1, q_interleave=1, smooth=True, lse=False, mask="", k_offset=2.0, outliers=0.0)
_PACKED = dict(kind="packed", nseq=16, lo=512, hi=32768, len_seed=2026, Hq=32, Hkv=8, D=128, dtype="bfloat16", causal=True, pv="fp16",
               BLKQ=128, BLKK=64, smooth=True, lse=False, k_offset=0.0)


def _fixed(name, **kw):
    return dict(_BASE, name=name, **kw)


def listed():
    return [
        # The smallest ordinary call: one image's worth of tokens over eight heads; latency and launches decide.
        _fixed("small_d64", D=64, dtype="float16", BLKK=128, k_offset=0.0),
        # One step of token generation: a single query row per head over a long history, four query heads per KV head.
        _fixed("decode_gqa", B=4, Hq=32, Hkv=8, Sq=1, Skv=8192),
        # Cross-attention of an image or video transformer: many query rows over the few hundred tokens of a prompt.
        _fixed("cross_short_kv", B=2, Hq=24, Hkv=24, Sq=4095, Skv=257, D=64, dtype="float16", layout="NHD"),
        # Self-attention under an explicit mask: documents packed into fixed-length rows, a boolean mask shared by the heads.
        _fixed("masked_documents", B=2, Hq=16, Hkv=16, Sq=1500, Skv=1500, D=64, dtype="float16", mask="documents"),
        # Attention whose partial results are merged later (sequence parallelism): the log-sum-exp comes back too.
        _fixed("lse_4k", B=1, Hq=32, Hkv=32, Sq=4096, Skv=4096, lse=True),
        # Prefill of a serving batch: many short prompts of very different lengths, grouped-query heads.
        dict(_PACKED, name="packed_prompts", nseq=96, lo=16, hi=1024, len_seed=7),
        # Quantise, then attend: the two calls of a program that handles the INT8 operands itself.
        _fixed("two_step_8k_d64", kind="steps", B=1, Hq=32, Hkv=32, Sq=8192, Skv=8192, D=64),
        # The fine-grained recipe: K scales for every 16 keys, V in FP8, causal.
        _fixed("recipe_128_16", B=2, Hq=16, Hkv=16, Sq=4096, Skv=4096, layout="NHD", causal=True, pv="fp8", BLKK=16),
        # Prefill of a batch of 4k prompts, FP16 P.V.
        _fixed("prefill_4k", B=4, Hq=32, Hkv=32, Sq=4096, Skv=4096, causal=True),
        # Long causal prefill, FP8 P.V: the benchmark's own workload.
        _fixed("prefill_16k_fp8", B=2, Hq=32, Hkv=32, Sq=16384, Skv=16384, causal=True, pv="fp8", BLKQ=64, BLKK=128),
        # Full attention over a video's tokens, a length that no tile divides, channels with outliers.
        _fixed("video_32760_fp8", B=1, Hq=24, Hkv=24, Sq=32760, Skv=32760, layout="NHD", pv="fp8", k_offset=0.0, outliers=0.01),
        # Long prompts of different lengths packed together, grouped-query heads, FP8 P.V: the largest call.
        dict(_PACKED, name="packed_long_gqa", pv="fp8"),
    ]


# ------------------------------------------------------------------------------------------------
# drawn cases
# ------------------------------------------------------------------------------------------------
def _log_int(rng, lo, hi):
    """An integer between lo and hi, uniform in its logarithm; odd and ragged values as they come, sometimes a round one."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.3 and n >= 64:
        n = n // 64 * 64
    return max(lo, min(hi, n))


def _heads(rng):
    hkv = rng.choice([2, 4, 8, 12, 16, 24, 32])
    return (hkv * 4, hkv) if hkv <= 8 and rng.random() < 0.5 else (hkv, hkv)


def draw(rng: random.Random):
    what = rng.choice(["self", "self", "self", "self", "decode", "cross", "mask", "lse", "steps", "packed", "packed", "recipe"])
    Hq, Hkv = _heads(rng)
    D = rng.choice([64, 128])
    dtype = rng.choice(["float16", "bfloat16"])
    pv = rng.choice(["fp16", "fp8"])
    BLKQ, BLKK = rng.choice([(128, 64), (128, 64), (64, 128), (128, 128), (32, 64)])
    common = dict(Hq=Hq, Hkv=Hkv, D=D, dtype=dtype, pv=pv, BLKQ=BLKQ, BLKK=BLKK)
    layout = rng.choice(["HND", "NHD"])
    if what == "packed":
        lo = _log_int(rng, 8, 512)
        hi = _log_int(rng, 2 * lo, 16384)
        nseq = _log_int(rng, 2, max(2, min(256, 262144 // hi)))
        return dict(_PACKED, **dict(common, nseq=nseq, lo=lo, hi=hi, len_seed=rng.randrange(1 << 20), causal=rng.random() < 0.8,
                                    smooth=rng.random() < 0.8, lse=rng.random() < 0.15, k_offset=rng.choice([0.0, 2.0])))
    c = dict(_BASE, **common)
    c.update(layout=layout, k_offset=rng.choice([0.0, 2.0]))
    if what == "decode":
        c.update(B=_log_int(rng, 1, 16), Sq=rng.choice([1, 1, 2, 4, 8]), Skv=_log_int(rng, 512, 32768))
        while c["B"] * Hkv * c["Skv"] > 1 << 22:
            c["B"] = max(1, c["B"] // 2)
            c["Skv"] = c["Skv"] if c["B"] > 1 else min(c["Skv"], (1 << 22) // Hkv)
        return c
    if what == "cross":
        c.update(B=rng.choice([1, 2, 4]), Sq=_log_int(rng, 512, 32768), Skv=_log_int(rng, 16, 1024))
        return c
    hi = {"self": 16384, "mask": 3000, "lse": 8192, "steps": 12000, "recipe": 8192}[what]
    S = _log_int(rng, 128, hi)
    c.update(Sq=S, Skv=S, B=max(1, min(rng.choice([1, 2, 4, 8]), 65536 // S)), causal=rng.random() < 0.5, smooth=rng.random() < 0.85)
    if what == "self" and not c["causal"] and rng.random() < 0.3:
        c["outliers"] = 0.01
    if what == "mask":
        c.update(causal=False, mask=rng.choice(["documents", "padding", "bias"]), BLKQ=128, BLKK=64, B=min(c["B"], 4))
    if what == "lse":
        c.update(lse=True)
    if what == "steps":
        c.update(kind="steps", lse=rng.random() < 0.3)
    if what == "recipe":
        if rng.random() < 0.5:
            c.update(pv="fp8", BLKQ=128, BLKK=16)
        else:
            c.update(BLKQ=32, BLKK=64, q_interleave=8, k_interleave=4)
    return c


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
def _lengths(case):
    rng = random.Random(case["len_seed"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["nseq"])]


def _mask(case, g):
    """documents: True where query and key belong to the same document of the row ([B, 1, Sq, Skv]); padding: True for the
    keys before each sequence's end ([B, 1, 1, Skv]); bias: an additive float32 bias that falls with the distance, with a
    slope and some noise of its own for every head ([1, Hq, Sq, Skv])."""
    B, Hq, Sq, Skv = case["B"], case["Hq"], case["Sq"], case["Skv"]
    if case["mask"] == "documents":
        starts = torch.rand((B, Skv), generator=g, device="cuda") < 4.0 / Skv
        doc = torch.cumsum(starts.int(), dim=1)
        return (doc[:, :Sq, None] == doc[:, None, :])[:, None].contiguous()
    if case["mask"] == "padding":
        ends = (torch.rand((B, 1), generator=g, device="cuda") * 0.5 + 0.5) * Skv
        return (torch.arange(Skv, device="cuda")[None] < ends.clamp(min=1))[:, None, None].contiguous()
    slope = torch.exp2(-torch.arange(1, Hq + 1, device="cuda") * (8.0 / Hq))[:, None, None]
    dist = (torch.arange(Sq, device="cuda")[:, None] - torch.arange(Skv, device="cuda")[None]).abs()
    noise = torch.randn((Hq, 1, Skv), generator=g, device="cuda") * 0.1
    return (noise - slope * dist)[None].contiguous()


def prepare(case, seed):
    """q, k, v ~ N(0, 1), K with an offset per channel (what K smoothing takes out) and, where asked, a share of the
    channels twenty times as large; the mask or the sequence boundaries a program has in hand."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype, D, Hq, Hkv = _DTYPES[case["dtype"]], case["D"], case["Hq"], case["Hkv"]
    if case["kind"] == "packed":
        lens = _lengths(case)
        T = sum(lens)
        cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")
        q = torch.randn((T, Hq, D), generator=g, device="cuda", dtype=dtype)
        k = torch.randn((T, Hkv, D), generator=g, device="cuda", dtype=dtype)
        v = torch.randn((T, Hkv, D), generator=g, device="cuda", dtype=dtype)
        if case["k_offset"]:
            k += torch.randn((1, Hkv, D), generator=g, device="cuda", dtype=dtype) * case["k_offset"]
        return dict(case=dict(case), q=q, k=k, v=v, cu=cu, longest=max(lens))
    nhd = case["layout"] == "NHD"

    def tensor(H, L):
        shape = (case["B"], L, H, D) if nhd else (case["B"], H, L, D)
        return torch.randn(shape, generator=g, device="cuda", dtype=dtype)

    q, k, v = tensor(Hq, case["Sq"]), tensor(Hkv, case["Skv"]), tensor(Hkv, case["Skv"])
    if case["k_offset"]:
        k += torch.randn((1, 1, Hkv, D) if nhd else (1, Hkv, 1, D), generator=g, device="cuda", dtype=dtype) * case["k_offset"]
    if case["outliers"]:
        large = (torch.rand((Hkv, D), generator=g, device="cuda") < case["outliers"]).to(dtype) * 19.0 + 1.0
        for t, H in ((q, Hq), (k, Hkv), (v, Hkv)):
            f = large.repeat_interleave(H // Hkv, 0)
            t *= f[None, None] if nhd else f[None, :, None]
    return dict(case=dict(case), q=q, k=k, v=v, mask=_mask(case, g) if case["mask"] else None)


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def run(state):
    c, q, k, v = state["case"], state["q"], state["k"], state["v"]
    blocks = dict(BLKQ=c["BLKQ"], BLKK=c["BLKK"])
    if c["kind"] == "packed":
        return sa.sageattn_varlen(q, k, v, state["cu"], state["cu"], state["longest"], state["longest"], is_causal=c["causal"],
                                  smooth_k=c["smooth"], pv_mode=c["pv"], return_lse=c["lse"], **blocks)
    blocks.update(q_interleave=c["q_interleave"], k_interleave=c["k_interleave"])
    if c["kind"] == "steps":
        km = sa.k_mean(k, c["layout"]) if c["smooth"] else None
        q8, qs, k8, ks = sa.per_block_int8(q, k, km=km, tensor_layout=c["layout"], **blocks)
        out, lse = sa.forward(q8, k8, v, qs, ks, tensor_layout=c["layout"], output_dtype=q.dtype, return_lse=c["lse"],
                              is_causal=c["causal"], pv_mode=c["pv"], **blocks)
        return dict(q8=q8, qs=qs, k8=k8, ks=ks, out=out, lse=lse)
    return sa.sageattn(q, k, v, tensor_layout=c["layout"], is_causal=c["causal"], smooth_k=c["smooth"], pv_mode=c["pv"],
                       return_lse=c["lse"], attn_mask=state["mask"], **blocks)


# ------------------------------------------------------------------------------------------------
# its work and tolerance
# ------------------------------------------------------------------------------------------------
def work(case):
    """Bytes: q, k, v (and the mask) read once, the outputs written once.  Operations: 4 * Hq * Sq * Skv * D per sequence
    (two products, a multiply and an add each), half of that when causal."""
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    half = 0.5 if case["causal"] else 1.0
    if case["kind"] == "packed":
        lens = _lengths(case)
        T = sum(lens)
        return {"bytes": 2 * D * T * (2 * Hq + 2 * Hkv) + (4 * Hq * T if case["lse"] else 0),
                "flops": half * sum(4.0 * Hq * n * n * D for n in lens)}
    B, Sq, Skv = case["B"], case["Sq"], case["Skv"]
    nbytes = 2 * D * B * (2 * Hq * Sq + 2 * Hkv * Skv)
    if case["lse"]:
        nbytes += 4 * B * Hq * Sq
    if case["mask"]:
        nbytes += {"documents": B * Sq * Skv, "padding": B * Skv, "bias": 4 * Hq * Sq * Skv}[case["mask"]]
    if case["kind"] == "steps":   # the INT8 operands and their scales are results too
        nbytes += D * B * (Hq * Sq + Hkv * Skv) + 4 * B * (Hq * -(-Sq // case["BLKQ"]) + Hkv * -(-Skv // case["BLKK"]))
    return {"bytes": nbytes, "flops": half * 4.0 * B * Hq * Sq * Skv * D}


def tolerance(case):
    """FP16 P.V: about four times what one pass differs from the same formula in 64 bits on the same INT8 operands (relative
    2.9e-4 for float16 outputs, 1.7e-3 for bfloat16 ones; with outlier channels 1.1e-3 and, largest, 0.09).  FP8 P.V: that
    comparison reads 3.1e-2 and 0.2 (e4m3 has three mantissa bits), so this is the size of the format's own rounding."""
    if case["pv"] == "fp8":
        return {"rel": 0.03, "max": 0.5}
    if case.get("outliers"):
        return {"rel": 6e-3, "max": 0.35}
    return {"rel": 6e-3, "max": 0.03} if case["dtype"] == "bfloat16" else {"rel": 1.2e-3, "max": 0.01}
