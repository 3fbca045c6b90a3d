"""Measurement cases of the FP8 attention forward: what a user of this package has it do, over its whole range.

    listed()          the named cases
    draw(rng)         one more case of the same ranges
    prepare(case, s)  the tensors a program holds before the call, on the GPU, from the seed alone
    run(state)        one call of `attention_cutlass_fp8.flash_attention_v2_cutlass`
    work(case)        bytes and operations the call cannot do without
    tolerance(case)   how far two correct implementations may be apart

A case is a flat dict: B, H, Hk (k/v heads), Nq, Nk, d, causal, bottom_right (mask alignment), dtype ("e4m3" / "e5m2"),
out ("fp16" or "fp8": the type of the inputs), vt (v handed over as [B,Hk,d,Nk]), lse (log-sum-exp wanted as well), scale ("d":
1/sqrt(d), "n": 1/sqrt(Nk), the reference's choice) and dist (distribution of q/k/v).
"""
import math

import torch

from attention_cutlass_fp8 import flash_attention_v2_cutlass

HEAD_DIMS = (32, 64, 96, 128, 160, 192, 224, 256)
# the most a drawn case may ask for: the logits of the largest listed case (weighted by the head dim above 128, at least 128 query
# rows per head), and the k/v bytes of a large decode batch
MAX_LOGITS = 16.0 * 16384 * 16384
MAX_KV_BYTES = 600e6


def _case(name=None, B=1, H=16, Hk=None, Nq=1024, Nk=None, d=128, causal=False, bottom_right=False, dtype="e4m3", out="fp16",
          vt=False, lse=False, scale="d", dist="normal"):
    c = dict(B=B, H=H, Hk=H if Hk is None else Hk, Nq=Nq, Nk=Nq if Nk is None else Nk, d=d, causal=causal,
             bottom_right=bottom_right, dtype=dtype, out=out, vt=vt, lse=lse, scale=scale, dist=dist)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest call anyone makes (a unit test, a toy model): launch latency
        _case("tiny-full-n128-d64", H=2, Nq=128, d=64),
        # first row of the reference's benchmark table in its own calling convention: v transposed, fp8 output, clamped inputs
        _case("table-causal-h16-n1024-d64", Nq=1024, d=64, causal=True, vt=True, out="fp8", scale="n", dist="clamped"),
        # a short-sequence encoder batch
        _case("encoder-full-b4-n1024-d64", B=4, Nq=1024, d=64),
        # last row of the reference's benchmark table: a long causal prefill with many heads
        _case("table-causal-h64-n4096-d128", H=64, Nq=4096, causal=True, scale="n", dist="clamped"),
        # the headline workload
        _case("headline-full-b2-h32-n4096-d128", B=2, H=32, Nq=4096),
        # a long causal prefill with few heads and peaked rows
        _case("causal-h8-n16000-d128-peaked", H=8, Nq=16000, causal=True, dist="student_t"),
        # the longest full attention of the shape sweep: the largest case
        _case("full-h16-n16384-d128", H=16, Nq=16384),
        # sequences as they come, no multiple of any tile, with the log-sum-exp a training or context-parallel program keeps
        _case("ragged-full-b2-h16-n2999-d128-lse", B=2, Nq=2999, lse=True),
        # one decode step of a serving batch, grouped k/v heads, odd context length
        _case("decode-b16-h32k8-n8191-d128", B=16, H=32, Hk=8, Nq=1, Nk=8191, causal=True, bottom_right=True),
        # one decode step of a single long conversation: latency
        _case("decode-b1-h32k8-n32768-d128", H=32, Hk=8, Nq=1, Nk=32768, causal=True, bottom_right=True),
        # one chunk of a chunked prefill against a long context
        _case("chunk-512-of-16384-h32k8-d128", H=32, Hk=8, Nq=512, Nk=16384, causal=True, bottom_right=True),
        # the other input format, the widest heads, fp8 output
        _case("e5m2-causal-h16-n2048-d256-fp8out", Nq=2048, d=256, causal=True, dtype="e5m2", out="fp8"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("self", "self", "self", "self", "decode", "decode", "chunk"))
    d = rng.choice((64, 128, 128, 128) + HEAD_DIMS)
    H = rng.choice((2, 4, 8, 12, 16, 24, 32, 40, 64))
    group = rng.choice([g for g in (1, 1, 2, 4, 8) if H % g == 0])
    dtype = rng.choice(("e4m3", "e4m3", "e4m3", "e5m2"))
    out = rng.choice(("fp16", "fp16", "fp8"))
    lse = rng.random() < 0.3
    dist = rng.choice(("normal", "normal", "normal_half", "student_t", "clamped"))
    scale = "n" if dist == "clamped" else "d"
    causal, bottom_right, vt = True, True, False
    if kind == "self":
        Nq = _log_int(rng, 64, 16384)
        if rng.random() < 0.5:
            Nq = max(64, Nq // 64 * 64)
        Nk, causal, bottom_right = Nq, rng.random() < 0.5, False
        vt = Nk % 16 == 0 and rng.random() < 0.3
        B = rng.choice((1, 1, 2, 4, 8))
    elif kind == "decode":
        Nq, Nk = rng.choice((1, 1, 1, 2, 4, 8)), _log_int(rng, 100, 131072)
        B = rng.choice((1, 2, 4, 8, 16, 32, 64))
    else:
        Nq = _log_int(rng, 16, 2048)
        Nk = Nq + _log_int(rng, 64, 65536)
        B = rng.choice((1, 1, 2))
    c = _case(B=B, H=H, Hk=H // group, Nq=Nq, Nk=Nk, d=d, causal=causal, bottom_right=bottom_right, dtype=dtype, out=out, vt=vt,
              lse=lse, scale=scale, dist=dist)

    def too_large():
        logits = c["B"] * c["H"] * _pairs(c) * max(1.0, 128.0 / c["Nq"]) * max(1.0, c["d"] / 128.0)
        return logits > MAX_LOGITS or 2.0 * c["B"] * c["Hk"] * c["Nk"] * c["d"] > MAX_KV_BYTES
    while too_large() and c["B"] > 1:
        c["B"] //= 2
    while too_large():  # fewer heads, then a shorter sequence
        if c["H"] > 2 * (c["H"] // c["Hk"]) and c["Hk"] % 2 == 0:
            c["H"], c["Hk"] = c["H"] // 2, c["Hk"] // 2
        else:
            c["Nk"] = c["Nk"] // 2 // 16 * 16
            c["Nq"] = c["Nk"] if kind == "self" else min(c["Nq"], c["Nk"])
    return c


def _values(shape, dist, gen):
    def normal():
        return torch.randn(shape, device="cuda", generator=gen, dtype=torch.float32)
    if dist == "normal":
        return normal()
    if dist == "normal_half":
        return normal().mul_(0.5)
    if dist == "clamped":  # the reference's recipe: nearly uniform attention
        return normal().mul_(0.5).clamp_(-0.1, 0.1)
    # Student-t with 3 degrees of freedom: a few keys dominate a row
    chi = normal().square_()
    for _ in range(2):
        chi.add_(normal().square_())
    return normal().div_(chi.div_(3.0).sqrt_()).clamp_(-448.0, 448.0)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = torch.float8_e5m2 if case["dtype"] == "e5m2" else torch.float8_e4m3fn
    q = _values((case["B"], case["H"], case["Nq"], case["d"]), case["dist"], gen).to(dtype)
    kv = (case["B"], case["Hk"], case["Nk"], case["d"])
    k = _values(kv, case["dist"], gen).to(dtype)
    if case["dist"] == "student_t":
        v = torch.rand(kv, device="cuda", generator=gen, dtype=torch.float32).mul_(2.0).sub_(1.0).to(dtype)
    else:
        v = _values(kv, case["dist"], gen).to(dtype)
    if case["vt"]:
        v = v.transpose(2, 3).contiguous()
    args = (q, k, v, bool(case["causal"]), 1.0 / math.sqrt(case["d"] if case["scale"] == "d" else case["Nk"]))
    options = {}
    if case["vt"]:
        options["v_transposed"] = True
    if case["out"] == "fp8":
        options["out_dtype"] = dtype
    if case["lse"]:
        options["return_lse"] = True
    if case["bottom_right"]:
        options["causal_bottom_right"] = True
    return args, options


def run(state):
    args, options = state
    return flash_attention_v2_cutlass(*args, **options)


def _pairs(case):
    """(query, key) pairs that are visible, per head"""
    nq, nk = case["Nq"], case["Nk"]
    if not case["causal"]:
        return float(nq) * nk
    shift = nk - nq if case["bottom_right"] else 0
    first, last = shift + 1, shift + nq  # keys seen by the first and by the last query, before the limits 0 and nk
    if first >= 1 and last <= nk:
        return 0.5 * nq * (first + last)
    return float(sum(min(nk, max(0, shift + 1 + i)) for i in range(nq)))


def work(case):
    q = float(case["B"]) * case["H"] * case["Nq"]
    kv = 2.0 * case["B"] * case["Hk"] * case["Nk"] * case["d"]
    out = q * case["d"] * (1 if case["out"] == "fp8" else 2) + (4.0 * q if case["lse"] else 0.0)
    return {"bytes": q * case["d"] + kv + out, "flops": 4.0 * case["B"] * case["H"] * _pairs(case) * case["d"]}


def tolerance(case):
    # The weights are rounded to fp8 against the running row maximum; sums are fp32.  Another correct order of those sums moves
    # an output by an ulp of its type now and then (fp16: 2^-11; fp8: one step of 2^-3 or 2^-2 of the value, for few values), and a
    # weight that lies on a rounding boundary by one fp8 step, seldom.
    if case["out"] == "fp8":
        return {"rel": 0.015, "max": 0.27} if case["dtype"] == "e5m2" else {"rel": 0.01, "max": 0.14}
    return {"rel": 0.003, "max": 0.12}
