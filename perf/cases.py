"""Performance cases of ``sageattn``: the attention calls that programs make with it, over the range of sizes they use.

Diffusion models call it for short cross-attention (text or conditioning tokens), for self-attention of image tokens
and for few-head, long self-attention (VAE-like blocks); language models for causal prefill, with grouped-query heads
and with K smoothing, and for a few new queries against a long key range.  The listed sizes are the repository's
benchmark shapes and configurations, or generic ones; ``draw`` spreads over the ranges they stand for.

Every case is one call of the public ``sageattn`` on tensors in GPU memory.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sageattention-rdna3_amd"))

from sageattention import sageattn  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, b, hq, hkv, sq, sk, d, dtype, layout, causal=False, smooth_k=False, lse=False, k_offset=0.0,
          outliers=0.0):
    c = dict(b=b, hq=hq, hkv=hkv, sq=sq, sk=sk, d=d, dtype=dtype, layout=layout, causal=causal, smooth_k=smooth_k,
             lse=lse, k_offset=k_offset, outliers=outliers)
    return dict(c, name=name) if name else c


def listed():
    return [
        # image tokens attending 77 text tokens (the benchmark's SDXL02): the smallest call, one short launch
        _case("text_cross", 1, 10, 10, 4096, 77, 64, "fp16", "NHD"),
        # image tokens attending 512 conditioning tokens (Anima02)
        _case("cond_cross", 1, 16, 16, 4096, 512, 128, "bf16", "NHD"),
        # self-attention of a small image or a deep block (SDXL04), the direct kernel
        _case("self_short", 1, 20, 20, 1024, 1024, 64, "fp16", "NHD"),
        # short causal prefill, the longest that the dispatch sends to the direct kernel at head_dim 128
        _case("causal_short", 1, 32, 32, 2048, 2048, 128, "bf16", "HND", causal=True),
        # few queries against a long key range (a decode step): one query of each sequence of a batch, grouped heads,
        # with the LSE that merging with other key ranges needs
        _case("few_queries", 8, 32, 8, 1, 8192, 128, "bf16", "HND", lse=True),
        # image self-attention at head_dim 64 (the basic configuration, SDXL01)
        _case("self_d64", 1, 10, 10, 4096, 4096, 64, "fp16", "HND"),
        # causal prefill of a mid length and few heads
        _case("causal_mid", 1, 16, 16, 4096, 4096, 128, "bf16", "HND", causal=True),
        # image self-attention at head_dim 128 in the layout such models hold (Anima03)
        _case("self_d128", 1, 16, 16, 6144, 6144, 128, "bf16", "NHD"),
        # causal prefill of a batch whose keys carry a channel bias, smoothed
        _case("causal_smooth", 2, 32, 32, 8192, 8192, 128, "bf16", "HND", causal=True, smooth_k=True, k_offset=2.0),
        # grouped-query causal prefill of a long prompt
        _case("causal_gqa", 1, 32, 8, 16384, 16384, 128, "fp16", "NHD", causal=True),
        # the headline shape: long causal prefill
        _case("causal_16k", 1, 32, 32, 16384, 16384, 128, "bf16", "HND", causal=True),
        # the largest: a long ragged sequence with outlier channels, smoothed
        _case("ragged_long", 1, 40, 40, 32891, 32891, 128, "bf16", "HND", smooth_k=True, outliers=0.01),
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]; one in three a multiple of 64 where that fits."""
    n = int(round(lo * (hi / lo) ** rng.random()))
    if rng.random() < 1 / 3 and n >= 64:
        n = n // 64 * 64
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["text", "cond", "short", "causal_short", "few", "self", "vae", "causal", "long"])
    d = rng.choice([64, 128])
    dtype = rng.choice(["fp16", "bf16"])
    layout = rng.choice(["HND", "NHD"])
    b = rng.choice([1, 1, 2])
    h = rng.choice([8, 10, 16, 20, 24, 32])
    lse = rng.random() < 0.2
    smooth = rng.random() < 0.25
    offset = 2.0 if smooth else 0.0
    if kind == "text":
        sk = rng.choice([77, 154, 231, rng.randint(16, 256)])
        return _case(None, b, h, h, _log(rng, 256, 16384), sk, d, dtype, layout, lse=lse)
    if kind == "cond":
        return _case(None, b, h, h, _log(rng, 1024, 9216), _log(rng, 256, 1024), d, dtype, layout, lse=lse)
    if kind == "short":
        s = _log(rng, 128, 2048)
        return _case(None, b, h, h, s, s, d, dtype, layout, lse=lse)
    if kind == "causal_short":
        s = _log(rng, 128, 2048)
        return _case(None, b, h, rng.choice([h, h // 2]), s, s, d, dtype, layout, causal=True, lse=lse)
    if kind == "few":
        group = rng.choice([1, 2, 4, 8])
        hkv = rng.choice([4, 8])
        return _case(None, rng.choice([1, 2, 4, 8]), hkv * group, hkv, _log(rng, 1, 64), _log(rng, 1024, 32768), d,
                     dtype, layout, lse=lse)
    if kind == "self":
        s = _log(rng, 2304, 12288)
        return _case(None, b, h, h, s, s, d, rng.choice([dtype, dtype, dtype, "fp32"]), layout, smooth_k=smooth, lse=lse,
                     k_offset=offset)
    if kind == "vae":
        s = _log(rng, 4096, 24576)
        h = rng.randint(1, 5)
        return _case(None, 1, h, h, s, s, 128, rng.choice([dtype, dtype, "fp32"]), layout, lse=lse)
    if kind == "causal":
        s = _log(rng, 2049, 16384)
        return _case(None, b, h, rng.choice([h, h // 2]), s, s, d, dtype, layout, causal=True, smooth_k=smooth, lse=lse,
                     k_offset=offset)
    s = _log(rng, 12288, 32768)
    return _case(None, 1, rng.choice([8, 16, 24]), 8, s, s, 128, dtype, layout, causal=rng.random() < 0.5, smooth_k=smooth,
                 lse=lse, outliers=0.01 if smooth else 0.0)


def _inputs(case, seed):
    """q, k, v of the case's dtype and layout on the GPU: normal values; K with a bias per channel (k_offset its
    deviation) and a share of Q/K channels at twenty times the others (outliers) where the case says so."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    d, nhd = case["d"], case["layout"] == "NHD"

    def normal(h, s):
        shape = (case["b"], s, h, d) if nhd else (case["b"], h, s, d)
        return torch.randn(shape, generator=g, device="cuda")

    q, k, v = normal(case["hq"], case["sq"]), normal(case["hkv"], case["sk"]), normal(case["hkv"], case["sk"])
    if case["k_offset"]:
        off = torch.randn((case["b"], case["hkv"], 1, d), generator=g, device="cuda") * case["k_offset"]
        k += off.transpose(1, 2) if nhd else off
    if case["outliers"]:
        chans = torch.randperm(d, generator=g, device="cuda")[: max(1, round(case["outliers"] * d))]
        q[..., chans] *= 20.0
        k[..., chans] *= 20.0
    dt = DTYPES[case["dtype"]]
    return q.to(dt), k.to(dt), v.to(dt)


def prepare(case, seed):
    return _inputs(case, seed) + (case,)


def run(state):
    q, k, v, case = state
    return sageattn(q, k, v, tensor_layout=case["layout"], is_causal=case["causal"], return_lse=case["lse"],
                    smooth_k=case["smooth_k"])


def work(case):
    e = DTYPES[case["dtype"]].itemsize
    b, hq, hkv, sq, sk, d = (case[n] for n in ("b", "hq", "hkv", "sq", "sk", "d"))
    pairs = sq * sk
    if case["causal"]:  # top-left mask: row i sees keys 0..i
        n = min(sq, sk)
        pairs = n * (n + 1) // 2 + (sq - n) * sk
    nbytes = e * d * b * (2 * hq * sq + 2 * hkv * sk) + (4 * b * hq * sq if case["lse"] else 0)
    return {"bytes": nbytes, "flops": 4 * b * hq * d * pairs}


def tolerance(case):
    # The output's rounding, and P's to fp16.  Measured over the listed and drawn cases: against 64 bits bf16 rel 1.7e-3,
    # max 1.3e-2, fp16 rel 3.0e-4, max 1.3e-2 (the first rows of causal fp16, few keys and small values); the sums in
    # another order (three key ranges) bf16 rel 9.4e-4, max 7.8e-3, fp16 rel 3.6e-4, max 2.1e-3.
    return {"rel": 5e-3 if case["dtype"] == "bf16" else 1.4e-3, "max": 5e-2}


def _direct(case):
    """The documented dispatch (default thresholds): short key ranges use Q and K as they are."""
    sq, sk = case["sq"], case["sk"]
    if case["d"] == 64:
        if case["causal"] or sq < sk:
            return sk <= 6144
        return sk <= (2048 if case["layout"] == "HND" else 3072)
    return sk <= (4096 if sq * 2 < sk else 2048)


def _dequantised(x, group, pre=None, mean=None):
    """x [b, h, n, d] after INT8 rounding in groups of tokens, in 64 bits (the rounding itself is 32-bit arithmetic, as
    the quantised path defines it); pre: a factor folded into the values before they are rounded."""
    x = x.float()
    if mean is not None:
        x = x - mean
    b, h, n, d = x.shape
    groups = -(-n // group)
    a = torch.nn.functional.pad((x if pre is None else x * pre).abs(), (0, 0, 0, groups * group - n))
    amax = a.reshape(b, h, groups, group * d).amax(-1).clamp_min(1e-7)
    inv = torch.full_like(amax, 127.0) / amax
    if pre is not None:
        inv = inv * pre
    t = x * inv.repeat_interleave(group, 2)[:, :, :n, None]
    q8 = torch.trunc(t + torch.where(t >= 0, 0.5, -0.5)).clamp(-128, 127)
    return q8.double() * (amax / 127.0).repeat_interleave(group, 2)[:, :, :n, None].double()


def exact(case, seed):
    """Softmax attention in 64 bits of the values that the path's definition feeds it: Q and K as given (direct) or after
    their INT8 rounding (with the mean of K taken off first for smooth_k), V as fp16."""
    q, k, v = _inputs(case, seed)
    if case["layout"] == "NHD":
        q, k, v = (x.transpose(1, 2) for x in (q, k, v))
    dt = q.dtype
    if dt == torch.float32:
        q, k, v = q.half(), k.half(), v.half()
    b, hq, sq, d = q.shape
    hkv, sk = k.shape[1:3]
    scale = torch.tensor(d ** -0.5, dtype=torch.float32, device="cuda")
    pre = scale * torch.tensor(1.4426950408889634, dtype=torch.float32, device="cuda")  # scores in log2 units
    if _direct(case):
        qd, kd = q.double() * pre.double(), k.double()
    else:
        mean = k.double().mean(2, keepdim=True).to(k.dtype).float() if case["smooth_k"] else None
        qd, kd = _dequantised(q, 32, pre=pre), _dequantised(k, 16, mean=mean)
    vd = v.half().double()
    out = torch.empty((b, hq, sq, d), dtype=torch.float64, device="cuda")
    lse = torch.empty((b, hq, sq), dtype=torch.float64, device="cuda")
    cols = torch.arange(sk, device="cuda")
    for i in range(b):
        for h in range(hq):
            j = h // (hq // hkv)
            for r in range(0, sq, 4096):
                e = min(sq, r + 4096)
                n = min(sk, e) if case["causal"] else sk
                s = qd[i, h, r:e] @ kd[i, j, :n].T
                if case["causal"]:
                    s.masked_fill_(cols[None, :n] > torch.arange(r, e, device="cuda")[:, None], float("-inf"))
                m = s.amax(1, keepdim=True)
                p = s.sub_(m).exp2_()
                total = p.sum(1, keepdim=True)
                out[i, h, r:e] = (p @ vd[i, j, :n]) / total
                lse[i, h, r:e] = ((m + total.log2()) * 0.6931471805599453).squeeze(1)
    if case["layout"] == "NHD":
        out = out.transpose(1, 2).contiguous()
    return (out, lse) if case["lse"] else out
