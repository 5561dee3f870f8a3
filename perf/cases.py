"""The calls whose speed this framework is judged by: what they are, their inputs, and their results.

Every case goes through a public entry point: `sageattn` (quantized attention, the K/V prologue and
the main loop in one call), or `HipPrologue.quant_kv` (the K/V quantization on its own, as a program
that keeps quantized K/V calls it). `listed()` names the calls that stand for real use, `draw(rng)`
gives others of the same ranges.

A case of `"op": "attn"` holds B, H, H_kv, N, N_kv, D, the dtype, the layout, `causal`, `lse`
(`return_lse`), `smooth_v`, `fused` (Q, K and V are views of one fused QKV projection) and
`outliers` (the share of K rows that are scaled by 50).
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "sageattention-rdna4_amd"))

#: the largest call that `draw` gives, in operations: the largest listed one's are 2.8e13
MAX_OPS = 1.2e13


def attn(name, B, H, N, D=128, *, H_kv=None, N_kv=None, dtype="fp16", layout="HND", causal=False,
         lse=False, smooth_v=False, fused=False, outliers=0.0):
    case = {"op": "attn", "B": B, "H": H, "H_kv": H_kv or H, "N": N, "N_kv": N_kv or N, "D": D,
            "dtype": dtype, "layout": layout, "causal": causal, "lse": lse, "smooth_v": smooth_v,
            "fused": fused, "outliers": outliers}
    if name:
        case["name"] = name
    return case


def quant(name, B, H, N, D=128, *, dtype="fp16", layout="HND"):
    case = {"op": "quant", "B": B, "H": H, "N": N, "D": D, "dtype": dtype, "layout": layout}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a short call (a text or low-resolution sequence, a few hundred tokens): launches and
        # latency are most of it
        attn("short_288", 1, 48, 288),
        # one image's tokens at low resolution
        attn("image_1024", 1, 48, 1024),
        # text conditioning of video tokens: many queries on a few hundred keys of another length
        attn("cross_512", 1, 24, 8771, N_kv=512, layout="NHD"),
        # a language model's prefill: grouped K/V heads, bf16, causal, with the logsumexp that a
        # caller needs to merge it with attention over cached keys; an odd length
        attn("prefill_gqa", 1, 32, 3001, H_kv=8, dtype="bf16", causal=True, lse=True),
        # a 1024 x 1024 image's self-attention at head_dim 64
        attn("image_d64", 1, 10, 4096, D=64),
        # a batched image model straight from its fused QKV projection, V smoothed
        attn("fused_smooth_v", 2, 24, 4250, layout="NHD", fused=True, smooth_v=True),
        # a batch of images, NHD
        attn("batch_nhd", 8, 24, 4096, layout="NHD"),
        # a short video, causal, with outlier tokens in K; a length that is no multiple of a tile
        attn("video_causal", 1, 48, 8771, causal=True, outliers=1e-3),
        # a long video at head_dim 64
        attn("video_d64", 1, 30, 17550, D=64),
        # a long bf16 prefill
        attn("long_bf16", 1, 48, 16384, dtype="bf16", causal=True),
        # the longest call: a long video, causal (the benchmark's default workload)
        attn("long_video", 1, 48, 47520, causal=True),
        # K and V quantized once, kept by the caller
        quant("quant_kv", 1, 48, 8771),
    ]


def ops(case):
    """Multiplies and adds of the two products, counted as 4 B H N N_kv D, halved when causal."""
    full = 4.0 * case["B"] * case["H"] * case["N"] * case["N_kv"] * case["D"]
    return full / 2 if case["causal"] else full


def _length(rng, lo, hi):
    """A length between lo and hi, spread over its logarithm; about half are multiples of 64."""
    n = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, n // 64 * 64) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(("self", "self", "self", "prefill", "cross", "quant"))
    dtype = rng.choice(("fp16", "fp16", "bf16"))
    layout = rng.choice(("HND", "NHD"))
    D = rng.choice((128, 128, 64))
    if kind == "quant":
        return quant(None, rng.choice((1, 1, 2)), rng.choice((8, 24, 48)),
                     _length(rng, 288, 47520), D, dtype=dtype, layout=layout)
    if kind == "prefill":
        H_kv = rng.choice((2, 4, 8))
        case = attn(None, rng.choice((1, 1, 2)), H_kv * rng.choice((4, 8)),
                    _length(rng, 288, 32768), D, H_kv=H_kv, dtype=rng.choice(("fp16", "bf16")),
                    layout=layout, causal=True, lse=rng.random() < 0.5)
    elif kind == "cross":
        case = attn(None, rng.choice((1, 2)), rng.choice((10, 24, 48)),
                    _length(rng, 1024, 32768), D, N_kv=_length(rng, 77, 1024), dtype=dtype,
                    layout=layout)
    else:
        smooth_v = rng.random() < 0.2
        fused = layout == "NHD" and rng.random() < 0.4
        case = attn(None, rng.choice((1, 1, 2, 8)), rng.choice((8, 10, 24, 30, 48)),
                    _length(rng, 256, 47520), D, dtype=dtype, layout=layout,
                    causal=rng.random() < 0.4, smooth_v=smooth_v, fused=fused,
                    outliers=rng.choice((0.0, 0.0, 1e-3)) if dtype == "fp16" else 0.0)
    while ops(case) > MAX_OPS:   # a shorter call of the same kind
        case["N"] = max(1, int(case["N"] * 0.7))
        if kind != "cross":
            case["N_kv"] = case["N"]
    return case


def _torch_dtype(case):
    return torch.float16 if case["dtype"] == "fp16" else torch.bfloat16


def _inputs(case, seed):
    """Q, K, V in the case's layout: unit normal, with the per-channel offsets that a projection's
    bias and its data give K (what smoothing K is for) and V, and outlier rows in K."""
    B, N, D = case["B"], case["N"], case["D"]
    H, H_kv, N_kv = case.get("H", 1), case.get("H_kv", case["H"]), case.get("N_kv", N)
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = _torch_dtype(case)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)

    def tensor(h, n, offset, outliers):
        x = normal(B, h, n, D)
        if outliers:
            rows = torch.rand(B, h, n, 1, generator=g, device="cuda") < outliers
            x = torch.where(rows, 50.0 * x, x)
        if offset:
            x += offset * normal(B, h, 1, D)
        return x.to(dt)

    q = tensor(H, N, 0.0, 0.0) if case["op"] == "attn" else None
    k = tensor(H_kv, N_kv, 2.0, case.get("outliers", 0.0))
    v = tensor(H_kv, N_kv, 0.5, 0.0)
    if case["layout"] == "NHD":
        if case.get("fused"):
            qkv = torch.stack([t.transpose(1, 2) for t in (q, k, v)], dim=2).contiguous()
            return [qkv[:, :, i] for i in range(3)]
        q, k, v = (None if t is None else t.transpose(1, 2).contiguous() for t in (q, k, v))
    return [q, k, v]


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    if case["op"] == "quant":
        from sageattention.sk1_backend.hip_prologue import HipPrologue
        if case["layout"] == "NHD":      # quant_kv takes logical (B, H, N, D) views
            k, v = k.transpose(1, 2), v.transpose(1, 2)
        return {"case": case, "k": k, "v": v, "prologue": HipPrologue.get()}
    from sageattention import sageattn
    return {"case": case, "q": q, "k": k, "v": v, "sageattn": sageattn}


def run(state):
    case = state["case"]
    if case["op"] == "quant":
        r = state["prologue"].quant_kv(state["k"], state["v"], smooth_k=True,
                                       int8=case["dtype"] == "fp16", fold=True)
        if r is None:
            raise RuntimeError("quant_kv: %s" % state["prologue"].last_error)
        k8, sk, v8t, sv, s = r
        return {"k8": k8.view(torch.uint8), "sk": sk, "v8t": v8t.view(torch.uint8), "sv": sv,
                "s": s}
    out = state["sageattn"](state["q"], state["k"], state["v"], tensor_layout=case["layout"],
                            is_causal=case["causal"], return_lse=case["lse"],
                            smooth_v=case["smooth_v"])
    return {"o": out[0], "lse": out[1]} if case["lse"] else {"o": out}


def work(case):
    B, N, D = case["B"], case["N"], case["D"]
    if case["op"] == "quant":
        n_pad, planes = (N + 63) // 64 * 64, B * case["H"]
        # K and V read once; K8, V8T, SK, SV and S written once
        return {"bytes": planes * (2 * 2 * N * D + 2 * n_pad * D + 2 * 4 * n_pad + 4), "flops": 0}
    q, kv = B * case["H"] * N * D * 2, B * case["H_kv"] * case["N_kv"] * D * 2
    lse = B * case["H"] * N * 4 if case["lse"] else 0
    return {"bytes": 2 * q + 2 * kv + lse, "flops": ops(case)}


def tolerance(case):
    # K8, V8T and the scales are fixed bit for bit by the scheme: one fp64 mean, correctly rounded
    # quotients, round half to even.
    if case["op"] == "quant":
        return "exact"
    # Against an implementation of the same scheme with its roundings and sums in another order:
    # scores that move by an fp32 rounding move a few e4m3 probabilities by one code. e4m3 Q.K
    # (bf16 inputs) has inexact matrix products besides, and outputs of 8 bits. About four times
    # what the scheme's emulation on the CPU differs by (rel 4.6e-5 and max 4e-3 for fp16, 4.4e-4
    # and 6.5e-2 for bf16, N = 288 .. 8771).
    if case["dtype"] == "fp16":
        return {"rel": 2e-4, "max": 2e-2}
    return {"rel": 2e-3, "max": 0.26}


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    if case["layout"] == "NHD":
        q, k, v = (None if t is None else t.transpose(1, 2) for t in (q, k, v))
    if case["op"] == "quant":
        return _exact_quant(case, k, v)
    B, H, N, D = q.shape
    H_kv, N_kv = k.shape[1], k.shape[2]
    sm = D ** -0.5
    out = torch.empty(B, H, N, D, dtype=torch.float64, device="cuda")
    lse = torch.empty(B, H, N, dtype=torch.float64, device="cuda") if case["lse"] else None
    rows = max(64, int(2e8) // N_kv)
    keys = torch.arange(N_kv, device="cuda")
    for b in range(B):
        for h in range(H):
            kk, vv = (t[b, h * H_kv // H].double() for t in (k, v))
            kt = kk.t().contiguous()
            for r0 in range(0, N, rows):
                r1 = min(N, r0 + rows)
                n = r1 if case["causal"] else N_kv     # later keys are masked for all these rows
                s = torch.mm(q[b, h, r0:r1].double(), kt[:, :n].contiguous()).mul_(sm)
                if case["causal"]:
                    live = keys[None, :n] <= torch.arange(r0, r1, device="cuda")[:, None]
                    s.masked_fill_(~live, float("-inf"))
                m = s.amax(dim=1, keepdim=True)
                s.sub_(m).exp_()
                total = s.sum(dim=1, keepdim=True)
                out[b, h, r0:r1] = torch.mm(s, vv[:n]) / total
                if lse is not None:
                    lse[b, h, r0:r1] = (m + total.log()).squeeze(1)
    if case["layout"] == "NHD":
        out = out.transpose(1, 2).contiguous()
    return {"o": out, "lse": lse} if case["lse"] else {"o": out}


def _exact_quant(case, k, v):
    B, H, N, D = k.shape
    n_pad = (N + 63) // 64 * 64
    kk, vv = (t.reshape(B * H, N, D).double() for t in (k, v))
    kk = kk - kk.mean(dim=1, keepdim=True)
    sk = torch.ones(B * H, n_pad, dtype=torch.float64, device="cuda")
    sv = torch.zeros(B * H, n_pad, dtype=torch.float64, device="cuda")
    sk[:, :N] = kk.abs().amax(dim=2).div(127.0 if case["dtype"] == "fp16" else 448.0).clamp_min(1e-12)
    sv[:, :N] = vv.abs().amax(dim=2).div(448.0).clamp_min(1e-12)
    s = sv.amax(dim=1).clamp_min(1.0)
    return {"k8": None, "sk": sk, "v8t": None, "sv": sv / s[:, None], "s": s}
