"""The work that this framework is used for, as cases that a timing program runs.

A case is one pass of one of the jobs below through the `Lane` calls that a
program makes for it, with the bank, the weights and the buffers that such a
program keeps already on the GPU:

  layer    the routed-expert layers of one decoded token: `layers` layer calls,
           each on its own hidden vector with its own picks (with `prenorm`,
           each from the residual stream that the pre-norm makes its input of)
  block    one token's MoE blocks: routed layer, shared-expert FFN, hc_post
  per32    the routed-expert layers in the per32 arithmetic
  grouped  one layer for T tokens at once (a batched decode step, a prefill chunk)
  shared   the shared-expert FFN of T tokens
  around   what surrounds the experts for T tokens: the pre-norm of the block's
           input, the router, hc_post

Decode cases walk several layers, so that the weights come from HBM as they do
in a model and not from a cache that the previous pass filled. All calls go to
one stream, as a decode loop's do.

`exact` evaluates the same layer arithmetic in 64 bits from the ggml blocks: the
activations are quantized as the formats define it, everything else is double.
"""
from __future__ import annotations

import numpy as np
import torch

import crosslane_amd as xl

XXS, XS, IQ1 = 16, 17, 29
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
IQ_BYTES = {XXS: 66, XS: 74, IQ1: 56}
DENSE = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}   # values, bytes per block
# Whole-expert type draw of the mixed layers (the benchmark's 40-layer pass)
MIX = ((XS, 0.17), (XXS, 0.19), (IQ1, 0.64))
H = 4            # hyper-connection streams
EPS = 1e-6


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # the smallest call: one expert of one layer (the lane's warm_compute)
        {"name": "layer_one_expert", "job": "layer", "dim": 4096, "ff": 3072, "experts": 64, "layers": 1, "kind": "iq2",
         "picks": 1, "limit": 0.0, "prenorm": False},
        # decode at batch 1, top-6, IQ2 experts: the headline benchmark's layer
        {"name": "layer_iq2", "job": "layer", "dim": 4096, "ff": 3072, "experts": 64, "layers": 8, "kind": "iq2",
         "picks": 6, "limit": 0.0, "prenorm": False},
        # the same at the real expert's shape and SwiGLU limit
        {"name": "layer_real", "job": "layer", "dim": 5120, "ff": 2304, "experts": 64, "layers": 8, "kind": "iq2",
         "picks": 6, "limit": 10.0, "prenorm": False},
        # decode over layers whose experts differ in type, the norm inside the call
        {"name": "layer_mixed", "job": "layer", "dim": 4096, "ff": 3072, "experts": 64, "layers": 8, "kind": "mixed",
         "picks": 6, "limit": 0.0, "prenorm": True},
        # one token's whole MoE blocks
        {"name": "block", "job": "block", "dim": 4096, "ff": 3072, "experts": 64, "layers": 6, "kind": "iq2",
         "picks": 6, "limit": 0.0, "shared": "q5q6"},
        # decode in the arithmetic of the production HIP lane
        {"name": "per32", "job": "per32", "dim": 4096, "ff": 3072, "experts": 64, "layers": 6, "kind": "iq2",
         "picks": 6, "limit": 0.0},
        # batched decode: a few tokens of different requests in one layer call
        {"name": "grouped_13", "job": "grouped", "dim": 5120, "ff": 2304, "experts": 384, "kind": "iq2", "tokens": 13,
         "picks": 6, "limit": 10.0, "routed": False},
        # a prefill chunk: the grouped benchmark
        {"name": "grouped_512", "job": "grouped", "dim": 4096, "ff": 3072, "experts": 384, "kind": "iq2",
         "tokens": 512, "picks": 6, "limit": 0.0, "routed": False},
        # a long prefill chunk, routed on the device
        {"name": "grouped_2048", "job": "grouped", "dim": 4096, "ff": 3072, "experts": 384, "kind": "iq2",
         "tokens": 2048, "picks": 6, "limit": 0.0, "routed": True},
        # a prefill chunk over a layer whose experts differ in type
        {"name": "grouped_mixed", "job": "grouped", "dim": 4096, "ff": 3072, "experts": 384, "kind": "mixed",
         "tokens": 512, "picks": 6, "limit": 0.0, "routed": False},
        # the shared expert of a prefill chunk
        {"name": "shared_512", "job": "shared", "dim": 4096, "ff": 3072, "tokens": 512, "types": "q5q6", "limit": 0.0},
        # norm, router and hc_post of a prefill chunk
        {"name": "around_512", "job": "around", "dim": 4096, "experts": 384, "tokens": 512, "picks": 6},
    ]


SHAPES = ((4096, 3072), (5120, 2304), (4096, 3072), (5120, 2304), (1024, 512), (2048, 1024))
SHARED_TYPES = {"q5q6": (Q5_K, Q5_K, Q6_K), "q4": (Q4_K, Q4_K, Q4_K), "q8": (Q8_0, Q8_0, Q8_0),
                "q4q6": (Q4_K, Q4_K, Q6_K)}


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    job = rng.choice(("layer", "layer", "block", "per32", "grouped", "grouped", "grouped", "shared", "shared", "around"))
    dim, ff = rng.choice(SHAPES)
    lim = rng.choice((0.0, 7.0, 10.0))
    kind = rng.choice(("iq2", "iq2", "iq1", "mixed"))
    k = rng.choice((1, 2, 3, 4, 5, 6, 6, 7, 8))
    if job == "layer":
        return {"job": job, "dim": dim, "ff": ff, "experts": rng.randint(24, 64), "layers": rng.randint(1, 8),
                "kind": kind, "picks": k, "limit": lim, "prenorm": rng.random() < 0.4}
    if job == "block":
        return {"job": job, "dim": dim, "ff": ff, "experts": rng.randint(24, 64), "layers": rng.randint(1, 6),
                "kind": kind, "picks": k, "limit": lim, "shared": rng.choice(sorted(SHARED_TYPES))}
    if job == "per32":
        return {"job": job, "dim": dim, "ff": ff, "experts": rng.randint(24, 64), "layers": rng.randint(1, 6),
                "kind": kind, "picks": k, "limit": lim}
    if job == "grouped":
        t = _log(rng, 2, 2048 if kind == "iq2" else 512)
        return {"job": job, "dim": dim, "ff": ff, "experts": rng.choice((64, 160, 256, 384)), "kind": kind,
                "tokens": t, "picks": k, "limit": lim, "routed": rng.random() < 0.5}
    if job == "shared":
        return {"job": job, "dim": dim, "ff": 256 * rng.randint(2, 12), "tokens": _log(rng, 1, 512),
                "types": rng.choice(sorted(SHARED_TYPES)), "limit": lim}
    return {"job": job, "dim": dim, "experts": rng.choice((64, 160, 256, 384)), "tokens": _log(rng, 1, 512), "picks": k}


# ---- inputs ------------------------------------------------------------------
def _types(case, seed):
    """Block types [layers, experts, 3] (gate, up, down)."""
    L, E = case.get("layers", 1), case["experts"]
    t = np.zeros((L, E, 3), np.int32)
    if case["kind"] == "mixed":
        rng = np.random.default_rng([seed, 3])
        t[:] = rng.choice([v for v, _ in MIX], size=(L, E), p=[p for _, p in MIX])[..., None]
    elif case["kind"] == "iq1":
        t[:] = IQ1
    else:
        t[..., :2], t[..., 2] = XXS, XS
    return t


def _route(logits, k):
    """Top-k of the softmax of each row, weights renormalized, in descending order."""
    ids = np.argsort(-logits, axis=1, kind="stable")[:, :k].astype(np.int32)
    p = np.exp(np.take_along_axis(logits, ids, 1).astype(np.float64))
    return ids, (p / p.sum(1, keepdims=True)).astype(np.float32)


def _dense(t, n, k, rng):
    """Random ggml blocks of a dense format with finite fp16 scales in [1e-3, 1e-2)."""
    values, size = DENSE[t]
    nb = n * (k // values)
    blk = rng.integers(0, 256, size=(nb, size), dtype=np.uint8)
    for off in {Q8_0: (0,), Q4_K: (0, 2), Q5_K: (0, 2), Q6_K: (208,)}[t]:
        blk[:, off:off + 2] = rng.uniform(1e-3, 1e-2, nb).astype(np.float16).view(np.uint8).reshape(nb, 2)
    return blk.reshape(-1)


def _inputs(case, seed):
    """Everything but the bank, as numpy arrays."""
    rng = np.random.default_rng([seed, 1])
    job, dim = case["job"], case["dim"]
    n = case["layers"] if job in ("layer", "block", "per32") else case["tokens"]
    a = {}
    if job != "shared":
        a["logits"] = rng.standard_normal((n, case["experts"])).astype(np.float32)
        a["ids"], a["w"] = _route(a["logits"], case["picks"])
    if job != "around":
        a["x"] = rng.standard_normal((n, dim)).astype(np.float32)
    if job == "layer" and case["prenorm"]:
        a["mix"] = np.zeros((n, 8), np.float32)
        a["mix"][:, 0] = 0.5 + rng.random(n)
        a["norm"] = (0.5 + rng.random(dim)).astype(np.float32)
    if job == "grouped":
        a["row"] = rng.standard_normal((n, dim)).astype(np.float32)   # the shared expert's rows
    if job == "block":
        a["res"] = rng.standard_normal((n, H, dim)).astype(np.float32)
    if job == "around":
        a["h"] = rng.standard_normal((n, H, dim)).astype(np.float32)
        a["y"] = rng.standard_normal((n, dim)).astype(np.float32)
        a["mix"] = rng.random((n, 8)).astype(np.float32)
        a["norm"] = (0.5 + rng.random(dim)).astype(np.float32)
    if job in ("block", "around"):
        a["post"] = (rng.random((n, 8)) * 2).astype(np.float32)
        a["comb"] = rng.random((n, 64)).astype(np.float32)
    if job in ("block", "shared"):
        ts = SHARED_TYPES[case["shared" if job == "block" else "types"]]
        ff = case["ff"]
        a["mats"] = [_dense(ts[0], ff, dim, rng), _dense(ts[1], ff, dim, rng), _dense(ts[2], dim, ff, rng)]
    return a


_STREAM = None


def _stream():
    """The one stream that the program's calls go to."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM.cuda_stream


def prepare(case, seed):
    job, dim = case["job"], case["dim"]
    a = _inputs(case, seed)
    d = {key: torch.from_numpy(v).cuda() for key, v in a.items() if key not in ("mats", "logits")}
    s = {"case": case, "stream": _stream(), "d": d}
    if job == "around":
        types = np.full((1, 1, 3), IQ1, np.int32)   # the calls use no bank
        s["lane"] = xl.Lane(256, 256, 1, 1, types)
        n, k = case["tokens"], case["picks"]
        s["logits"] = torch.from_numpy(a["logits"]).cuda()
        s["x"] = torch.zeros((n, dim), device="cuda")
        s["ids"] = torch.zeros((n, k), dtype=torch.int32, device="cuda")
        s["w"] = torch.zeros((n, k), device="cuda")
        s["out"] = torch.zeros((n, H, dim), device="cuda")
        return s
    if job == "shared":
        s["lane"] = xl.Lane(dim, 256, 1, 1, np.full((1, 1, 3), IQ1, np.int32), swiglu_limit=case["limit"])
        s["mats"] = [torch.from_numpy(m).cuda() for m in a["mats"]]
        s["work"] = torch.empty(xl.shared_work_bytes(dim, case["ff"], case["tokens"]), dtype=torch.uint8, device="cuda")
        s["out"] = torch.zeros((case["tokens"], dim), device="cuda")
        return s
    T = case["tokens"] if job == "grouped" else 0
    lane = s["lane"] = xl.Lane(dim, case["ff"], case.get("layers", 1), case["experts"], _types(case, seed),
                               max_picks=8, max_tokens=T, swiglu_limit=case["limit"])
    lane.generate(seed)
    s["out"] = torch.zeros_like(d["x"])
    if job == "grouped":
        s["logits"] = torch.from_numpy(a["logits"]).cuda() if case["routed"] else None
        return s
    n = case["layers"]
    # one layer's arguments each, as a decode loop keeps them
    s["per"] = [{key: d[key][l] for key in ("ids", "w", "x", "res", "post", "comb") if key in d} for l in range(n)]
    for l in range(n):
        s["per"][l]["out"] = s["out"][l]
    if job == "per32":
        s["y"] = torch.zeros((n, case["picks"], dim), device="cuda")
    if job == "layer" and case["prenorm"]:
        s["xn"] = torch.zeros_like(d["x"])
        for l in range(n):
            s["per"][l].update(h=d["x"][l].view(1, dim), mix=d["mix"][l], xn=s["xn"][l])
    if job == "block":
        s["mats"] = [torch.from_numpy(m).cuda() for m in a["mats"]]
        s["work"] = torch.empty(xl.shared_work_bytes(dim, case["ff"], 1), dtype=torch.uint8, device="cuda")
        s["post_out"] = torch.zeros_like(d["res"])
        for l in range(n):
            s["per"][l]["post_out"] = s["post_out"][l]
    return s


def run(s):
    case, lane, sp, d = s["case"], s["lane"], s["stream"], s["d"]
    job = case["job"]
    if job == "layer" and case["prenorm"]:
        for l, p in enumerate(s["per"]):
            lane.layer_forward_prenorm_async(l, p["ids"], p["w"], p["h"], p["mix"], d["norm"], p["xn"], p["out"],
                                             eps=EPS, stream=sp)
        return {"x": s["xn"], "out": s["out"]}
    if job == "layer":
        for l, p in enumerate(s["per"]):
            lane.layer_forward_async(l, p["ids"], p["w"], p["x"], p["out"], stream=sp)
        return {"out": s["out"]}
    if job == "per32":
        for l, p in enumerate(s["per"]):
            lane.layer_forward_per32_async(l, p["ids"], p["x"], s["y"][l], w=p["w"], out=p["out"], stream=sp)
        return {"y": s["y"], "out": s["out"]}
    if job == "block":
        ts = SHARED_TYPES[case["shared"]]
        for l, p in enumerate(s["per"]):
            lane.moe_block_async(l, p["ids"], p["w"], p["x"], ts, *s["mats"], case["ff"], s["work"], p["res"],
                                 p["post"], p["comb"], p["out"], p["post_out"], stream=sp)
        return {"out": s["out"], "post": s["post_out"]}
    if job == "grouped":
        if case["routed"]:
            lane.grouped_forward_routed_async(0, s["logits"], case["picks"], d["x"], s["out"], shared=d["row"], stream=sp)
        else:
            lane.grouped_forward_async(0, d["ids"], d["w"], d["x"], s["out"], shared=d["row"], stream=sp)
        return {"out": s["out"]}
    if job == "shared":
        lane.shared_forward_async(SHARED_TYPES[case["types"]], *s["mats"], case["ff"], d["x"], s["out"], s["work"],
                                  stream=sp)
        return {"out": s["out"]}
    lane.hc_pre_norm_async(d["h"], d["mix"], d["norm"], s["x"], eps=EPS, stream=sp)
    lane.route_async(s["logits"], case["picks"], s["ids"], s["w"], stream=sp)
    lane.hc_post_async(d["y"], d["h"], d["post"], d["comb"], s["out"], stream=sp)
    return {"x": s["x"], "ids": s["ids"], "w": s["w"], "out": s["out"]}


# ---- what a pass cannot do without ---------------------------------------------
def _expert_bytes(kind, dim, ff):
    per = dim * ff / 256
    if kind == "iq2":
        return per * (2 * IQ_BYTES[XXS] + IQ_BYTES[XS])
    if kind == "iq1":
        return per * 3 * IQ_BYTES[IQ1]
    return per * 3 * sum(IQ_BYTES[t] * p for t, p in MIX)


def work(case):
    job, dim, ff = case["job"], case["dim"], case.get("ff", 0)
    if job in ("layer", "block", "per32"):
        n, k = case["layers"], case["picks"]
        b = n * (k * (_expert_bytes(case["kind"], dim, ff) + 8) + 8 * dim)
        f = n * k * 6.0 * dim * ff
        if job == "layer" and case["prenorm"]:
            b += 4 * dim * (n + 1) + 32 * n
        if job == "per32":
            b += 4 * n * k * dim
        if job == "block":
            ts = SHARED_TYPES[case["shared"]]
            b += sum(dim * ff // DENSE[t][0] * DENSE[t][1] for t in ts) + n * (2 * H * dim * 4 + 72 * 4)
            f += n * 6.0 * dim * ff
        return {"bytes": float(b), "flops": float(f)}
    T = case["tokens"]
    if job == "grouped":
        E, k = case["experts"], case["picks"]
        touched = E * (1 - (1 - k / E) ** T)   # experts that T independent draws of k meet
        b = touched * _expert_bytes(case["kind"], dim, ff) + 12 * T * dim + (4 * E if case["routed"] else 8 * k) * T
        return {"bytes": float(b), "flops": 6.0 * T * k * dim * ff}
    if job == "shared":
        b = sum(dim * ff // DENSE[t][0] * DENSE[t][1] for t in SHARED_TYPES[case["types"]]) + 8 * T * dim
        return {"bytes": float(b), "flops": 6.0 * T * dim * ff}
    b = 4 * T * (H * dim + dim) + 4 * T * (dim + 2 * H * dim) + 4 * dim + T * (32 + 72 * 4) + T * (4 * case["experts"] + 8 * case["picks"])
    return {"bytes": float(b), "flops": T * dim * (2.0 * H + 4 + 2.0 * H * (H + 1))}


def tolerance(case):
    """The layers quantize h to 8 bits between their products: a sum in another
    order moves h by some units in the last place, and where that crosses a
    rounding midpoint one quant moves by a step, about 2e-3 of that pick's output
    (less in a group of tokens). The rest is 32-bit sums."""
    job = case["job"]
    if job == "around":   # 32-bit sums of a few terms: 5e-8 .. 7e-8 from 64 bits
        return {"rel": 3e-7, "max": 1e-5, "differ": 1e-3}
    if job == "per32":    # 1.2e-7 from 64 bits without a moved quant, which would be a few 1e-4 of one pick's row
        return {"rel": 1e-3, "max": 2e-2}
    T = case.get("tokens", 1)
    if job == "shared":   # 9e-6 from 64 bits at 512 tokens, a few moved quants among them
        return {"rel": 1e-3 * min(1.0, (4 / T) ** 0.5), "max": 2e-2}
    # layers: 1e-7 without a moved quant; grouped: 3e-5 .. 7e-5 at 13 .. 2048 tokens
    return {"rel": 4e-3 * min(1.0, (4 / T) ** 0.5), "max": 5e-2}


# ---- the same in 64 bits ---------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _u8(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_dev())


def _half(b):
    """fp16 values of byte pairs [..., 2]."""
    return b.contiguous().view(torch.float16)[..., 0].double()


_TABLES = {}


def _tables():
    """The formats' grids [n, 8] and sign rows [128, 8] as doubles."""
    if not _TABLES:
        def grid(which):
            raw = np.frombuffer(xl.codebook(which).astype("<u8").tobytes(), np.int8).reshape(-1, 8)
            return torch.from_numpy(raw.astype(np.float64)).to(_dev())
        signs = (xl.codebook(3)[:, None] >> np.arange(8, dtype=np.uint64)[None, :]) & np.uint64(1)
        _TABLES.update(xxs=grid(0), xs=grid(1), iq1=grid(2),
                       sign=torch.from_numpy(1.0 - 2.0 * signs.astype(np.float64)).to(_dev()))
    return _TABLES


def _iq_matrix(t, raw, n, k):
    """ggml IQ blocks as an n x k double matrix."""
    T = _tables()
    b = _u8(raw).view(-1, IQ_BYTES[t])
    nb = b.shape[0]
    if t == XXS:
        d = _half(b[:, 0:2])
        sub = b[:, 2:].reshape(nb, 8, 8).long()
        aux = sub[..., 4] | (sub[..., 5] << 8) | (sub[..., 6] << 16) | (sub[..., 7] << 24)
        sg = torch.stack([(aux >> (7 * j)) & 127 for j in range(4)], -1)
        s = (2 * (aux >> 28) + 1).double()
        v = T["xxs"][sub[..., :4]] * T["sign"][sg] * s[..., None, None]
    elif t == XS:
        d = _half(b[:, 0:2])
        c = b[:, 2:66].reshape(nb, 8, 4, 2).long()
        c = c[..., 0] | (c[..., 1] << 8)
        sc = b[:, 66:74].long()
        s = (2 * torch.stack([sc & 15, sc & 15, sc >> 4, sc >> 4], -1) + 1).double()
        v = T["xs"][c & 511] * T["sign"][c >> 9] * s[..., None]
    else:
        w = b[:, 48:56].reshape(nb, 4, 2).long()
        w = w[..., 0] | (w[..., 1] << 8)
        bits = (w[:, 0] >> 12) | ((w[:, 1] >> 8) & 0xF0) | ((w[:, 2] >> 4) & 0xF00) | (w[:, 3] & 0xF000)
        d = torch.stack([bits & 255, bits >> 8], -1).to(torch.uint8)
        d = _half(d)
        qs = b[:, :32].reshape(nb, 8, 4).long()
        qh = b[:, 32:48].reshape(nb, 8, 2).long()
        nib = torch.stack([qh & 15, qh >> 4], -1).reshape(nb, 8, 4)
        sub = torch.arange(8, device=b.device)
        ww = w[:, sub >> 1]
        s0 = 2 * ((ww >> (6 * (sub & 1))) & 7) + 1
        s1 = 2 * ((ww >> (6 * (sub & 1) + 3)) & 7) + 1
        s = torch.stack([s0, s0, s1, s1], -1).double()
        delta = torch.where((nib & 8) > 0, -1.0, 1.0).double()
        v = (8 * T["iq1"][qs | ((nib & 7) << 8)] + delta[..., None]) * s[..., None]
    return (v.reshape(nb, 256) * (d[:, None] / 8)).view(n, k)


def _dense_matrix(t, raw, n, k):
    """ggml Q8_0 / Q4_K / Q5_K / Q6_K blocks as an n x k double matrix."""
    b = _u8(raw).view(-1, DENSE[t][1])
    nb = b.shape[0]
    if t == Q8_0:
        return (b[:, 2:].contiguous().view(torch.int8).double() * _half(b[:, 0:2])[:, None]).view(n, k)
    if t == Q6_K:
        ql, qh = b[:, :128].view(nb, 2, 2, 32).int(), b[:, 128:192].view(nb, 2, 32).int()
        q = torch.stack([(ql[:, :, c & 1] >> (4 * (c >> 1)) & 15) | ((qh >> (2 * c) & 3) << 4) for c in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(nb, 16, 1)
        return ((q.double() - 32).view(nb, 16, 16) * sc * _half(b[:, 208:210])[:, None, None]).view(n, k)
    d, m = _half(b[:, 0:2]), _half(b[:, 2:4])
    sb = b[:, 4:16].int()
    sc = torch.cat([sb[:, :4] & 63, (sb[:, 8:12] & 15) | (sb[:, :4] >> 6 << 4)], 1).double()
    mn = torch.cat([sb[:, 4:8] & 63, (sb[:, 8:12] >> 4) | (sb[:, 4:8] >> 6 << 4)], 1).double()
    qs = b[:, 48:176] if t == Q5_K else b[:, 16:144]
    qs = qs.reshape(nb, 4, 32).int()
    q = torch.stack([qs & 15, qs >> 4], 2).view(nb, 8, 32)
    if t == Q5_K:
        qh = b[:, 16:48].int()
        q = q | (torch.stack([qh >> c & 1 for c in range(8)], 1) << 4)
    return ((d[:, None] * sc)[..., None] * q.double() - (m[:, None] * mn)[..., None]).view(n, k)


def _q8k(x):
    """Q8_K of rows of float32 values, as the doubles that the quants stand for."""
    v = np.ascontiguousarray(x, np.float32).reshape(-1, 256)
    mx = np.take_along_axis(v, np.abs(v).argmax(1)[:, None], 1)
    with np.errstate(divide="ignore", invalid="ignore"):
        inv = np.float32(-127.0) / mx
        q = np.minimum(np.rint(inv * v), 127).astype(np.float64)
        d = (np.float32(1.0) / inv).astype(np.float64)
    q = np.where(mx == 0, 0.0, q * np.where(mx == 0, 0.0, d))
    return torch.from_numpy(q.reshape(x.shape)).to(_dev())


def _q32(x):
    """Per-32 quants (d = max / 127) of rows of float32 values, as doubles."""
    v = np.ascontiguousarray(x, np.float32).reshape(-1, 32)
    d = np.abs(v).max(1, keepdims=True) / np.float32(127.0)
    with np.errstate(divide="ignore", invalid="ignore"):
        q = np.where(d > 0, np.rint(v / d), 0).astype(np.float64)
    return torch.from_numpy((q * d.astype(np.float64)).reshape(x.shape)).to(_dev())


def _swiglu(g, u, lim):
    if lim > 0:
        g, u = g.clamp(max=lim), u.clamp(-lim, lim)
    return g / (1 + torch.exp(-g)) * u


def _ffn(mats, x, quant, lim):
    """down . quant(SwiGLU(gate . quant(x), up . quant(x))) of rows x (float32)."""
    a = quant(x)
    h = _swiglu(a @ mats[0].T, a @ mats[1].T, lim)
    return quant(h.float().cpu().numpy()) @ mats[2].T


def _expert(case, types, seed, layer, e):
    dim, ff = case["dim"], case["ff"]
    out = []
    for r in range(3):
        t = int(types[layer, e, r])
        n, k = (ff, dim) if r < 2 else (dim, ff)
        out.append(_iq_matrix(t, xl.generate_host(t, seed, layer, e, r, n, k), n, k))
    return out


def _pre_norm(h, mix, norm):
    """h [n, H, D], mix [n, >= H], norm [D]: mixed streams, then the RMS norm."""
    v = np.einsum("nj,njd->nd", mix[:, :h.shape[1]].astype(np.float64), h.astype(np.float64))
    return v / np.sqrt((v * v).mean(1, keepdims=True) + EPS) * norm.astype(np.float64)


def _post(y, res, post, comb):
    n, hh, _ = res.shape
    c = comb[:, :hh * hh].astype(np.float64).reshape(n, hh, hh)
    return post[:, :hh, None].astype(np.float64) * y[:, None, :] + np.einsum("njk,njd->nkd", c, res.astype(np.float64))


def _router(logits, k):
    """Scores sqrt(softplus(l)) (l itself above 20), top-k, weights normalized."""
    l = logits.astype(np.float64)
    s = np.sqrt(np.where(l > 20, l, np.log1p(np.exp(np.minimum(l, 20)))))
    ids = np.argsort(-s, axis=1, kind="stable")[:, :k]
    p = np.take_along_axis(s, ids, 1)
    return ids, p / (p.sum(1, keepdims=True) + 1e-20)


def exact(case, seed):
    job, dim = case["job"], case["dim"]
    a = _inputs(case, seed)
    lim = case.get("limit", 0.0)
    if job == "around":
        _, w = _router(a["logits"], case["picks"])
        return {"x": _pre_norm(a["h"], a["mix"], a["norm"]), "ids": None, "w": w,
                "out": _post(a["y"].astype(np.float64), a["h"], a["post"], a["comb"])}
    shared = None
    if job in ("shared", "block"):
        ts, ff = SHARED_TYPES[case["types" if job == "shared" else "shared"]], case["ff"]
        shared = [_dense_matrix(t, m, *((ff, dim) if r < 2 else (dim, ff)))
                  for r, (t, m) in enumerate(zip(ts, a["mats"]))]
    if job == "shared":
        return {"out": _ffn(shared, a["x"], _q32, lim)}
    types = _types(case, seed)
    if job == "grouped":
        ids, w = _router(a["logits"], case["picks"]) if case["routed"] else (a["ids"], a["w"])
        out = torch.from_numpy(a["row"]).to(_dev()).double()
        for e in np.unique(ids):
            tok, pick = np.nonzero(ids == e)
            y = _ffn(_expert(case, types, seed, 0, int(e)), a["x"][tok], _q8k, lim)
            out[torch.from_numpy(tok).to(_dev())] += torch.from_numpy(w[tok, pick].astype(np.float64)).to(_dev())[:, None] * y
        return {"out": out}
    x = a["x"]
    if job == "layer" and case["prenorm"]:
        x64 = _pre_norm(x[:, None, :], a["mix"], a["norm"])
        x = x64.astype(np.float32)
    quant = _q32 if job == "per32" else _q8k
    n, k = case["layers"], case["picks"]
    y = torch.zeros((n, k, dim), dtype=torch.float64, device=_dev())
    for l in range(n):
        for i in range(k):
            y[l, i] = _ffn(_expert(case, types, seed, l, int(a["ids"][l, i])), x[l:l + 1], quant, lim)[0]
    out = (y * torch.from_numpy(a["w"]).to(_dev()).double()[..., None]).sum(1)
    if job == "per32":
        return {"y": y, "out": out}
    if job == "block":
        out = out + _ffn(shared, x, _q32, lim)
        return {"out": out, "post": _post(out.cpu().numpy(), a["res"], a["post"], a["comb"])}
    return {"x": x64, "out": out} if case["prenorm"] else {"out": out}
