"""The work this framework is timed on: what a serving or fine-tuning program
has the grouped 4-bit expert GEMM do, through its public entry points.

A case is one call pattern with its sizes:

  fwd    one projection: ``gemm_4bit_grouped`` / ``gemm_mxfp4_grouped`` (a
         decode step's call, a mixed batch, a prefill chunk)
  dgrad  the input gradient: ``dgrad_4bit_grouped`` / ``dgrad_mxfp4_grouped``
  step   one decode token's expert FFN through ``layers`` MoE layers, each
         with its own weights, captured once as a HIP graph and replayed:
         how a decode loop runs
  moe    the same with the routing on the device: ``moe_layer`` from router
         logits, ``layers`` of them in one graph
  train  ``fused_grouped_lora`` forward and backward: gradients of the
         activations and of the low-rank adapters

Shapes: "qwen" and "gptoss" are the two models whose expert shapes the
benchmark uses (128 experts of gate_up [1536, 2048] / down [2048, 768] with 8
per token; 32 experts of [5760, 2880] / [2880, 2880] with 4 per token); the
others are generic. ``tokens`` are routed to ``top_k`` distinct experts each,
uniformly or with a Zipf-like popularity (``skew``), and the calls get the
active experts' rows grouped, as a caller's MoE block groups them.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "grouped-nf4-gemm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mxfp4_grouped  # noqa: E402
import nf4_ffn  # noqa: E402
import nf4_grouped  # noqa: E402
import nf4_qlora  # noqa: E402
import nf4_route  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # the smallest call: one projection of one decode token, called eagerly
        dict(name="nf4_decode_1", kind="fwd", fmt="nf4", E=128, N=1536, K=2048, top_k=8,
             tokens=1, skew=0.0, ids="host", act="bf16"),
        # a decode token through 16 layers' own weights, one graph replay
        dict(name="nf4_step_1", kind="step", fmt="nf4", E=128, H=768, K=2048, top_k=8,
             tokens=1, skew=0.0, layers=16),
        # batch-16 decode with the routing on the device, one graph replay
        dict(name="nf4_moe_16", kind="moe", fmt="nf4", E=128, H=768, K=2048, top_k=8,
             tokens=16, skew=0.0, layers=4),
        # batch-64 decode of the second model and format, ids from its router
        dict(name="mxfp4_decode_64", kind="fwd", fmt="mxfp4", E=32, N=5760, K=2880, top_k=4,
             tokens=64, skew=0.0, ids="device", act="bf16"),
        # a small batch of a chunked prefill: about 32 rows an expert
        dict(name="nf4_chunk_512", kind="fwd", fmt="nf4", E=128, N=1536, K=2048, top_k=8,
             tokens=512, skew=0.0, ids="host", act="bf16"),
        # a generic shape off the tile sizes, ragged skewed groups, fp16 in
        dict(name="nf4_ragged_fp16", kind="fwd", fmt="nf4", E=60, N=1412, K=1408, top_k=6,
             tokens=1009, skew=0.8, ids="host", act="fp16"),
        # prefill of 4096 tokens, popular experts far larger than the others
        dict(name="nf4_prefill_skew", kind="fwd", fmt="nf4", E=128, N=1536, K=2048, top_k=8,
             tokens=4096, skew=1.0, ids="host", act="bf16"),
        # its second projection (short rows), even routing
        dict(name="nf4_prefill_down", kind="fwd", fmt="nf4", E=128, N=2048, K=768, top_k=8,
             tokens=4096, skew=0.0, ids="host", act="bf16"),
        # prefill of 2048 tokens of the second model and format
        dict(name="mxfp4_prefill", kind="fwd", fmt="mxfp4", E=32, N=5760, K=2880, top_k=4,
             tokens=2048, skew=0.0, ids="host", act="bf16"),
        # fine-tuning: the input gradients of both formats
        dict(name="nf4_dgrad", kind="dgrad", fmt="nf4", E=128, N=2048, K=768, top_k=8,
             tokens=2048, skew=0.0, ids="host"),
        dict(name="mxfp4_dgrad", kind="dgrad", fmt="mxfp4", E=32, N=5760, K=2880, top_k=4,
             tokens=1024, skew=0.0, ids="host"),
        # fine-tuning: a projection with fp32 adapters, forward and backward
        dict(name="nf4_lora_train", kind="train", fmt="nf4", E=128, N=1536, K=2048, top_k=8,
             tokens=1024, skew=0.0, rank=16),
    ]


# flops of the largest listed forward case (32768 rows of 1536 x 2048)
_MOST_FLOPS = 2.0 * 32768 * 1536 * 2048


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same kinds: sizes over the same ranges."""
    kind = rng.choice(["fwd", "fwd", "fwd", "fwd", "dgrad", "dgrad", "step", "moe", "train"])
    model = rng.choice(["qwen", "gptoss", "generic", "generic"])
    # the low-rank delta pads the groups to the widest, so fine-tuning batches
    # are the even ones
    skew = 0.0 if kind == "train" else rng.choice([0.0, 0.0, 0.5, 0.8, 1.0])
    if kind in ("step", "moe"):
        if model == "qwen":
            E, H, K, k = 128, 768, 2048, 8
        else:
            E, H, K = rng.randint(8, 128), 64 * rng.randint(4, 24), 64 * rng.randint(8, 48)
            k = rng.randint(1, min(8, E))
        return dict(kind=kind, fmt="nf4", E=E, H=H, K=K, top_k=k, tokens=rng.randint(1, 16),
                    skew=skew, layers=rng.randint(1, 4))
    if kind == "train":
        fmt = "nf4"
    else:
        fmt = {"qwen": "nf4", "gptoss": "mxfp4"}.get(model) or rng.choice(["nf4", "mxfp4"])
    if model == "qwen":
        E, k = 128, 8
        N, K = rng.choice([(1536, 2048), (2048, 768)])
    elif model == "gptoss" and fmt == "mxfp4":
        E, k = 32, 4
        N, K = rng.choice([(5760, 2880), (2880, 2880)])
    else:
        E = rng.randint(4, 128)
        k = rng.randint(1, min(8, E))
        # output widths that are multiples of 4 (any of them for the forward,
        # whole absmax blocks for a contraction over them)
        N = 64 * rng.randint(4, 48) if kind in ("dgrad", "train") else 4 * rng.randint(64, 768)
        K = 64 * rng.randint(4, 48)
    tokens = _log_int(rng, {"fwd": 1, "dgrad": 64, "train": 512}[kind], 4096)
    most = int(_MOST_FLOPS / (2.0 * N * K * k * (4 if kind == "train" else 1)))
    tokens = max(1, min(tokens, most))
    case = dict(kind=kind, fmt=fmt, E=E, N=N, K=K, top_k=k, tokens=tokens, skew=skew)
    if kind == "train":
        case["rank"] = rng.choice([8, 16, 32])
    else:
        case["ids"] = rng.choice(["host", "host", "device"])
        if kind == "fwd":
            case["act"] = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    return case


# ------------------------------------------------------------------ inputs --

# The two formats' codebooks (NF4: bitsandbytes' 16 normal quantiles; MXFP4:
# e2m1, index = sign << 3 | magnitude).
_NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
        -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
        0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
        0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]


def _bucket(x, table):
    """Index (into the ascending ``table``) of the entry nearest to each x."""
    t = torch.tensor(table, dtype=torch.float32, device=x.device)
    return torch.bucketize(x, (t[1:] + t[:-1]) / 2, out_int32=True).to(torch.uint8)


def _weights(fmt, E, N, K, gen):
    """A stack of N(0, 0.02) weights as a checkpoint of the format holds it:
    (packed [E, N, K/2] u8, absmax [E, N, K/64] f32 or e8m0 [E, N, K/32])."""
    dev = gen.device
    B = torch.empty(E, N, K // 2, dtype=torch.uint8, device=dev)
    S = torch.empty(E, N, K // (64 if fmt == "nf4" else 32), device=dev,
                    dtype=torch.float32 if fmt == "nf4" else torch.uint8)
    step = max(1, (1 << 26) // (N * K))
    for e in range(0, E, step):
        n = min(step, E - e)
        w = torch.randn(n, N, K, generator=gen, device=dev) * 0.02
        if fmt == "nf4":
            w = w.view(n, N, K // 64, 64)
            s = w.abs().amax(-1)
            c = _bucket(w / s.unsqueeze(-1), _NF4).view(n, N, K // 2, 2)
            B[e:e + n] = (c[..., 0] << 4) | c[..., 1]
            S[e:e + n] = s
        else:
            w = w.view(n, N, K // 32, 32)
            x = torch.ceil(torch.log2(w.abs().amax(-1) / 6.0))
            w = w / torch.exp2(x).unsqueeze(-1)
            c = _bucket(w.abs(), _E2M1[:8]) | ((w < 0).to(torch.uint8) << 3)
            c = c.view(n, N, K // 2, 2)
            B[e:e + n] = c[..., 0] | (c[..., 1] << 4)
            S[e:e + n] = (x + 127.0).to(torch.uint8)
    return B, S


def _decoded(fmt, B, S, e):
    """Expert e's weights [N, K] in float64."""
    N, half = B.shape[1], B.shape[2]
    b = B[e].to(torch.int64)
    hi, lo = b >> 4, b & 15
    t = torch.tensor(_NF4 if fmt == "nf4" else _E2M1, dtype=torch.float32, device=B.device)
    c = torch.stack((hi, lo) if fmt == "nf4" else (lo, hi), -1).view(N, half * 2)
    w = t.to(torch.float64)[c].view(N, S.shape[2], -1)
    s = S[e].to(torch.float64)
    return (w * (s if fmt == "nf4" else torch.exp2(s - 127.0)).unsqueeze(-1)).view(N, half * 2)


def _logits(case, rng, layers=1):
    """Router logits [layers, tokens, E] whose top-k is the case's routing:
    Gumbel noise over the experts' log popularity."""
    E = case["E"]
    pop = -case["skew"] * np.log(np.arange(1, E + 1))
    return np.stack([pop[rng.permutation(E)] + rng.gumbel(size=(case["tokens"], E))
                     for _ in range(layers)]).astype(np.float32)


def _groups(logits, k):
    """(sizes, ids) of the active experts, ascending, from logits [T, E]."""
    top = np.argsort(-logits, axis=1, kind="stable")[:, :k]
    count = np.bincount(top.reshape(-1), minlength=logits.shape[1])
    ids = np.nonzero(count)[0]
    return [int(count[e]) for e in ids], [int(e) for e in ids]


def _inputs(case, seed):
    """Every random input of a case, from the seed alone."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    randn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    d = {}
    if case["kind"] in ("step", "moe"):
        E, H, K, L = case["E"], case["H"], case["K"], case["layers"]
        lg = _logits(case, rng, L)
        gu = _weights(case["fmt"], E, 2 * H, K, gen)
        dn = _weights(case["fmt"], E, K, H, gen)
        d["layers"] = []
        for i in range(L):
            # a layer's own weights: the experts of the first, in turned order
            w = [gu, dn] if i == 0 else [tuple(t.roll(i, 0) for t in p) for p in (gu, dn)]
            sizes, ids = _groups(lg[i], case["top_k"])
            rows = case["tokens"] if case["kind"] == "moe" else sum(sizes)
            d["layers"].append(dict(gu=w[0], dn=w[1], sizes=sizes, ids=ids,
                                    x=randn(rows, K).to(torch.bfloat16),
                                    logits=torch.from_numpy(lg[i]).cuda()))
        return d
    E, N, K = case["E"], case["N"], case["K"]
    d["sizes"], d["ids"] = _groups(_logits(case, rng)[0], case["top_k"])
    T = sum(d["sizes"])
    d["B"], d["S"] = _weights(case["fmt"], E, N, K, gen)
    if case["kind"] == "dgrad":
        d["g"] = (randn(T, N) * 0.01).to(torch.bfloat16)
        return d
    d["x"] = randn(T, K).to(_DTYPES[case.get("act", "bf16")])
    if case["kind"] == "train":
        r = case["rank"]
        d["A"] = randn(E, r, K) / math.sqrt(K)
        d["Bl"] = randn(E, N, r) * 0.01
        d["g"] = (randn(T, N) * 0.01).to(torch.bfloat16)
    return d


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind in ("step", "moe"):
        if kind == "step":
            def once():
                return [nf4_ffn.gemm_nf4_ffn_grouped(l["x"], *l["gu"], *l["dn"], l["sizes"],
                                                     l["ids"]) for l in s["layers"]]
        else:
            def once():
                return [nf4_route.moe_layer(l["x"], l["logits"], case["top_k"], *l["gu"],
                                            *l["dn"], norm=True) for l in s["layers"]]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            once()
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = once()
        return s
    if case.get("ids") == "device":
        s["ids"] = torch.tensor(s["ids"], dtype=torch.int32, device="cuda")
    if kind == "train":
        for n in ("x", "A", "Bl"):
            s[n].requires_grad_(True)
    return s


def run(s):
    case = s["case"]
    kind, nf4 = case["kind"], case["fmt"] == "nf4"
    if kind in ("step", "moe"):
        s["graph"].replay()
        return s["out"]
    if kind == "fwd":
        op = nf4_grouped.gemm_4bit_grouped if nf4 else mxfp4_grouped.gemm_mxfp4_grouped
        return op(s["x"], s["B"], s["S"], s["sizes"], s["ids"])
    if kind == "dgrad":
        op = nf4_grouped.dgrad_4bit_grouped if nf4 else mxfp4_grouped.dgrad_mxfp4_grouped
        return op(s["g"], s["B"], s["S"], s["sizes"], s["ids"])
    out = nf4_qlora.fused_grouped_lora(s["x"], s["B"], s["S"], s["sizes"], s["ids"], s["A"],
                                       s["Bl"], scaling=2.0)
    return [out.detach(), *torch.autograd.grad(out, (s["x"], s["A"], s["Bl"]), s["g"])]


# ---------------------------------------------------------------- measures --

def _elem_bytes(fmt):
    """Bytes of one packed weight with its share of the block scale."""
    return 0.5 + (4 / 64 if fmt == "nf4" else 1 / 32)


def work(case):
    rng = np.random.default_rng(0)
    k, w = case["top_k"], _elem_bytes(case["fmt"])
    kind = case["kind"]
    if kind in ("step", "moe"):
        H, K, L = case["H"], case["K"], case["layers"]
        groups = [_groups(x, k) for x in _logits(case, rng, L)]
        T = case["tokens"] * k
        rows = case["tokens"] if kind == "moe" else T
        by = sum(len(ids) for _s, ids in groups) * 3 * H * K * w + L * rows * 2 * K * 2
        return {"bytes": by, "flops": L * 2.0 * T * 3 * H * K}
    N, K = case["N"], case["K"]
    sizes, ids = _groups(_logits(case, rng)[0], k)
    T, G = sum(sizes), len(ids)
    packed, flops = G * N * K * w, 2.0 * T * N * K
    if kind == "dgrad":
        return {"bytes": packed + T * (N + K) * 2, "flops": flops}
    if kind == "fwd":
        return {"bytes": packed + T * (K * (4 if case["act"] == "fp32" else 2) + N * 2),
                "flops": flops}
    r = case["rank"]
    lora = (K + N) * r
    # forward: x, weights, adapters, out; backward: the gradient, the weights
    # again, x and the adapters again, and the three gradients
    by = 2 * packed + T * (2 * N + 3 * K) * 2 + (2 * G + case["E"]) * lora * 4
    return {"bytes": by, "flops": 2 * flops + 6.0 * T * lora}


def tolerance(case):
    """bf16 outputs and bf16 operands: against float64 the paths measure 1.7e-3
    (one bf16 rounding of the output) to 2.9e-3 (bf16 weights too), a whole
    layer, whose intermediates are bf16 as well, up to 4.4e-3; the largest single
    difference is 6 standard deviations of that over millions of values."""
    return {"rel": 1e-2, "max": 8e-2}


def _by_group(fn, sizes, ids):
    out, row = [], 0
    for m, e in zip(sizes, ids):
        out.append(fn(e, slice(row, row + m)))
        row += m
    return torch.cat(out)


def exact(case, seed):
    d = _inputs(case, seed)
    f64 = lambda t: t.to(torch.float64)  # noqa: E731
    fmt, kind = case["fmt"], case["kind"]
    if kind in ("step", "moe"):
        H, outs = case["H"], []
        for l in d["layers"]:
            def ffn(e, x):
                gu = x @ _decoded(fmt, *l["gu"], e).T
                return (torch.nn.functional.silu(gu[:, :H]) * gu[:, H:]) @ _decoded(fmt, *l["dn"], e).T
            if kind == "step":
                x = f64(l["x"])
                outs.append(_by_group(lambda e, r: ffn(e, x[r]), l["sizes"], l["ids"]))
                continue
            w, ids = torch.softmax(f64(l["logits"]), -1).topk(case["top_k"], dim=-1)
            w = w / w.sum(-1, keepdim=True)
            y = torch.zeros(l["x"].shape, dtype=torch.float64, device="cuda")
            for e in ids.unique().tolist():
                t, j = (ids == e).nonzero(as_tuple=True)
                y.index_add_(0, t, ffn(e, f64(l["x"])[t]) * w[t, j].unsqueeze(-1))
            outs.append((y, ids, w))
        return outs
    B, S, sizes, ids = d["B"], d["S"], d["sizes"], d["ids"]
    if kind == "dgrad":
        return _by_group(lambda e, r: f64(d["g"][r]) @ _decoded(fmt, B, S, e), sizes, ids)
    x = f64(d["x"])
    if kind == "fwd":
        # fp16 and fp32 activations are rounded to bf16 first: the op's contract
        x = f64(d["x"].to(torch.bfloat16))
        return _by_group(lambda e, r: x[r] @ _decoded(fmt, B, S, e).T, sizes, ids)
    g, A, Bl, c = f64(d["g"]), f64(d["A"]), f64(d["Bl"]), 2.0
    out = _by_group(lambda e, r: x[r] @ _decoded(fmt, B, S, e).T + c * (x[r] @ A[e].T) @ Bl[e].T,
                    sizes, ids)
    gx = _by_group(lambda e, r: g[r] @ _decoded(fmt, B, S, e) + c * (g[r] @ Bl[e]) @ A[e],
                   sizes, ids)
    gA, gB, row = torch.zeros_like(A), torch.zeros_like(Bl), 0
    for m, e in zip(sizes, ids):
        r = slice(row, row + m)
        gA[e] = c * (g[r] @ Bl[e]).T @ x[r]
        gB[e] = c * g[r].T @ (x[r] @ A[e].T)
        row += m
    return [out, gx, gA, gB]
