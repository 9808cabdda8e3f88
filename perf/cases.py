"""Measured workloads of the routed-MoE path: what a server of GLM-style models has this framework do.

A case is one layer call (or one captured decode step) through a public entry point:

  layer   ops.moe_layer: router GEMM, sigmoid + bias top-k, permutation, EXL3 4-bit experts, combine
  apply   Exl3MoEMethod.apply, the vLLM quant-method call on router ids and weights (optionally one expert-parallel
          rank of a larger layer, through the layer's expert_map)
  step    a HIP graph holding the routed layers of one decode step, each layer with its own experts and router
  e4m3    ops.moe_forward_ids_e4m3: the trellis-sourced e4m3 numerics
  fp8     fp8.moe_forward_ids: block-scaled e4m3 experts with per-token e4m3 activations

Sizes: 288 experts, top-8, hidden 4096 and intermediate 1024 is one rank's shard at tensor-parallel 2; intermediate
512 and 256 are those at 4 and 8. Scales are calibrated so that a few percent of the gate values meet the SwiGLU
limit. exact() restates each path in float64 with plain torch.
"""
from __future__ import annotations

import importlib
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "glm-5.3-flash-dgx-spark-vllm-optimization_amd"))
mi355moe = importlib.import_module("mi355moe")
ops, synthetic, fp8 = mi355moe.ops, mi355moe.synthetic, mi355moe.fp8

LIMIT, SCALE = 10.0, 2.5
HAD = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name, kind, T, n=288, K=4096, N=1024, topk=8, **more):
    c = {"kind": kind, "T": T, "n": n, "K": K, "N": N, "topk": topk, **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one user, one token at a time: the smallest call, where launches and latency count
        _case("decode_t1", "layer", 1),
        # speculative verification of one stream: 1 + 7 rows
        _case("decode_t8", "layer", 8),
        # six verify rows on a tensor-parallel-8 shard, as vLLM hands them over (fp16 rows, 64-bit ids)
        _case("verify_t6_tp8", "apply", 6, N=256, dtype="fp16", ids64=True),
        # the captured decode step of a served model with skewed expert popularity
        _case("step_t8_zipf", "step", 8, layers=10),
        # 64 concurrent streams, one token each
        _case("batch_t64", "layer", 64),
        # a mixed batch: decode rows and the ragged end of a prompt
        _case("mixed_t333", "apply", 333),
        # an ordinary prompt chunk, odd length
        _case("chunk_t1791", "apply", 1791),
        # a long prompt chunk on an expert-parallel rank holding half of the experts, skewed routing
        _case("ep_t4289_zipf", "apply", 4289, n=144, n_global=288, zipf=True),
        # the largest prefill chunk, from the hidden states
        _case("prefill_t8192", "layer", 8192),
        # prefill with the e4m3 numerics
        _case("e4m3_t2048", "e4m3", 2048),
        # block-scaled e4m3 experts: decode of a few streams, and a prefill chunk
        _case("fp8_t12", "fp8", 12),
        _case("fp8_t2048", "fp8", 2048),
    ]


def draw(rng):
    def logint(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    N, K = rng.choice([256, 512, 1024, 1024]), rng.choice([2048, 4096, 4096])
    n, topk = rng.choice([96, 144, 288, 288]), rng.choice([4, 6, 8, 8])
    kind = rng.choice(["layer", "layer", "apply", "apply", "apply", "step", "e4m3", "fp8", "fp8"])
    d = dict(n=n, K=K, N=N, topk=topk)
    if kind == "layer":
        return _case(None, kind, logint(1, 8000), **d)
    if kind == "apply":
        d.update(dtype=rng.choice(["bf16", "fp16"]), ids64=rng.random() < 0.5, zipf=rng.random() < 0.5)
        if rng.random() < 0.3:
            d["n_global"] = 2 * n
        return _case(None, kind, logint(1, 4500), **d)
    if kind == "step":
        return _case(None, kind, logint(1, 64), layers=rng.randint(3, 10), **d)
    if kind == "e4m3":
        return _case(None, kind, logint(256, 4096), **d)
    d["n"] = min(n, 144) if N == 1024 and rng.random() < 0.5 else n
    return _case(None, kind, logint(1, 2048), **d)


# ---------------------------------------------------------------------------------------------- inputs


def _seeds(seed, k):
    return [int(seed) * 1000 + 7 * i + 1 for i in range(k)]


def _layer(c, seed):
    # every expert shares the layer's input rotation, as in the real checkpoints
    return synthetic.calibrated_layer(c["n"], c["K"], c["N"], seed=seed, uniform_suh=True)


def _picks(c, seed):
    """(ids [T, topk] over the layer's global experts, weights fp32) of one call."""
    E = c.get("n_global", c["n"])
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    score = torch.rand(c["T"], E, generator=g, device="cuda").clamp_min(1e-12).log().neg().log().neg()   # Gumbel
    if c.get("zipf"):
        rank = torch.randperm(E, generator=g, device="cuda").float()
        score = score - 1.2 * torch.log(rank + 1.0)
    ids = torch.topk(score, c["topk"], dim=1).indices
    w = torch.softmax(torch.randn(c["T"], c["topk"], generator=g, device="cuda"), -1) * SCALE
    return ids.to(torch.int64 if c.get("ids64") else torch.int32).contiguous(), w


def _expert_map(c):
    """An expert-parallel rank's map: the first half of the global experts is local."""
    if "n_global" not in c:
        return None
    m = torch.full((c["n_global"],), -1, dtype=torch.int64, device="cuda")
    m[:c["n"]] = torch.arange(c["n"], device="cuda")
    return m


def _dtype(c):
    return DTYPES[c.get("dtype", "bf16")]


def _inputs(c, seed):
    """Everything the case's inputs and weights consist of, from the seed alone."""
    s = _seeds(seed, 40)
    T, K, n = c["T"], c["K"], c["n"]
    if c["kind"] == "layer":
        w, b = synthetic.router(n, K, seed=s[1])
        return {"experts": _layer(c, s[0]), "x": synthetic.activations(T, K, seed=s[2]), "rw": w, "rb": b}
    if c["kind"] == "step":
        v = {"experts": [], "x": [], "rw": [], "rb": []}
        for i in range(c["layers"]):
            w, b = synthetic.zipf_router(n, K, seed=s[3 * i + 1], rank_seed=s[3 * i + 1] + 3)
            v["experts"].append(_layer(c, s[3 * i]))
            v["x"].append(synthetic.zipf_activations(T, K, seed=s[3 * i + 2]))
            v["rw"].append(w)
            v["rb"].append(b)
        return v
    ids, w = _picks(c, s[3])
    x = synthetic.activations(T, K, seed=s[2], dtype=_dtype(c))
    if c["kind"] == "fp8":
        return {"experts": synthetic.fp8_layer(n, K, c["N"], seed=s[0]), "x": x, "ids": ids, "w": w}
    return {"experts": _layer(c, s[0]), "x": x, "ids": ids, "w": w, "map": _expert_map(c)}


def prepare(case, seed):
    v = _inputs(case, seed)
    if case["kind"] == "apply":
        # the layer as vLLM holds it after loading: parameters on a module, the quant method beside it
        ex, method, layer = v["experts"], mi355moe.Exl3MoEMethod(topk=case["topk"]), torch.nn.Module()
        for name in ("w13_trellis", "w13_suh", "w13_svh", "w2_trellis", "w2_suh", "w2_svh"):
            layer.register_parameter(name, torch.nn.Parameter(getattr(ex, name), requires_grad=False))
        layer.expert_map = v["map"]
        method.process_weights_after_loading(layer)
        v["layer"], v["method"] = layer, method
    if case["kind"] == "step":
        T, K, k = case["T"], case["K"], case["topk"]
        v["out"] = [torch.empty(T, K, dtype=torch.bfloat16, device="cuda") for _ in v["x"]]
        v["picks"] = [(torch.empty(T, k, dtype=torch.int32, device="cuda"),
                       torch.empty(T, k, dtype=torch.float32, device="cuda")) for _ in v["x"]]

        def step():
            for i, ex in enumerate(v["experts"]):
                ops.moe_layer(ex, v["x"][i], router_w=v["rw"][i], topk=k, bias=v["rb"][i], routed_scale=SCALE,
                              limit=LIMIT, out=v["out"][i], picks_out=v["picks"][i])

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        v["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(v["graph"]):
            step()
    v["case"] = dict(case)
    return v


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "layer":
        return ops.moe_layer(state["experts"], state["x"], router_w=state["rw"], topk=c["topk"], bias=state["rb"],
                             routed_scale=SCALE, limit=LIMIT, return_picks=True)
    if kind == "step":
        state["graph"].replay()
        return [state["out"], state["picks"]]
    if kind == "apply":
        return state["method"].apply(state["layer"], state["x"], state["w"], state["ids"])
    if kind == "e4m3":
        return ops.moe_forward_ids_e4m3(state["experts"], state["x"], state["ids"], state["w"], limit=LIMIT)
    return fp8.moe_forward_ids(state["experts"], state["x"], state["ids"], state["w"], limit=LIMIT)


# ---------------------------------------------------------------------------------------------- work, tolerance


def _distinct(c):
    """Expected number of local experts that a call reads, and of pairs that it multiplies."""
    E, T, k = c.get("n_global", c["n"]), c["T"], c["topk"]
    share = c["n"] / E
    if not (c.get("zipf") or c["kind"] == "step"):
        return c["n"] * (1.0 - (1.0 - k / E) ** T), T * k * share
    g = torch.Generator().manual_seed(1)
    p = 1.0 / (torch.arange(E, dtype=torch.float64) + 1.0) ** 1.2
    ids = torch.multinomial(p.expand(min(T, 2048), E), k, replacement=False, generator=g)
    return float(ids.unique().numel()) * share, T * k * share


def work(case):
    T, K, N, n = case["T"], case["K"], case["N"], case["n"]
    d, pairs = _distinct(case)
    if case["kind"] == "fp8":
        expert = 3 * K * N + 4 * 3 * (K // 128) * (N // 128)
    else:
        expert = 3 * K * N // 2 + 2 * 3 * (K + N)
    size = torch.empty(0, dtype=_dtype(case)).element_size()
    b = d * expert + 2 * T * K * size
    f = pairs * 6.0 * K * N
    if case["kind"] in ("layer", "step"):
        b += n * K * 2 + n * 4 + T * case["topk"] * 8
        f += 2.0 * T * K * n
    else:
        b += T * case["topk"] * (4 + (8 if case.get("ids64") else 4))
    m = case.get("layers", 1)
    return {"bytes": m * b, "flops": m * f}


def tolerance(case):
    # Measured against exact(): 1.8e-3 with bf16 outputs (whose own rounding is 1.7e-3 of their 2-norm), 7e-4 with fp16
    # outputs (the fp16 inputs of the two products make most of it), 1.6e-3 to 3.6e-3 for block-scaled e4m3, where a
    # code next to a tie may round the other way. About four times that. Router ids are whole numbers of a fixed
    # definition and agree.
    if case["kind"] in ("e4m3", "fp8"):
        return {"rel": 1.2e-2 if case["kind"] == "fp8" else 8e-3, "max": 0.2}
    if case.get("dtype") == "fp16":
        return {"rel": 3e-3, "max": 0.03}
    return {"rel": 8e-3, "max": 0.05}


# ---------------------------------------------------------------------------------------------- float64


def _codebook():
    """The value of each of the 65,536 16-bit trellis states: the sum of the two fp16 halves, rounded to fp16."""
    s = torch.arange(65536, dtype=torch.int64)
    x = (((s * 0xCBAC1FED) & 0xFFFFFFFF) & 0x8FFF8FFF) ^ 0x3B603B60

    def half(v):
        return torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.float16).double()

    return (half(x & 0xFFFF) + half(x >> 16)).to(torch.float16).double()


def _unpack(trellis, book):
    """float64 [K, N] of a 4-bit trellis int16 [K/16, N/16, 64]."""
    kt, nt = trellis.shape[:2]
    u = trellis.to(torch.int64) & 0xFFFF
    w = u[..., 0::2] | (u[..., 1::2] << 16)                              # 32 words per tile
    pair = (torch.roll(w, 1, -1) & 0xFFFF) << 32 | w                     # the word before gives at most 12 bits
    shift = (28 - 4 * torch.arange(8, device=w.device))
    v = book[(pair[..., None] >> shift) & 0xFFFF].reshape(kt, nt, 256)
    p = torch.arange(256, device=w.device)
    word, j = p >> 3, p & 7
    row = 2 * (word & 3) + (j & 1) + 8 * ((j >> 1) & 1)
    col = (word >> 2) + 8 * (j >> 2)
    out = torch.empty(kt, nt, 16, 16, dtype=torch.float64, device=w.device)
    out[:, :, row, col] = v
    return out.permute(0, 2, 1, 3).reshape(kt * 16, nt * 16)


def _rotate(x, had):
    return (x.reshape(x.shape[0], -1, HAD) @ had).reshape(x.shape)


def _hadamard(device):
    i = torch.arange(HAD, device=device)
    bits = i[:, None] & i[None, :]
    odd = sum((bits >> b) & 1 for b in range(7)) & 1
    return (1.0 - 2.0 * odd.double()) / math.sqrt(HAD)


def _quant(v):
    """Per-row e4m3 values and scales: s = amax / 448 (1 if 0), q = e4m3(v / s)."""
    s = v.abs().amax(1, keepdim=True) / 448.0
    s = torch.where(s > 0, s, torch.ones_like(s))
    return (v / s).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn).double(), s


def _experts64(v, c, ids, w, x=None):
    """The routed output float64 [T, K] of x's rows for local expert ids (below 0: no expert)."""
    ex, x = v["experts"], (v["x"] if x is None else x).double()
    T, K, dev = x.shape[0], c["K"], x.device
    out = torch.zeros(T, K, dtype=torch.float64, device=dev)
    flat, wf = ids.reshape(-1).long(), w.reshape(-1).double()
    token = torch.arange(T, device=dev).repeat_interleave(ids.shape[1])
    order = torch.argsort(flat, stable=True)
    counts = torch.bincount(flat.clamp_min(-1) + 1, minlength=c["n"] + 1).tolist()
    block = c["kind"] == "fp8"
    e4m3 = c["kind"] == "e4m3"
    had, book = _hadamard(dev), _codebook().to(dev)
    if e4m3:
        book = book.float().to(torch.float8_e4m3fn).double()
    if block:
        xq = _quant(x)
    at = counts[0]
    for e in range(c["n"]):
        m = counts[e + 1]
        rows = order[at:at + m]
        at += m
        if not m:
            continue
        t = token[rows]
        if block:
            def weight(q, s):
                return q.view(torch.float8_e4m3fn).double() * s.double().repeat_interleave(HAD, 0).repeat_interleave(HAD, 1)
            z = (xq[0][t] @ weight(ex.w13[e], ex.w13_scale[e]).T) * xq[1][t]
            g, u = z[:, :c["N"]].clamp_max(LIMIT), z[:, c["N"]:].clamp(-LIMIT, LIMIT)
            q, s = _quant((torch.nn.functional.silu(g) * u).to(torch.float16).double())
            y = (q @ weight(ex.w2[e], ex.w2_scale[e]).T) * s
        else:
            h, s = _rotate(x[t] * ex.w13_suh[e, 0].double(), had), 1.0
            if e4m3:
                h, s = _quant(h)
            g = _rotate((h @ _unpack(ex.w13_trellis[e, 0], book)) * s, had) * ex.w13_svh[e, 0].double()
            u = _rotate((h @ _unpack(ex.w13_trellis[e, 1], book)) * s, had) * ex.w13_svh[e, 1].double()
            # (the limit is met before or after SiLU by call size and numerics: 5e-5 apart on a value that meets it)
            a = torch.nn.functional.silu(g.clamp_max(LIMIT)) * u.clamp(-LIMIT, LIMIT)
            if e4m3:
                a = a.to(torch.float16).double()
            h, s = _rotate(a * ex.w2_suh[e].double(), had), 1.0
            if e4m3:
                h, s = _quant(h)
            y = _rotate((h @ _unpack(ex.w2_trellis[e], book)) * s, had) * ex.w2_svh[e].double()
        out.index_add_(0, t, y * wf[rows, None])
    return out


def _route64(x, rw, rb, topk):
    logits = (x.double() @ rw.double().T).to(torch.bfloat16)
    score = torch.sigmoid(logits.double())
    order = torch.sort(score.float() + rb, dim=1, descending=True, stable=True).indices[:, :topk]
    w = torch.gather(score, 1, order)
    return order, w / w.sum(1, keepdim=True) * SCALE


def exact(case, seed):
    v = _inputs(case, seed)
    if case["kind"] == "layer":
        ids, w = _route64(v["x"], v["rw"], v["rb"], case["topk"])
        return _experts64(v, case, ids, w), None, w
    if case["kind"] == "step":
        outs, picks = [], []
        for i, ex in enumerate(v["experts"]):
            ids, w = _route64(v["x"][i], v["rw"][i], v["rb"][i], case["topk"])
            outs.append(_experts64({"experts": ex}, case, ids, w, x=v["x"][i]))
            picks.append((None, w))
        return [outs, picks]
    ids = v["ids"] if v.get("map") is None else v["map"][v["ids"].long()]
    return _experts64(v, case, ids, v["w"])
