"""Performance cases of the FP4 MoE expert path: what a serving program has the framework do, from one decoded token to
a long prefill, through the public entry points of dsv41_amd.

A case is a dict of plain values; `kind` names the path:
  moe      moe.MoE.__call__: one MoE layer (router, gate, shared expert, routed experts) on `tokens` rows, `layers` layers one
           after another (one layer's selected experts would stay in the last-level cache between passes at one token; a
           model's layers do not). `graph`: the calls replayed from one captured graph, as a decode loop runs them.
  experts  moe.prefill_experts: the routed experts alone, given Zipf routing (popular experts beside rarely used ones).
  linear   w8.linear_w: FP8 dense weights on `rows` activation rows; n = 0 stands for the five projections of a layer
           (DENSE), otherwise one n x k weight.
  grouped  moe_kernels.GroupedPairs + grouped_fp4_gemm: the expert math of a prefill chunk, called op by op.
  gemm_tc  hipkern.moe_dispatch + fp4_gemm_tc: the expert math of a decode batch, called op by op.
  hc       fused2.hc_pre_norm_quant2 + hc_post2_: the hyper-connection steps either side of a layer's experts.

exact() evaluates a case with plain torch in 64 bits: the roundings that the path defines (FP8 and bf16 intermediates) are
applied where it defines them, every product and sum in between is float64.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "deepseekv4.1-a100-custom_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dsv41_amd import fused, fused2, hipkern, moe, moe_kernels, quant, w8  # noqa: E402

LIMIT = 10.0                                                     # swiglu clamp of the model
DENSE = ((5120, 8192), (4608, 5120), (32768, 1280), (1280, 5120), (5120, 2304))   # (n, k) of a layer's FP8 projections
# (hidden, intermediate, experts, top-k, gate): the benchmark's layer, the reference model's, a smaller generic one
SHAPES = ((7168, 1664, 384, 8, "softmax"), (5120, 2304, 384, 6, "sqrtsoftplus"), (4096, 2048, 128, 8, "sigmoid"))
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _moe(name, tokens, shape, layers=1, graph=False, shared="fp8"):
    H, I, E, k, score = SHAPES[shape]
    c = {"kind": "moe", "tokens": tokens, "hidden": H, "inter": I, "experts": E, "topk": k, "score": score, "layers": layers,
         "graph": graph, "shared": shared}
    return dict(c, name=name) if name else c


def _sized(kind, name, tokens, shape):
    H, I, E, k, _ = SHAPES[shape]
    c = {"kind": kind, "tokens": tokens, "hidden": H, "inter": I, "experts": E, "topk": k}
    return dict(c, name=name) if name else c


def _linear(name, rows, n=0, k=0, graph=False):
    c = {"kind": "linear", "rows": rows, "n": n, "k": k, "graph": graph}
    return dict(c, name=name) if name else c


def listed():
    return [
        _moe("decode 1 token", 1, 0, layers=4, graph=True),                # one stream decoding
        _moe("decode 16 tokens", 16, 0, graph=True, shared="bf16"),        # speculative verification / a small batch
        _moe("batch 48 tokens", 48, 1),                                    # a decode batch beyond the fused decode launches
        _moe("chunk 333 tokens", 333, 0),                                  # a short prompt, or a chunk of a long one
        _moe("prefill 2048 tokens", 2048, 0),                              # a whole prompt through one layer
        _sized("experts", "experts 8192 tokens, Zipf", 8192, 0),           # a long prefill with skewed routing
        _linear("dense FP8 1 row", 1, graph=True),                         # the projections of a layer, one token
        _linear("dense FP8 48 rows", 48, graph=True),                      # and for a decode batch
        _linear("dense FP8 700 rows", 700),                                # and for a prompt
        _sized("grouped", "grouped_fp4_gemm 512 tokens", 512, 0),          # a caller of the op-by-op prefill surface
        _sized("gemm_tc", "fp4_gemm_tc 24 tokens", 24, 1),                 # a caller of the op-by-op decode surface
        {"kind": "hc", "name": "hyper-connections 1500 rows", "rows": 1500, "hidden": 5120},   # the steps around a prompt's experts
    ]


def _log(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(("moe", "moe", "moe", "experts", "linear", "linear", "grouped", "gemm_tc", "hc"))
    shape = rng.randrange(len(SHAPES))
    if kind == "moe":
        t = _log(rng, 1, 2048)
        return _moe("", t, shape, layers=4 if t <= 2 else 1, graph=t <= 16 and rng.random() < 0.75, shared=rng.choice(("fp8", "bf16")))
    if kind == "experts":
        return _sized(kind, "", _log(rng, 17, 8000), shape)
    if kind == "linear":
        rows = _log(rng, 1, 1000)
        graph = rows <= 64 and rng.random() < 0.75
        if rng.random() < 0.5:
            return _linear("", rows, graph=graph)
        return _linear("", rows, 8 * _log(rng, 64, 4096), 64 * _log(rng, 12, 128), graph)
    if kind == "grouped":
        return _sized(kind, "", _log(rng, 9, 1024), shape)
    if kind == "gemm_tc":
        return _sized(kind, "", _log(rng, 2, 64), shape)
    return {"kind": "hc", "rows": _log(rng, 1, 4096), "hidden": rng.choice((4096, 5120, 7168))}


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _bytes(g, *shape):
    """Uniform random bytes (two E2M1 codes each)."""
    n = math.prod(shape)
    return torch.randint(-(2 ** 63), 2 ** 63 - 1, ((n + 7) // 8,), generator=g, device="cuda", dtype=torch.int64).view(torch.uint8)[:n].view(*shape)


def _scales(g, *shape):
    """E8M0 bytes 119 .. 123, four of them from each random word."""
    n = math.prod(shape)
    r = torch.randint(0, 5 ** 4, ((n + 3) // 4,), generator=g, device="cuda", dtype=torch.int16)
    out = torch.empty(r.numel(), 4, device="cuda", dtype=torch.uint8)
    for i in range(4):
        out[:, i] = (r % 5 + 119).to(torch.uint8)
        r = r // 5
    return out.view(-1)[:n].view(*shape)


def _experts(g, c):
    E, H, I = c["experts"], c["hidden"], c["inter"]
    return moe.ExpertWeights(_bytes(g, E, 2 * I, H // 2), _scales(g, E, 2 * I, H // 32), _bytes(g, E, H, I // 2), _scales(g, E, H, I // 32),
                             tiled=True)


def _fp8_weights(g, n, k):
    """E4M3 bytes [n, k] of N(0, 1) values and the E8M0 scales of a k-long dot product."""
    w = torch.randn(n, k, generator=g, device="cuda").clamp_(-400, 400).to(torch.float8_e4m3fn).view(torch.uint8)
    s = torch.randint(119, 124, ((n + 31) // 32, k // 32), generator=g, device="cuda", dtype=torch.uint8)
    return w, s


def _zipf(g, tokens, experts, topk):
    """topk distinct experts per token by Zipf(1.1) popularity (Gumbel draws of the log popularity), softmax weights."""
    pop = -1.1 * torch.log(torch.arange(1, experts + 1, device="cuda", dtype=torch.float32))
    pop = pop[torch.randperm(experts, generator=g, device="cuda")]
    u = torch.rand(tokens, experts, generator=g, device="cuda").clamp_(1e-7, 1 - 1e-7)
    eid = torch.topk(pop - torch.log(-torch.log(u)), topk, dim=-1).indices.to(torch.int32)
    wt = torch.softmax(torch.randn(tokens, topk, generator=g, device="cuda"), -1)
    return eid.contiguous(), wt.contiguous()


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)


def _layer_inputs(c, g):
    """The tensors of one MoE layer: experts, router, shared expert, activations."""
    H, I, E = c["hidden"], c["inter"], c["experts"]
    d = {"ex": _experts(g, c), "gate_w": torch.randn(E, H, generator=g, device="cuda") / math.sqrt(H), "x": _randn(g, c["tokens"], H)}
    d["bias"] = 0.1 * torch.randn(E, generator=g, device="cuda") if c["score"] != "softmax" else None
    if c["shared"] == "fp8":
        d["s13"], d["s2"] = _fp8_weights(g, 2 * I, H), _fp8_weights(g, H, I)
    else:
        d["s13"], d["s2"] = _randn(g, 2 * I, H) / math.sqrt(H), _randn(g, H, I) / math.sqrt(I)
    return d


def _graph(call):
    """One captured pass of `call` (after a warm-up pass, as a decode loop does it) and its output buffers."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


def _dims(c):
    return DENSE if c["n"] == 0 else ((c["n"], c["k"]),)


def prepare(case, seed):
    c, g = case, _gen(seed)
    state = {"kind": c["kind"], "case": c}
    if c["kind"] == "moe":
        layers, xs = [], []
        for _ in range(c["layers"]):
            d = _layer_inputs(c, g)
            sh = (w8.W8(*d["s13"]), w8.W8(*d["s2"])) if c["shared"] == "fp8" else (d["s13"], d["s2"])
            layers.append(moe.MoE(d["ex"], d["gate_w"], d["bias"], topk=c["topk"], score_func=c["score"], route_scale=1.0,
                                  norm_topk_prob=True, swiglu_limit=LIMIT, sh_w13=sh[0], sh_w2=sh[1]))
            xs.append(d["x"])
        state["layers"], state["x"] = layers, xs
    elif c["kind"] == "experts":
        state["ex"] = _experts(g, c)
        state["xq"] = quant.fake_quant_fp8(_randn(g, c["tokens"], c["hidden"]))
        state["eid"], state["wt"] = _zipf(g, c["tokens"], c["experts"], c["topk"])
        state["out"] = torch.empty(c["tokens"], c["hidden"], dtype=torch.bfloat16, device="cuda")
    elif c["kind"] == "linear":
        state["w"] = [w8.W8(*_fp8_weights(g, n, k)) for n, k in _dims(c)]
        state["x"] = [_randn(g, c["rows"], k) for _, k in _dims(c)]
    elif c["kind"] in ("grouped", "gemm_tc"):
        T, k = c["tokens"], c["topk"]
        state["ex"] = _experts(g, c)
        state["xq"] = quant.fake_quant_fp8(_randn(g, T, c["hidden"]))
        state["eid"], state["wt"] = _zipf(g, T, c["experts"], k)
        state["tok"] = torch.arange(T, device="cuda", dtype=torch.int32).repeat_interleave(k)
        state["rows"] = torch.arange(T * k, device="cuda", dtype=torch.int32)
        state["ones"] = torch.ones(T * k, device="cuda")
    else:
        B, d = c["rows"], c["hidden"]
        state["x"] = _randn(g, B, 1, 4, d)
        state["pre"] = torch.softmax(torch.randn(B, 4, generator=g, device="cuda"), -1)
        state["post"] = torch.rand(B, 4, generator=g, device="cuda")
        # each new stream mixes the four old ones; below 1 in all, so that a state that is passed over again stays bounded
        state["comb"] = 0.9 * torch.softmax(torch.randn(B, 4, 4, generator=g, device="cuda"), 1)
        state["w"] = (1 + 0.1 * torch.randn(d, generator=g, device="cuda")).to(torch.bfloat16)
        state["y"] = _randn(g, B, d)                     # the layer's output between the two steps
    if c.get("graph"):
        state["graph"], state["out"] = _graph(lambda: _pass(state))
    return state


# --------------------------------------------------------------------------- one pass
def _pass(s):
    c = s["case"]
    if c["kind"] == "moe":
        out = []
        for layer, x in zip(s["layers"], s["x"]):
            y = layer(x)
            out.append((y, *layer.last_routing))
        return out
    if c["kind"] == "experts":
        return moe.prefill_experts(s["xq"], s["eid"], s["wt"], s["ex"], LIMIT, out=s["out"])
    if c["kind"] == "linear":
        return [w8.linear_w(x, w) for x, w in zip(s["x"], s["w"])]
    if c["kind"] == "grouped":
        P, ex = c["tokens"] * c["topk"], s["ex"]
        eid, wt = s["eid"].reshape(-1), s["wt"].reshape(-1)
        pairs = moe_kernels.GroupedPairs(eid, s["tok"], s["rows"], s["ones"], 64, n_experts=c["experts"])
        gu = moe_kernels.grouped_fp4_gemm(s["xq"], ex.w13, ex.s13, pairs, P, tiled=True)
        h = fused.swiglu_quant(gu, wt, c["inter"], LIMIT)
        pairs = moe_kernels.GroupedPairs(eid, s["rows"], s["rows"], s["ones"], 64, n_experts=c["experts"])
        y = moe_kernels.grouped_fp4_gemm(h, ex.w2, ex.s2, pairs, P, tiled=True)
        return y.view(c["tokens"], c["topk"], -1).sum(1)
    if c["kind"] == "gemm_tc":
        P, ex, E = c["tokens"] * c["topk"], s["ex"], c["experts"]
        most = min(c["tokens"], hipkern.FP4_W_MAX)
        tok, wt, inv, ge, gs = hipkern.moe_dispatch(s["eid"], s["wt"], c["topk"], E, most, s["xq"].device)
        gu = hipkern.fp4_gemm_tc(hipkern.permute_x(s["xq"]), ex.w13, ex.s13, ge, gs, tok, P, most)
        h = fused.swiglu_quant(gu, wt, c["inter"], LIMIT, permute=True)
        y = hipkern.fp4_gemm_tc(h, ex.w2, ex.s2, ge, gs, s["rows"], P, most)
        return y[inv.long()].view(c["tokens"], c["topk"], -1).sum(1)
    y, yq, _ = fused2.hc_pre_norm_quant2(s["x"], s["pre"], s["w"], 1e-6)
    return y, yq, fused2.hc_post2_(s["y"], s["x"], s["post"], s["comb"])


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _pass(state)


# --------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    c = case
    if c["kind"] == "linear":
        M, dims = c["rows"], _dims(c)
        return {"bytes": sum(n * k + ((n + 31) // 32) * (k // 32) + 2 * M * (n + k) for n, k in dims),
                "flops": sum(2 * M * n * k for n, k in dims)}
    if c["kind"] == "hc":
        B, d = c["rows"], c["hidden"]
        # the four streams read and written once, the layer's output read, y and yq written
        return {"bytes": B * d * 2 * (4 + 4 + 1 + 2), "flops": B * d * 60}
    T, H, I, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["topk"]
    per = (3 * H * I) // 2 + (3 * H * I) // 32
    if c["kind"] == "moe":
        touched = E * (1 - (1 - k / E) ** T)                      # experts that some token picks, uniform routing
    else:
        pop = [(r + 1) ** -1.1 for r in range(E)]
        tot = sum(pop)
        touched = sum(1 - (1 - min(1.0, k * p / tot)) ** T for p in pop)
    b, f = touched * per + T * H * 4, T * k * 6 * H * I
    if c["kind"] == "moe":
        b += E * H * 4 + 3 * H * I * (1 if c["shared"] == "fp8" else 2)
        f += T * (6 * H * I + 2 * H * E)
    n = c.get("layers", 1)
    return {"bytes": n * b, "flops": n * f}


def tolerance(case):
    kind = case["kind"]
    if kind == "moe":
        # bf16 outputs; a rounding that falls the other way inside (an FP8 code of h) reaches a whole output row, a near
        # tie of the router another expert
        return {"rel": 1e-2, "differ": 2e-3}
    # bf16 outputs are 1.7e-3 off 64 bits; in the fp32 outputs of the op-by-op calls FP8 codes of h that fall the other way
    # show up to 1.3e-3 (few tokens)
    return {"rel": 5e-3}


# --------------------------------------------------------------------------- 64-bit results
def _d(b):
    """E8M0 bytes -> 2^(b - 127)."""
    return torch.pow(2.0, b.to(torch.float64) - 127)


def _bf16(v):
    return v.to(torch.bfloat16).to(torch.float64)


def _fq8(v):
    """Per-32 FP8 fake quantisation (power-of-two scale of the amax over 448, E4M3 to nearest even) of bf16-valued v."""
    b = v.reshape(*v.shape[:-1], -1, 32)
    m, e = torch.frexp(b.abs().amax(-1, keepdim=True).clamp_min(1e-4) / 448.0)
    s = torch.ldexp(torch.ones_like(m), torch.where(m == 0.5, e - 1, e))
    return ((b / s).to(torch.float32).to(torch.float8_e4m3fn).to(torch.float64) * s).reshape(v.shape)


def _expert(w, s):
    """One expert's matrix [N, K] from its tiled packed bytes [N, K / 2] and tiled scales [N, K / 32]."""
    N, Kh = w.shape
    w = w.view(N // 16, Kh // 64, 16, 64).permute(0, 2, 1, 3).reshape(N, Kh)
    s = s.view(N // 16, Kh // 64, 16, 4).permute(0, 2, 1, 3).reshape(N, Kh // 16)
    table = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=w.device)
    v = table[torch.stack((w & 15, w >> 4), -1).long()].reshape(N, Kh // 16, 32)
    return (v * _d(s).unsqueeze(-1)).reshape(N, 2 * Kh)


def _dense(w, s):
    n, k = w.shape
    v = w.view(torch.float8_e4m3fn).to(torch.float64)
    return v * _d(s).repeat_interleave(32, 0)[:n].repeat_interleave(32, 1)


def _swiglu(gu, inter, wt=None):
    g, u = gu[:, :inter].clamp_max(LIMIT), gu[:, inter:].clamp(-LIMIT, LIMIT)
    h = g * torch.sigmoid(g) * u
    return _fq8(_bf16(h if wt is None else h * wt[:, None]))


def _routed(ex, xq, eid, wt, inter):
    """[T, H] sum of the picked experts, one expert at a time."""
    y = torch.zeros(xq.shape[0], ex.H, dtype=torch.float64, device=xq.device)
    for e in torch.unique(eid).tolist():
        t, j = torch.where(eid == e)
        h = _swiglu(xq[t] @ _expert(ex.w13[e], ex.s13[e]).t(), inter, wt[t, j].double())
        y.index_add_(0, t, h @ _expert(ex.w2[e], ex.s2[e]).t())
    return y


def _gate(c, d, x):
    s = x @ d["gate_w"].double().t()
    if c["score"] == "softmax":
        s = torch.softmax(s, -1)
    elif c["score"] == "sigmoid":
        s = torch.sigmoid(s)
    else:
        s = torch.sqrt(torch.nn.functional.softplus(s))
    eid = torch.topk(s if d["bias"] is None else s + d["bias"].double(), c["topk"], dim=-1).indices
    w = s.gather(-1, eid)
    return eid, w / (w.sum(-1, keepdim=True) + 1e-20)


def exact(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "moe":
        out = []
        for _ in range(c["layers"]):
            d = _layer_inputs(c, g)
            x = d["x"].double()
            eid, wt = _gate(c, d, x)
            xq = _fq8(x)
            y = _routed(d["ex"], xq, eid, wt, c["inter"])
            s13, s2 = (_dense(*d["s13"]), _dense(*d["s2"])) if c["shared"] == "fp8" else (d["s13"].double(), d["s2"].double())
            ys = _bf16(_swiglu(_bf16(xq @ s13.t()), c["inter"]) @ s2.t())
            out.append((y + ys, eid.to(torch.int32), wt))
        return out
    if c["kind"] in ("experts", "grouped", "gemm_tc"):
        ex = _experts(g, c)
        xq = _fq8(_randn(g, c["tokens"], c["hidden"]).double())
        eid, wt = _zipf(g, c["tokens"], c["experts"], c["topk"])
        return _routed(ex, xq, eid, wt, c["inter"])
    if c["kind"] == "linear":
        w = [_dense(*_fp8_weights(g, n, k)) for n, k in _dims(c)]
        x = [_randn(g, c["rows"], k).double() for _, k in _dims(c)]
        return [a @ b.t() for a, b in zip(x, w)]
    s = prepare(case, seed)
    x, pre, w = s["x"].double()[:, 0], s["pre"].double(), s["w"].double()
    a = _bf16(torch.einsum("bh,bhd->bd", pre, x))
    y = a * torch.rsqrt(a.square().mean(-1, keepdim=True) + 1e-6) * w
    post, comb, o = s["post"].double(), s["comb"].double(), s["y"].double()
    r = post[:, :, None] * o[:, None] + torch.einsum("bji,bjd->bid", comb, x)
    return y, _fq8(_bf16(y)), r[:, None]
