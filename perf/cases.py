"""Performance cases of the S14 expert path: what a program calls, at the
sizes it calls it with.

Six kinds of call, each through the public Python entry points:

  chain    one MXFP4 expert, one token (s14.expert_chain)
  matvec   one quantised matrix, one token (S14NumericPipelines bind + cmd)
  layer    router + top-6 routed + shared experts, one token
  block    the same for a speculative-verify block of 2 to 8 tokens
  prefill  the same for a prompt of up to 1,024 tokens
  linear   activation quant + FP8 projection (s14.act_quant_e4m3, s14.fp8_linear)

Hidden size 4,096, expert width 2,048, 256 experts, and the projections'
[n, k] are the model configuration the package fixes.  Pages hold uniform
E2M1 codes with UE8M0 scale exponents in [-10, -4], the shared FP8 page and
the projections normal E4M3 weights; activations are N(0, 1), adjacent block
tokens correlated, prefill routes Zipf(1.1)-popular.  Every input is drawn on
the GPU from the seed.
"""

from __future__ import annotations

import functools
import math

import torch

from colormlm_amd import _native as N
from colormlm_amd import s14, synth

H, I, E, K = synth.HIDDEN, synth.INTER, synth.N_EXPERTS, 6
MODES = {"exact": s14.EXACT, "fast": s14.FAST, "official": s14.OFFICIAL}
MX, F8 = synth.page_offsets("mxfp4"), synth.page_offsets("fp8")

# the FP8 projections beside the expert layer, [n, k]
PROJECTIONS = {"wq_b": (32768, 1024), "wkv": (512, 4096), "wo_a": (8192, 4096), "wo_b": (4096, 8192)}


def listed():
    return [
        # decode, the smallest call: one routed expert of one token
        {"name": "chain_exact", "kind": "chain", "mode": "exact"},
        # decode, the query down-projection of one token, f32 tile scales
        {"name": "matvec_wq_a", "kind": "matvec", "format": "fp8", "n": 1024, "k": 4096, "mode": "exact"},
        # decode, one token through the whole layer: the headline call
        {"name": "layer_exact", "kind": "layer", "router": "sigmoid", "shared": "mxfp4", "mode": "exact"},
        # the same where throughput is wanted and the sums' order is free
        {"name": "layer_fast", "kind": "layer", "router": "sigmoid", "shared": "mxfp4", "mode": "fast"},
        # decode with the model's own semantics, router and FP8 shared page
        {"name": "layer_official", "kind": "layer", "router": "softplus", "shared": "fp8", "mode": "official"},
        # speculative verify, a full block
        {"name": "block8_exact", "kind": "block", "tokens": 8, "router": "sigmoid", "shared": "mxfp4", "mode": "exact"},
        # speculative verify, a shorter odd block with the model's semantics
        {"name": "block5_official", "kind": "block", "tokens": 5, "router": "softplus", "shared": "mxfp4",
         "mode": "official"},
        # an ordinary prompt
        {"name": "prefill_512", "kind": "prefill", "tokens": 512, "mode": "exact"},
        # the longest prompt of one call, the model's semantics
        {"name": "prefill_1024_official", "kind": "prefill", "tokens": 1024, "mode": "official"},
        # a projection of one decoded token
        {"name": "linear_wq_b_1", "kind": "linear", "m": 1, "n": 32768, "k": 1024, "scale": "ue8m0", "bf16": False,
         "mode": "exact"},
        # a projection of an odd-sized prompt, bf16 output as the model takes it
        {"name": "linear_wo_a_333", "kind": "linear", "m": 333, "n": 8192, "k": 4096, "scale": "ue8m0", "bf16": True,
         "mode": "exact"},
        # a projection of an ordinary prompt, the sums' order free
        {"name": "linear_wo_b_512_fast", "kind": "linear", "m": 512, "n": 4096, "k": 8192, "scale": "ue8m0",
         "bf16": False, "mode": "fast"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chain", "matvec", "layer", "layer", "block", "block", "prefill", "prefill", "linear", "linear",
                       "linear"])
    if kind == "chain":
        # route weights as the router gives them
        return {"kind": kind, "mode": rng.choice(list(MODES)), "route_w": round(rng.uniform(0.05, 0.4), 4)}
    if kind == "matvec":
        fmt = rng.choice(["mxfp4", "fp8"])
        k = 1024 * rng.randint(1, 4)
        return {"kind": kind, "format": fmt, "n": _log_int(rng, 500, 8192), "k": k, "mode": rng.choice(["exact", "fast"])}
    if kind == "layer":
        return {"kind": kind, "router": rng.choice(["sigmoid", "softplus", "hash"]),
                "shared": rng.choice(["mxfp4", "mxfp4", "fp8"]), "mode": rng.choice(list(MODES)),
                "bank": rng.randint(0, 1 << 20)}
    if kind == "block":
        return {"kind": kind, "tokens": rng.randint(2, 8), "router": rng.choice(["sigmoid", "softplus"]),
                "shared": rng.choice(["mxfp4", "mxfp4", "fp8"]), "mode": rng.choice(list(MODES)),
                "bank": rng.randint(0, 1 << 20)}
    if kind == "prefill":
        return {"kind": kind, "tokens": _log_int(rng, 9, 1000), "mode": rng.choice(["exact", "official"])}
    n, k = rng.choice(list(PROJECTIONS.values()) + [(_log_int(rng, 300, 8192), 128 * rng.randint(3, 32))])
    return {"kind": kind, "m": _log_int(rng, 1, 300), "n": n, "k": k, "scale": rng.choice(["ue8m0", "ue8m0", "f32"]),
            "bf16": rng.random() < 0.5, "mode": rng.choice(["exact", "fast"])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


@functools.lru_cache(maxsize=1)
def _context():
    return s14.Context(0)  # a program keeps one


def _gen(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + int(case.get("bank", 0)) * 7 + 11)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _bytes(g, lo, hi, *shape):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)


def _e4m3(v):
    return v.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)


def _mx_pages(g, n):
    words = torch.randint(-(1 << 31), 1 << 31, (n, MX["total"] // 4), generator=g, device="cuda", dtype=torch.int32)
    pages = words.view(torch.uint8)
    for s, end in (("s1", "w3"), ("s3", "w2"), ("s2", "total")):
        pages[:, MX[s]:MX[end]] = _bytes(g, 117, 124, n, MX[end] - MX[s])
    return pages


def _fp8_page(g):
    page = torch.empty(F8["total"], dtype=torch.uint8, device="cuda")
    for w, s, end in (("w1", "s1", "w3"), ("w3", "s3", "w2"), ("w2", "s2", "total")):
        page[F8[w]:F8[s]] = _e4m3(_randn(g, F8[s] - F8[w]))
        page[F8[s]:F8[end]] = _bytes(g, 120, 123, F8[end] - F8[s])
    return page


def _zipf_bias(g, weight):
    """Router biases that give the experts Zipf(1.1) popularity: each is nudged
    by the log ratio of its wanted and seen share over calibration tokens."""
    target = torch.from_numpy(synth.zipf_top6_inclusion(1.1)).to("cuda", torch.float32)
    target = target[torch.randperm(E, generator=g, device="cuda")]
    scores = torch.sigmoid(_randn(g, 4096, H) @ weight.T)
    bias = 0.05 * target.log()
    for _ in range(150):
        top = (scores + bias).topk(K, dim=1).indices
        seen = torch.bincount(top.flatten(), minlength=E).float() / scores.shape[0]
        bias = bias + 0.025 * ((target + 1e-4).log() - (seen + 1e-4).log())
    return bias


def _inputs(case, seed):
    """The case's inputs as tensors; exact() makes the same ones again."""
    g = _gen(case, seed)
    kind = case["kind"]
    if kind == "chain":
        return {"page": _mx_pages(g, 1)[0], "x": _randn(g, H)}
    if kind == "matvec":
        n, k = case["n"], case["k"]
        if case["format"] == "mxfp4":
            return {"w": _bytes(g, 0, 256, n, k // 2), "s": _bytes(g, 117, 124, n, k // 32), "x": _randn(g, k)}
        tiles = (-(-n // 128), -(-k // 128))
        s = torch.exp2(torch.rand(tiles, generator=g, device="cuda") * 6.0 - 6.0)
        return {"w": _e4m3(0.02 * _randn(g, n, k)), "s": s, "x": _randn(g, k).bfloat16()}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        tiles = (-(-n // 128), -(-k // 128))
        if case["scale"] == "f32":
            s = torch.exp2(torch.rand(tiles, generator=g, device="cuda") * 3.0 - 8.0)
        else:
            s = _bytes(g, 119, 122, *tiles)
        return {"w": _e4m3(_randn(g, n, k)), "s": s, "x": _randn(g, m, k)}
    tokens = case.get("tokens", 1)
    weight = 0.02 * _randn(g, E, H)
    t = {"pages": _mx_pages(g, E), "weight": weight, "tid2eid": None, "token_ids": None}
    t["bias"] = _zipf_bias(g, weight) if kind == "prefill" else 0.01 * _randn(g, E)
    t["shared"] = _fp8_page(g) if case.get("shared") == "fp8" else _mx_pages(g, 1)[0]
    x = _randn(g, tokens, H)
    if kind == "block":  # adjacent tokens share some of their experts
        a = synth.BLOCK_CORRELATION
        for i in range(1, tokens):
            x[i] = a * x[i - 1] + math.sqrt(1.0 - a * a) * x[i]
    t["x"] = x
    if case.get("router") == "hash":
        vocab = 1024
        t["tid2eid"] = torch.rand(vocab, E, generator=g, device="cuda").topk(K, dim=1).indices.contiguous()
        t["token_ids"] = torch.randint(0, vocab, (tokens,), generator=g, device="cuda", dtype=torch.int32)
    return t


def _softplus(case):
    return case.get("router") in ("softplus", "hash")


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    st = {"case": case, "ctx": _context(), "mode": MODES[case["mode"]], **t}
    if kind == "chain":
        st["y"] = torch.empty(H, device="cuda")
    elif kind == "matvec":
        pipes = s14.S14NumericPipelines(st["ctx"])
        shape = s14.S14MatvecShape.new(case["n"], case["k"])
        st["y"] = torch.empty(case["n"], device="cuda")
        bind = pipes.bind_mxfp4 if case["format"] == "mxfp4" else pipes.bind_fp8
        st["dispatch"] = bind(shape, t["x"], t["w"], t["s"], st["y"], mode=st["mode"])
        st["cmd"] = pipes.cmd_mxfp4_matvec if case["format"] == "mxfp4" else pipes.cmd_fp8_matvec
    elif kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        st["q"] = torch.empty((m, k), dtype=torch.uint8, device="cuda")
        st["qs"] = torch.empty((m, k // 128), dtype=torch.uint8, device="cuda")
        st["y"] = torch.empty((m, n), device="cuda")
    else:
        tokens = case.get("tokens", 1)
        st["table"] = torch.tensor([t["pages"][e].data_ptr() for e in range(E)], dtype=torch.int64).cuda()
        soft = _softplus(case)
        st["route"] = s14.Router(
            t["weight"], t["bias"], score_fn=N.S14_SCORE_SQRT_SOFTPLUS if soft else N.S14_SCORE_SIGMOID,
            route_scale=1.5 if soft else 1.0, tid2eid=t["tid2eid"], token_ids=t["token_ids"])
        st["format"] = N.S14_PAGE_FP8 if case.get("shared") == "fp8" else N.S14_PAGE_MXFP4
        st["y"] = torch.empty((tokens, H), device="cuda")
        st["ids"] = torch.empty((tokens, K), dtype=torch.int16, device="cuda")
        st["weights"] = torch.empty((tokens, K), device="cuda")
    return st


def run(st):
    case, ctx, mode = st["case"], st["ctx"], st["mode"]
    kind = case["kind"]
    if kind == "chain":
        s14.expert_chain(ctx, st["page"], st["x"], case.get("route_w", 0.17), st["y"], mode=mode)
        return {"y": st["y"]}
    if kind == "matvec":
        st["cmd"](st["dispatch"])
        return {"y": st["y"]}
    if kind == "linear":
        s14.act_quant_e4m3(ctx, st["x"], st["q"], st["qs"])
        s14.fp8_linear(ctx, st["q"], st["qs"], st["w"], st["s"], st["y"], round_bf16=case["bf16"], mode=mode)
        return {"y": st["y"], "q": st["q"], "scales": st["qs"]}
    args = (st["route"], st["table"], st["shared"], st["x"], st["y"])
    outs = {"ids_out": st["ids"], "weights_out": st["weights"], "mode": mode}
    if kind == "layer":
        s14.moe_layer_route(ctx, *args, shared_format=st["format"], **outs)
    elif kind == "block":
        s14.moe_block_route(ctx, case["tokens"], *args, shared_format=st["format"], **outs)
    else:
        s14.moe_prefill(ctx, case["tokens"], *args, **outs)
    return {"y": st["y"], "ids": st["ids"], "weights": st["weights"]}


# ---------------------------------------------------------------------------
# what the path cannot do without
# ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "chain":
        return {"bytes": MX["total"] + 8 * H, "flops": 6 * H * I}
    if kind in ("matvec", "linear"):
        n, k, m = case["n"], case["k"], case.get("m", 1)
        if kind == "matvec":
            b = n * k // 2 + n * k // 32 + 4 * k if case["format"] == "mxfp4" else n * k + 2 * k
            return {"bytes": b + 4 * n, "flops": 2 * n * k}
        # f32 activations in, their codes out and back in, weights, f32 outputs
        return {"bytes": 4 * m * k + 2 * m * k + n * k + 4 * m * n, "flops": 2 * m * n * k}
    tokens = case.get("tokens", 1)
    if kind == "prefill":
        p = synth.zipf_top6_inclusion(1.1)
        distinct = float((1.0 - (1.0 - p) ** tokens).sum())
    else:
        distinct = K + 5.07 * (tokens - 1)  # adjacent tokens share 0.57 of six; others meet by chance
    shared = F8["total"] if case.get("shared") == "fp8" else MX["total"]
    b = distinct * MX["total"] + shared + 4 * E * H + 8 * tokens * H
    return {"bytes": b, "flops": tokens * (K + 1) * 6 * H * I + 2 * tokens * E * H}


def tolerance(case):
    """Exact-order calls are bit-identical to the CPU oracle; the others'
    bounds are four times what another order of the sums was seen to give."""
    kind, mode = case["kind"], case["mode"]
    if kind == "prefill":
        # a sum one rounding off moves a few E4M3 codes of h by one step
        # (against 64 bits: 2.3e-4 at 512 tokens, official 1.2e-4 at 1,024)
        return {"rel": 5e-4 if mode == "official" else 1e-3, "max": 0.1}
    if mode == "fast":
        if kind == "linear" and case["bf16"]:  # a bf16 rounding flips here and there
            return {"rel": 1e-4, "max": 0.01}
        return {"rel": 2e-6, "max": 2e-4}  # 2.2e-7 against 64 bits
    return "exact"


# ---------------------------------------------------------------------------
# 64-bit results, in plain torch
# ---------------------------------------------------------------------------

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _mx64(codes, scales):
    """[n, k / 2] E2M1 pairs and [n, k / 32] UE8M0 codes -> [n, k] in 64 bits."""
    table = torch.tensor(_E2M1, dtype=torch.float64, device="cuda")
    c = codes.long()
    v = torch.stack([table[c & 15], table[c >> 4]], dim=-1).flatten(-2)
    s = torch.exp2(scales.double() - 127.0)
    return (v.unflatten(-1, (-1, 32)) * s[..., None]).flatten(-2)


def _f8_64(codes, scales):
    """[n, k] E4M3 codes and [ceil(n / 128), ceil(k / 128)] tile scales."""
    n, k = codes.shape
    s = torch.exp2(scales.double() - 127.0) if scales.dtype == torch.uint8 else scales.double()
    s = s.repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]
    return codes.view(torch.float8_e4m3fn).double() * s


def _page64(page, fp8=False):
    o, per = (F8, 1) if fp8 else (MX, 2)
    out = []
    for w, s, end, n, k in (("w1", "s1", "w3", I, H), ("w3", "s3", "w2", I, H), ("w2", "s2", "total", H, I)):
        codes, scales = page[o[w]:o[s]].view(n, k // per), page[o[s]:o[end]]
        out.append(_f8_64(codes, scales.view(n // 128, k // 128)) if fp8 else _mx64(codes, scales.view(n, k // 32)))
    return out


def _requant(v, group):
    """E4M3 codes and UE8M0 scales of `v` per `group` values: (codes, scales, values)."""
    a = v.to(torch.float32).unflatten(-1, (-1, group))
    m, e = torch.frexp(a.abs().amax(-1).clamp_min(1e-4).double() / 448.0)
    e = torch.where(m == 0.5, e - 1, e)  # ceil(log2)
    q = (a.double() * torch.exp2(-e.double())[..., None]).float().clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    back = (q.double() * torch.exp2(e.double())[..., None]).flatten(-2)
    return q.view(torch.uint8).flatten(-2), (e + 127).to(torch.uint8), back


def _bf16(v):
    return v.float().bfloat16().double()


def _swiglu64(g, u):
    g, u = g.clamp_max(10.0), u.clamp(-10.0, 10.0)
    return g / (1.0 + torch.exp(-g)) * u


def _expert64(w, x, mode, route_w, group):
    """One expert's rows of x (already requantised where the path does), the
    route weight applied: [t, H]."""
    g, u = x @ w[0].T, x @ w[1].T
    if mode == "official":
        h = _bf16(_swiglu64(_bf16(g), _bf16(u)).mul(route_w[:, None]))
        return _bf16(_requant(h, 128)[2] @ w[2].T)
    h = _swiglu64(g, u)
    if group:
        h = _requant(h, group)[2]
    return route_w[:, None] * (h @ w[2].T)


def _route64(case, t):
    z = t["x"].double() @ t["weight"].double().T
    s = torch.nn.functional.softplus(z).sqrt() if _softplus(case) else torch.sigmoid(z)
    if t["tid2eid"] is not None:
        ids = t["tid2eid"][t["token_ids"].long()]
    else:
        ids = (s + t["bias"].double()).topk(K, dim=1).indices
    w = s.gather(1, ids)
    return ids, w / w.sum(1, keepdim=True) * (1.5 if _softplus(case) else 1.0)


def exact(case, seed):
    t = _inputs(case, seed)
    kind, mode = case["kind"], case["mode"]
    if kind == "matvec":
        w = _mx64(t["w"], t["s"]) if case["format"] == "mxfp4" else _f8_64(t["w"], t["s"])
        return {"y": w @ t["x"].double()}
    if kind == "linear":
        q, s, x = _requant(t["x"], 128)
        y = x @ _f8_64(t["w"], t["s"]).T
        return {"y": _bf16(y) if case["bf16"] else y, "q": q, "scales": s}
    if kind == "chain":
        x = t["x"].double()[None]
        if mode == "official":
            x = _requant(t["x"][None], 128)[2]
        w = torch.full((1,), case.get("route_w", 0.17), dtype=torch.float32, device="cuda").double()
        return {"y": _expert64(_page64(t["page"]), x, mode, w, 0)[0]}
    ids, weights = _route64(case, t)
    group = 32 if kind == "prefill" and mode != "official" else 0
    if mode == "official":
        x = _requant(t["x"], 128)[2]
    else:
        x = _requant(t["x"], group)[2] if group else t["x"].double()
    ones = torch.ones(x.shape[0], dtype=torch.float64, device="cuda")
    y = _expert64(_page64(t["shared"], case.get("shared") == "fp8"), x, mode, ones, group)
    for e in ids.unique().tolist():
        row, slot = (ids == e).nonzero(as_tuple=True)
        y.index_add_(0, row, _expert64(_page64(t["pages"][e]), x[row], mode, weights[row, slot], group))
    return {"y": _bf16(y) if mode == "official" else y, "ids": None, "weights": weights}
