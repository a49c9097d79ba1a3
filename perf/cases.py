"""The layer calls whose time and results are followed from change to change: a serving program's decode steps and
prefill chunks of one routed int4 MoE layer (hidden 6144, expert width 2048, 256 experts, top-8), through the public
entry points of hecate_amd.

A case is a dict of plain values:
  kind       "layer"    the whole layer of `rows` tokens, MoELayer.forward: decode up to 16 rows, prefill above
             "partial"  the routed experts a GPU holds, added into an fp32 partial: MoELayer.decode with y up to 16 rows,
                        above it the operators a program drives itself (router_fused, the dispatch plan, moe4p.forward)
             "step"     one decode layer in the serving stack's own operators: norm_route, moe4.forward, combine_norm
             "stack"    `layers` layers of a decode step with the norms between them, replayed as one hipGraph
  rows       tokens of the call
  resident   experts held on the GPU (of 256; picks of the others contribute nothing)
  popularity "even" (a small random selection bias) or "zipf" (expert popularity falling as rank^-1.1)

Inputs and weights are drawn from the seed on the device: int4 codes uniform in -8..7, bf16 group scales |N(0, 0.004)|,
shared expert N(0, 0.02), router N(0, 0.02), tokens N(0, 1).
"""
import math

import torch

from hecate_amd import cn, moe4, moe4p, router, stack, tier

H, I, E, TOPK, SCALE, EPS = 6144, 2048, 256, 8, 2.5, 1e-5
EXPERT_BYTES = 3 * (I * H // 2) + 3 * (I * H // 128) * 2
SHARED_BYTES = 3 * I * H * 2
MATS = (("gate", I, H), ("up", I, H), ("down", H, I))


def listed():
    return [
        # one request decoding: the latency-bound step
        dict(name="decode-1", kind="layer", rows=1, resident=256, popularity="even"),
        # a tier that holds 176 experts, a few requests, its partial joined with another tier's later
        dict(name="partial-decode-3", kind="partial", rows=3, resident=176, popularity="zipf"),
        # 8 requests
        dict(name="decode-8", kind="layer", rows=8, resident=256, popularity="even"),
        # 8 requests with a draft row each, experts of uneven popularity: the largest decode call
        dict(name="decode-16-zipf", kind="layer", rows=16, resident=256, popularity="zipf"),
        # the serving stack's own operators around one decode layer
        dict(name="norm-step-5", kind="step", rows=5, resident=256, popularity="even"),
        # a decode step through consecutive layers as a captured graph
        dict(name="stack-4x4", kind="stack", rows=4, resident=256, popularity="even", layers=4),
        # more requests than a decode call takes
        dict(name="prefill-33", kind="layer", rows=33, resident=256, popularity="even"),
        # a short prompt
        dict(name="prefill-150", kind="layer", rows=150, resident=256, popularity="even"),
        # an ordinary prompt on a tier that holds part of the experts
        dict(name="partial-prefill-450", kind="partial", rows=450, resident=176, popularity="even"),
        # an ordinary prompt with uneven experts
        dict(name="prefill-1000-zipf", kind="layer", rows=1000, resident=256, popularity="zipf"),
        # a full prefill chunk
        dict(name="prefill-2048", kind="layer", rows=2048, resident=256, popularity="even"),
        # a long chunk (the long-prefill operator)
        dict(name="prefill-8192", kind="layer", rows=8192, resident=256, popularity="even"),
    ]


def draw(rng):
    pop = rng.choice(("even", "even", "zipf"))
    kind = rng.choice(("decode", "decode", "step", "prefill", "prefill", "prefill", "prefill", "partial"))
    if kind == "decode":
        rows, res = rng.randint(1, 16), rng.choice((256, 256, 176, rng.randint(64, 255)))
        return dict(kind="layer" if res == 256 else "partial", rows=rows, resident=res, popularity=pop)
    if kind == "step":
        return dict(kind="step", rows=rng.randint(1, 16), resident=256, popularity=pop)
    rows = int(round(math.exp(rng.uniform(math.log(17), math.log(2048 if kind == "partial" else 8192)))))
    if kind == "partial":
        return dict(kind="partial", rows=rows, resident=rng.choice((176, rng.randint(64, 255))), popularity=pop)
    return dict(kind="layer", rows=rows, resident=256, popularity=pop)


# ---- inputs and weights ------------------------------------------------------------------------------------------
def _weights(case, g, dev):
    """one layer's router, bias, resident experts and shared expert, drawn from the generator g"""
    n = case["resident"]
    wg = torch.empty(E, H, device=dev).normal_(0, 0.02, generator=g)
    if case["popularity"] == "zipf":
        rank = torch.randperm(E, generator=g, device=dev).float() + 1
        if n < E:                                        # the tier holds the most popular experts
            rank = rank.sort().values
        lz = -1.1 * rank.log()
        bias = 0.0585 * (lz - lz.mean())
    else:
        bias = torch.empty(E, device=dev).normal_(0, 0.01 if case["rows"] <= 16 else 0.001, generator=g)
    bank = tier.ExpertBank(n, dev)
    for m, _, _ in MATS:
        bank.buf[m + "_q"].random_(0, 256, generator=g)
        bank.buf[m + "_s"].view(torch.bfloat16).normal_(0, 0.004, generator=g).abs_()
    shared = tuple(torch.empty(N * K, dtype=torch.bfloat16, device=dev).normal_(0, 0.02, generator=g).half()
                   for _, N, K in MATS)
    return wg, bias, bank, shared


def _inputs(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    R = case["rows"]
    s = dict(case=case, x=torch.empty(R, H, dtype=torch.bfloat16, device=dev).normal_(0, 1, generator=g))
    s["weights"] = [_weights(case, g, dev) for _ in range(case.get("layers", 1))]
    if case["kind"] == "stack":
        s["norms"] = [torch.empty(H, device=dev).normal_(1, 0.1, generator=g) for _ in range(case["layers"])]
    if case["kind"] == "step":
        s["h"] = torch.empty(R, H, device=dev).normal_(0, 1, generator=g)           # the attention output
        s["r0"] = torch.empty(R, H, device=dev).normal_(0, 1, generator=g)          # the residual before it
        s["norms"] = [torch.empty(H, device=dev).normal_(1, 0.1, generator=g) for _ in range(2)]
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    R, n, kind, dev = case["rows"], case["resident"], case["kind"], s["x"].device
    layers = [tier.MoELayer(wg, b, bank, None if kind == "partial" else sh, lo=0, n_hot=n, topk=TOPK, scale=SCALE,
                            max_rows=R) for wg, b, bank, sh in s["weights"]]
    s["lay"] = layers[0]
    if kind == "partial":
        s["y"] = torch.zeros(R, H, device=dev)
        if R > 16:
            s["pf"] = tier.PrefillBuffers(R, TOPK, 0, n, E, dev, bm=128)
    elif kind == "step":
        s["r"], s["y"] = torch.empty_like(s["r0"]), torch.zeros(R, H, device=dev)
        s["x2"], s["xn"] = (torch.empty(R, H, dtype=torch.bfloat16, device=dev) for _ in range(2))
        s["sel"] = torch.zeros(R, TOPK, dtype=torch.int64, device=dev)
        s["rw"] = torch.zeros(R, TOPK, dtype=torch.float16, device=dev)
        s["cand"], s["ctr"] = router.norm_route_buffers(R, dev)
        s["scr"] = moe4.scratch(dev)
    elif kind == "stack":
        s["stack"] = stack.DecodeStack(layers, s["norms"], R, EPS)
        s["stack"].capture()
    return s


def run(s):
    case, lay, x = s["case"], s["lay"], s["x"]
    kind, R = case["kind"], case["rows"]
    if kind == "layer":
        return lay.forward(x)
    if kind == "partial":
        y = s["y"]
        y.zero_()
        if R <= 16:
            lay.decode(x, y=y, out=False, with_shared=False)
            return y
        pf = s["pf"]
        router.router_fused(x, lay.wg, lay.bias, pf.logits, lay.ctr, pf.sel, pf.rw, TOPK, SCALE, pf.xh)
        pf.run(pf.sel, pf.rw)
        gq, uq, dq, gs, us, ds = lay.bank.tables()
        moe4p.forward(pf.xh, pf.tok, pf.eid, pf.wt, pf.rbt, gq, uq, dq, gs, us, ds, *pf.scr, y, inv=pf.inv, meta=pf.meta)
        return y
    if kind == "step":
        r, y, x2, xn, sel, rw = s["r"], s["y"], s["x2"], s["xn"], s["sel"], s["rw"]
        r.copy_(s["r0"])
        router.norm_route(s["h"], r, s["norms"][0], x2, lay.wg, lay.bias, sel, rw, s["cand"], s["ctr"], SCALE, EPS)
        gq, uq, dq, gs, us, ds = lay.bank.tables()
        moe4.forward(x2, sel, rw, lay.n_hot, gq, uq, dq, gs, us, ds, *s["scr"], y, 0, 0, 0, *lay.shared)
        cn.combine_norm(None, 0, y, R, 0, 0, r, s["norms"][1], xn, EPS)
        return {"residual": r, "normed": xn}
    s["stack"].x.copy_(x)
    return s["stack"].replay()


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _expected(case):
    """(distinct resident experts, resident picks) of a call, in expectation"""
    R, n = case["rows"], case["resident"]
    if case["popularity"] == "zipf":
        w = [(e + 1) ** -1.1 for e in range(E)]
        t = sum(w)
        p = [min(1.0, TOPK * v / t) for v in w][:n]
    else:
        p = [TOPK / E] * n
    return sum(1 - (1 - q) ** R for q in p), R * min(TOPK, sum(p))


def work(case):
    R, L = case["rows"], case.get("layers", 1)
    distinct, picks = _expected(case)
    sh = case["kind"] != "partial"
    size = distinct * EXPERT_BYTES + (SHARED_BYTES if sh else 0) + E * H * 4 + R * H * (2 + (2 if sh else 4))
    if case["kind"] in ("step", "stack"):
        size += R * H * 12 + 2 * H * 4
    return {"bytes": L * size, "flops": L * ((picks + (R if sh else 0)) * 6 * H * I + R * 2 * E * H)}


def tolerance(case):
    if case["kind"] == "partial":            # fp32 sums of f16-rounded weights and activations
        return {"rel": 2e-3, "max": 2e-2}
    if case["kind"] == "stack":              # fp32 residual over layers whose inputs are rounded to bf16
        return {"rel": 2.5e-2, "max": 3e-1}
    return {"rel": 7e-3, "max": 5e-2}        # bf16 outputs


# ---- the same in 64 bits -----------------------------------------------------------------------------------------
def _int4(q, s, N, K):
    """an I4G128 matrix (include/hecate_moe.h) as float64 [N, K]"""
    w = q.view(torch.int32).view(N // 16, K // 128, 4, 16, 4, 1)
    shift = torch.tensor([4 * (e // 2) + 16 * (e % 2) for e in range(8)], dtype=torch.int32, device=q.device)
    v = ((w >> shift) & 15) - 8                                             # [nb, kg, c, row, j, e]
    v = v.permute(0, 3, 1, 4, 2, 5).reshape(N, K // 128, 128).double()
    sc = s.view(torch.bfloat16).view(N // 16, K // 512, 16, 4).permute(0, 2, 1, 3).reshape(N, K // 128, 1)
    return (v * sc.double()).view(N, K)


def _dense(t, N, K):
    """an F16T matrix (include/hecate_moe.h) as float64 [N, K]"""
    return t.view(N // 16, K // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(N, K).double()


def _mlp(x, g, u, d):
    a = x @ g.T
    return (a * torch.sigmoid(a) * (x @ u.T)) @ d.T


def _moe(x, weights, shared):
    """one layer of x (float64 [R, H])"""
    wg, bias, bank, sh = weights
    a = torch.sigmoid(x @ wg.double().T)
    sel = (a + bias.double()).topk(TOPK, dim=1).indices
    rw = a.gather(1, sel)
    rw = rw * SCALE / (rw.sum(1, keepdim=True) + 1e-20)
    y = torch.zeros_like(x)
    for e in torch.unique(sel).tolist():
        if e >= bank.n:
            continue
        t, k = (sel == e).nonzero(as_tuple=True)
        m = [_int4(bank.view(m + "_q", e), bank.view(m + "_s", e), N, K) for m, N, K in MATS]
        y[t] += _mlp(x[t], *m) * rw[t, k, None]
    if shared:
        y += _mlp(x, *(_dense(t, N, K) for t, (_, N, K) in zip(sh, MATS)))
    return y


def _norm(r, w):
    return r * w.double() / (r.square().mean(1, keepdim=True) + EPS).sqrt()


def exact(case, seed):
    s = _inputs(case, seed)
    x, kind = s["x"].double(), case["kind"]
    if kind in ("layer", "partial"):
        return _moe(x, s["weights"][0], kind == "layer")
    if kind == "step":
        r = s["h"].double() + s["r0"].double()
        x2 = _norm(r, s["norms"][0]).bfloat16().double()                    # (the layer's input is bf16)
        r = r + _moe(x2, s["weights"][0], True)
        return {"residual": r, "normed": _norm(r, s["norms"][1])}
    h = x
    for w, nw in zip(s["weights"], s["norms"]):
        h = h + _moe(_norm(h, nw).bfloat16().double(), w, True)
    return h
