"""The workloads that a user of this package runs, and how each one is made, run and checked.

Kinds (every size is a field of the case):
  products  the decode products of one layer, each over its own resident rows, as a recorded plan: the int8 rows
            (linear.quantize), then q/k/v, o, gate/up and down (Linear.gemv_q), 1 to 16 tokens, hp or not
  step      a decode step through a stack of layers as a captured graph, with the fused input producers: rmsfold, q/k/v,
            fold, o, rmsfold, gate/up, smfold, down a layer (attention itself is not part of the package: o takes q's
            rows), a final norm at the end
  prompt    a short prompt: one layer's seven products above the decode range (linear.quantize, Linear.gemm)
  mlp       the feed-forward block of a prompt chunk: rmsfold, gate, up, smfold, down (group scales, fp32 outputs)
  chunk     prefill products over resident int8 trit copies: linear.quantize per token row, Linear.gemm8, fp16 outputs
  moe       one q8_0 MoE feed-forward: MoE.decode at few tokens (tokens x picks up to 64), MoE.forward above
  q8        one dense q8_0 product: q8_quantize, Q8Matrix.gemv

Ternary weights are i.i.d. trits (0.3 / 0.4 / 0.3) with one fp16 scale a 128-column group, q8_0 weights int8 codes with
one fp16 scale a 32-column block, activations N(0, 1) with a spread of row sizes, as a model's stream has them.
"""
import math

import torch

from kindi_amd import linear, moe

DEV = "cuda"

# model classes: hidden width, key/value rows, feed-forward width, Hadamard blocks of the hidden and feed-forward rows
CLASSES = {
    "2b": dict(hidden=2048, kv=512, ff=6144, hb=1024, hbf=1024),
    "9b": dict(hidden=4096, kv=1024, ff=12288, hb=4096, hbf=4096),
    "27b": dict(hidden=5120, kv=1024, ff=17408, hb=1024, hbf=1024),
}


def listed():
    return [
        # one token through a small model's layer: launch latency is what a user waits for
        dict(name="products_2b_1", kind="products", cls="2b", M=1, hp=False),
        # four tokens in the two-row high-precision form on a mid-size model
        dict(name="products_9b_hp_4", kind="products", cls="9b", M=4, hp=True),
        # single-stream generation on the large model (8 of its layers: more weights than the caches hold)
        dict(name="step_27b_1", kind="step", cls="27b", M=1, layers=8),
        # 16 streams (or a 16-token speculative check) on the large model
        dict(name="step_27b_16", kind="step", cls="27b", M=16, layers=4),
        # a chat turn: a prompt of a few dozen tokens, an odd count
        dict(name="prompt_27b_61", kind="prompt", cls="27b", M=61),
        # a chunk of a long prompt through a feed-forward block, group scales, a ragged count
        dict(name="mlp_9b_1000", kind="mlp", cls="9b", M=1000),
        # a full prefill chunk over the int8 trit copies, fp16 rows out
        dict(name="chunk_9b_2048", kind="chunk", cls="9b", M=2048),
        # one token of a 30B-class mixture of experts: 128 experts, 6 picks
        dict(name="moe_1", kind="moe", M=1, E=128, k=6, H=2688, F=1856, score="softmax"),
        # a speculative check of 7 tokens with the sigmoid router: 42 experts touched or fewer
        dict(name="moe_7", kind="moe", M=7, E=128, k=6, H=2688, F=1856, score="sigmoid"),
        # many streams at once, or a short prompt: every expert is touched, a dozen tokens each
        dict(name="moe_256", kind="moe", M=256, E=128, k=6, H=2688, F=1856, score="softmax"),
        # a prefill chunk: about a hundred tokens an expert
        dict(name="moe_2048", kind="moe", M=2048, E=128, k=6, H=2688, F=1856, score="sigmoid"),
        # a dense q8_0 projection beside the experts, a short prompt
        dict(name="q8_dense_50", kind="q8", M=50, R=4096, C=2688),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["products", "step", "prompt", "mlp", "chunk", "moe", "moe", "moe", "q8"])
    cls = rng.choice(sorted(CLASSES))
    if kind == "products":
        return dict(kind=kind, cls=cls, M=_log_int(rng, 1, 16), hp=rng.random() < 0.3)
    if kind == "step":
        return dict(kind=kind, cls=cls, M=_log_int(rng, 1, 16), layers=rng.randint(2, 6))
    if kind == "prompt":
        return dict(kind=kind, cls=cls, M=_log_int(rng, 17, 400))
    if kind == "mlp":
        return dict(kind=kind, cls=rng.choice(["2b", "9b"]), M=_log_int(rng, 64, 1000))
    if kind == "chunk":
        return dict(kind=kind, cls=rng.choice(["2b", "9b"]), M=_log_int(rng, 256, 2048))
    if kind == "moe":
        return dict(kind=kind, M=_log_int(rng, 1, 2048), E=rng.choice([60, 64, 96, 128]), k=rng.choice([4, 6]),
                    H=32 * rng.randint(32, 84), F=32 * rng.randint(16, 58), score=rng.choice(["softmax", "sigmoid"]))
    return dict(kind=kind, M=_log_int(rng, 1, 600), R=8 * rng.randint(64, 1024) + rng.randint(0, 7),
                C=32 * rng.randint(32, 128))


# ------------------------------------------------------------------------------------------------ inputs
def _mats(case):
    c = CLASSES[case["cls"]]
    H, KV, F = c["hidden"], c["kv"], c["ff"]
    return [("q", H, H), ("k", KV, H), ("v", KV, H), ("o", H, H), ("gate", F, H), ("up", F, H), ("down", H, F)]


def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000 + stream)
    return g


def _tern_raw(R, C, seed, stream):
    """digits uint8 [C/4, R, 4] (trit + 1 of columns 4 i + j) and scales fp16 [C/128, R]"""
    g = _gen(seed, stream)
    u = torch.rand((C // 4, R, 4), generator=g, device=DEV)
    d = (u >= 0.3).to(torch.uint8) + (u >= 0.7).to(torch.uint8)
    s = torch.exp(torch.randn((C // 128, R), generator=g, device=DEV) * 0.3 - 3.0).to(torch.float16)
    return d, s


def _tern(R, C, seed, stream):
    d, s = _tern_raw(R, C, seed, stream)
    b = d[..., 0] + 3 * d[..., 1] + 9 * d[..., 2] + 27 * d[..., 3]
    return linear.TernaryMatrix(b.contiguous(), s.view(torch.int16).contiguous(), R, C, device=DEV)


def _tern64(R, C, seed, stream):
    """the same matrix dense in 64 bits, [R, C]"""
    d, s = _tern_raw(R, C, seed, stream)
    w = d.permute(1, 0, 2).reshape(R, C).double() - 1.0
    return w * s.double().t().repeat_interleave(128, dim=1)


def _rows(M, C, seed, stream):
    """fp32 rows N(0, 1), each row with a size of its own"""
    g = _gen(seed, stream)
    x = torch.randn((M, C), generator=g, device=DEV)
    return (x * torch.exp(0.5 * torch.randn((M, 1), generator=g, device=DEV))).contiguous()


def _signs(C, seed, stream):
    return torch.where(torch.rand(C, generator=_gen(seed, stream), device=DEV) < 0.5, -1.0, 1.0).float()


def _norm_w(C, seed, stream):
    return 1.0 + 0.1 * torch.randn(C, generator=_gen(seed, stream), device=DEV)


def _q8_raw(R, C, seed, stream):
    """codes int8 [R, C/32, 32], scales fp16 [R, C/32, 1]"""
    g = _gen(seed, stream)
    c = torch.randint(-127, 128, (R, C // 32, 32), generator=g, device=DEV, dtype=torch.int8)
    s = torch.exp(torch.randn((R, C // 32, 1), generator=g, device=DEV) * 0.5 - 6.0).to(torch.float16)
    return c, s


def _q8_rows(R, C, seed, stream):
    c, s = _q8_raw(R, C, seed, stream)
    return torch.cat([s.view(torch.uint8), c.view(torch.uint8)], dim=2).reshape(R, C // 32 * 34).contiguous()


def _q8_64(R, C, seed, stream):
    c, s = _q8_raw(R, C, seed, stream)
    return (c.double() * s.double()).reshape(R, C)


def _bias(E, seed):
    return 0.1 * torch.randn(E, generator=_gen(seed, 7), device=DEV)


ROUTE_SCALE = 2.5                                   # the sigmoid router's scale of the normalized weights


# ------------------------------------------------------------------------------------------------ prepare
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_products(case, seed):
    c, M, hp = CLASSES[case["cls"]], case["M"], case["hp"]
    L = linear.Linear({n: _tern(R, C, seed, i) for i, (n, R, C) in enumerate(_mats(case))}, device=DEV, hp=hp)
    H, KV, F = c["hidden"], c["kv"], c["ff"]
    groups = [(("q", "k", "v"), H), (("o",), H), (("gate", "up"), H), (("down",), F)]
    rows = {"q": H, "k": KV, "v": KV, "o": H, "gate": F, "up": F, "down": H}
    xs = [_rows(M, C, seed, 20 + i) for i, (_, C) in enumerate(groups)]
    Mq = 2 * M if hp else M
    acts = [linear.Act(torch.empty((Mq, C), dtype=torch.int8, device=DEV),
                       torch.empty((Mq, C // 128), dtype=torch.float32, device=DEV),
                       torch.empty((Mq, C // 128), dtype=torch.int32, device=DEV), M, C, False, hp) for _, C in groups]
    outs = {n: torch.empty((M, R), dtype=torch.float32, device=DEV) for n, R in rows.items()}

    def step():
        for (names, _), x, a in zip(groups, xs, acts):
            L.gemv_q(list(names), linear.quantize(x, out=a, hp=hp), [outs[n] for n in names])

    return dict(L=L, xs=xs, acts=acts, outs=outs, plan=linear.Plan(step, 16), run=_run_products)


def _run_products(s):
    s["plan"].launch()
    return s["outs"]


def _prepare_step(case, seed):
    c, M, n = CLASSES[case["cls"]], case["M"], case["layers"]
    H, KV, F, HB, HBF = c["hidden"], c["kv"], c["ff"], c["hb"], c["hbf"]
    L = linear.Linear({"%s%d" % (m, l): _tern(R, C, seed, 100 * l + i)
                       for l in range(n) for i, (m, R, C) in enumerate(_mats(case))}, device=DEV)
    x = _rows(M, H, seed, 20)
    sg = [[_signs(w, seed, 100 * l + 30 + j) for j, w in enumerate((H, H, H, F))] for l in range(n)]
    nw = [[_norm_w(H, seed, 100 * l + 40 + j) for j in range(2)] for l in range(n)]
    sf, wf = _signs(H, seed, 50), _norm_w(H, seed, 51)

    def f32(w):
        return torch.empty((M, w), dtype=torch.float32, device=DEV)

    def act(w):
        return linear.Act(torch.empty((M, w), dtype=torch.int8, device=DEV),
                          torch.empty((M, w // 128), dtype=torch.float32, device=DEV),
                          torch.empty((M, w // 128), dtype=torch.int32, device=DEV), M, w, False)

    a1, a2, a3, a4 = act(H), act(H), act(H), act(F)
    xa, xb, xn = f32(H), f32(H), f32(H)
    q, o, gt, up, dn = f32(H), f32(H), f32(F), f32(F), f32(H)
    ks, vs = [f32(KV) for _ in range(n)], [f32(KV) for _ in range(n)]

    def step():
        cur, part = x, None
        for l in range(n):
            s = sg[l]
            a = linear.rmsfold(cur, nw[l][0], s[0], HB, r=part, nparts=0 if part is None else 1,
                               xw=None if part is None else xa, out=a1)
            cur = cur if part is None else xa
            L.gemv_q(["q%d" % l, "k%d" % l, "v%d" % l], a, [q, ks[l], vs[l]])
            L.gemv_q(["o%d" % l], linear.fold(q, s[1], HB, out=a2), [o])
            a = linear.rmsfold(cur, nw[l][1], s[2], HB, r=o, nparts=1, xw=xb, out=a3)
            cur = xb
            L.gemv_q(["gate%d" % l, "up%d" % l], a, [gt, up])
            L.gemv_q(["down%d" % l], linear.smfold(gt, up, s[3], HBF, out=a4), [dn])
            part = dn
        linear.rmsfold(cur, wf, sf, HB, r=part, nparts=1, xw=xa, xn=xn, out=a1)

    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        step()
    torch.cuda.current_stream().wait_stream(st)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    return dict(L=L, x=x, keep=(sg, nw, sf, wf, a1, a2, a3, a4, xb, q, o, gt, up, dn), graph=g,
                outs=dict(x=xa, xn=xn, k=ks, v=vs), run=_run_step)


def _run_step(s):
    s["graph"].replay()
    return s["outs"]


def _prepare_prompt(case, seed):
    c, M = CLASSES[case["cls"]], case["M"]
    L = linear.Linear({n: _tern(R, C, seed, i) for i, (n, R, C) in enumerate(_mats(case))}, device=DEV)
    widths = (c["hidden"], c["hidden"], c["hidden"], c["ff"])
    return dict(L=L, xs=[_rows(M, C, seed, 20 + i) for i, C in enumerate(widths)], run=_run_prompt)


def _run_prompt(s):
    L, outs = s["L"], {}
    for x, names in zip(s["xs"], (("q", "k", "v"), ("o",), ("gate", "up"), ("down",))):
        a = linear.quantize(x)
        for n in names:
            outs[n] = L.gemm(n, a)
    return outs


def _prepare_mlp(case, seed):
    c, M = CLASSES[case["cls"]], case["M"]
    H, F = c["hidden"], c["ff"]
    L = linear.Linear({n: _tern(R, C, seed, i) for i, (n, R, C) in enumerate(_mats(case)) if i >= 4}, device=DEV)
    return dict(L=L, c=c, x=_rows(M, H, seed, 20), r=_rows(M, H, seed, 21), w=_norm_w(H, seed, 40),
                sg=_signs(H, seed, 30), sgf=_signs(F, seed, 31),
                xw=torch.empty((M, H), dtype=torch.float32, device=DEV), run=_run_mlp)


def _run_mlp(s):
    L, c = s["L"], s["c"]
    a = linear.rmsfold(s["x"], s["w"], s["sg"], c["hb"], r=s["r"], nparts=1, xw=s["xw"])
    h = linear.smfold(L.gemm("gate", a), L.gemm("up", a), s["sgf"], c["hbf"])
    return dict(xw=s["xw"], y=L.gemm("down", h))


def _prepare_chunk(case, seed):
    c, M = CLASSES[case["cls"]], case["M"]
    H, F = c["hidden"], c["ff"]
    L = linear.Linear({n: _tern(R, C, seed, i) for i, (n, R, C) in enumerate(_mats(case)) if n in ("up", "down")},
                      device=DEV, per_row=True)
    return dict(L=L, w8={n: L.w[n].expand() for n in ("up", "down")}, x=_rows(M, H, seed, 20), h=_rows(M, F, seed, 21),
                y={"up": torch.empty((M, F), dtype=torch.float16, device=DEV),
                   "down": torch.empty((M, H), dtype=torch.float16, device=DEV)}, run=_run_chunk)


def _run_chunk(s):
    L = s["L"]
    for n, x in (("up", s["x"]), ("down", s["h"])):
        L.gemm8(n, linear.quantize(x, per_row=True), s["w8"][n], Y16=s["y"][n])
    return s["y"]


def _prepare_moe(case, seed):
    M, E, k, H, F = (case[n] for n in ("M", "E", "k", "H", "F"))
    up = moe.Q8Experts([_q8_rows(F, H, seed, 100 + e) for e in range(E)], F, H, device=DEV)
    down = moe.Q8Experts([_q8_rows(H, F, seed, 400 + e) for e in range(E)], H, F, device=DEV)
    sig = case["score"] == "sigmoid"
    layer = moe.MoE(up, down, k, device=DEV, score=case["score"], bias=_bias(E, seed) if sig else None,
                    scale=ROUTE_SCALE if sig else 1.0)
    few = M * k <= 64
    x0 = _rows(M, H, seed, 20)
    return dict(layer=layer, x0=x0, x=torch.empty_like(x0), logits=_logits(M, E, seed),
                work=layer.workspace(M) if few else layer.buffers(M), run=_run_moe_few if few else _run_moe_many)


def _logits(M, E, seed):
    return torch.randn((M, E), generator=_gen(seed, 21), device=DEV)


def _run_moe_few(s):
    s["x"].copy_(s["x0"])                          # the residual stream that the layer before left: updated in place
    return s["layer"].decode(s["x"], s["logits"], s["work"])


def _run_moe_many(s):
    s["x"].copy_(s["x0"])
    return s["layer"].forward(s["x"], s["logits"], s["work"])[0]


def _prepare_q8(case, seed):
    R, C = case["R"], case["C"]
    return dict(W=moe.Q8Matrix(_q8_rows(R, C, seed, 0), R, C, device=DEV), x=_rows(case["M"], C, seed, 20), run=_run_q8)


def _run_q8(s):
    Q, D = moe.q8_quantize(s["x"])
    return s["W"].gemv(Q, D)


# ------------------------------------------------------------------------------------------------ bytes, operations
def work(case):
    kind = case["kind"]
    if kind in ("products", "prompt", "step"):
        M, ms = case["M"], _mats(case)
        n = case.get("layers", 1)
        w = sum(R * C for _, R, C in ms)
        c = CLASSES[case["cls"]]
        if kind == "step":
            io = M * 4 * (c["hidden"] * 3 + n * 2 * c["kv"]) + n * 4 * (5 * c["hidden"] + c["ff"])
        else:
            io = M * 4 * (3 * c["hidden"] + c["ff"] + sum(R for _, R, _ in ms))
        two = 2 if case.get("hp") else 1
        return {"bytes": n * w * 17 // 64 + io, "flops": 2 * n * M * two * w}
    if kind == "mlp":
        c, M = CLASSES[case["cls"]], case["M"]
        H, F = c["hidden"], c["ff"]
        return {"bytes": 3 * H * F * 17 // 64 + M * 4 * 4 * H + 4 * (2 * H + F), "flops": 6 * M * H * F}
    if kind == "chunk":
        c, M = CLASSES[case["cls"]], case["M"]
        H, F = c["hidden"], c["ff"]
        return {"bytes": 2 * H * F * 65 // 64 + M * (H + F) * 6, "flops": 4 * M * H * F}
    if kind == "moe":
        M, E, k, H, F = (case[n] for n in ("M", "E", "k", "H", "F"))
        hit = E * (1.0 - (1.0 - k / E) ** M)       # experts that M tokens touch, on average
        return {"bytes": int(hit * 2 * H * F * 17 / 16 + M * 8 * H + M * E * 4), "flops": 4 * M * k * H * F}
    M, R, C = case["M"], case["R"], case["C"]
    return {"bytes": R * C * 17 // 16 + M * 4 * (R + C), "flops": 2 * M * R * C}


# ------------------------------------------------------------------------------------------------ 64-bit results
def tolerance(case):
    kind = case["kind"]
    return {
        # fp32 sums of exact integer unit values in another order (1e-7 to 2e-7 from the 64-bit sums)
        "products": {"rel": 1e-6, "max": 1e-5},
        "prompt": {"rel": 1e-6, "max": 1e-5},
        "q8": {"rel": 1e-6, "max": 1e-5},
        # the intermediate rows are rounded to int8 again: last-bit differences move a few of them by one step
        "mlp": {"rel": 2e-3, "max": 3e-2},
        "moe": {"rel": 1e-3, "max": 3e-2},
        # rounded to int8 four times a layer, and a layer's moved values move the next layer's
        "step": {"rel": 6e-2, "max": 4e-1},
        # fp16 outputs
        "chunk": {"rel": 1e-3, "max": 1e-2},
    }[kind]


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _div(a, b):
    """a / b rounded once in fp32 (torch multiplies by a reciprocal where an operand is a Python number)"""
    one = torch.ones_like(a if isinstance(a, torch.Tensor) else b)
    return (a * one) / (b * one)


def _round_q(x64, amax):
    """the int8 rows as the format defines them: fp32 x times fp32 (127 / amax), to the nearest, ties to even"""
    a = amax.float()
    inv = torch.where(a > 0, _div(127.0, torch.where(a > 0, a, torch.ones_like(a))), torch.zeros_like(a))
    return torch.round(x64.float() * inv).double()


def _quant64(x64, hp=None):
    """rows rounded to int8 a 128-column group, times their scales; hp: with the residual's row added"""
    M, C = x64.shape
    x = x64.float().reshape(M, C // 128, 128)
    amax = x.abs().amax(dim=2, keepdim=True)
    q = _round_q(x, amax)
    y = q * (amax.double() / 127.0)
    if hp:
        r = (x.double() - q * _div(amax, 127.0).double()).float()
        a2 = _div(amax, 254.0)
        q2 = _round_q(r, a2).clamp(-127, 127)
        y = y + q2 * (a2.double() / 127.0)
    return y.reshape(M, C)


def _fold64(x64, HB):
    M, C = x64.shape
    h = torch.ones((1, 1), dtype=torch.float64, device=x64.device)
    while h.shape[0] < HB:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x64.reshape(M * C // HB, HB) @ h).reshape(M, C) / math.sqrt(HB)


def _rms64(x64, w, sg, HB):
    xn = x64 / torch.sqrt((x64 * x64).mean(dim=1, keepdim=True) + 1e-6) * w.double()
    return xn, _quant64(_fold64(sg.double() * xn, HB))


def _smfold64(g, u, sg, HB):
    return _quant64(_fold64(sg.double() * (g / (1.0 + torch.exp(-g)) * u), HB))


def _exact_layer(case, seed, hp):
    c, M = CLASSES[case["cls"]], case["M"]
    widths = {"q": 0, "k": 0, "v": 0, "o": 1, "gate": 2, "up": 2, "down": 3}
    xs = [_quant64(_rows(M, C, seed, 20 + i), hp) for i, C in enumerate((c["hidden"],) * 3 + (c["ff"],))]
    return {n: xs[widths[n]] @ _tern64(R, C, seed, i).t() for i, (n, R, C) in enumerate(_mats(case))}


def _exact_products(case, seed):
    return _exact_layer(case, seed, case["hp"])


def _exact_prompt(case, seed):
    return _exact_layer(case, seed, False)


def _exact_step(case, seed):
    c, M, n = CLASSES[case["cls"]], case["M"], case["layers"]
    H, F, HB, HBF = c["hidden"], c["ff"], c["hb"], c["hbf"]
    x = _rows(M, H, seed, 20).double()
    ks, vs = [], []
    for l in range(n):
        w = {m: (R, C, seed, 100 * l + i) for i, (m, R, C) in enumerate(_mats(case))}
        sg = [_signs(d, seed, 100 * l + 30 + j) for j, d in enumerate((H, H, H, F))]
        nw = [_norm_w(H, seed, 100 * l + 40 + j) for j in range(2)]
        _, a = _rms64(x, nw[0], sg[0], HB)
        q = a @ _tern64(*w["q"]).t()
        ks.append(a @ _tern64(*w["k"]).t())
        vs.append(a @ _tern64(*w["v"]).t())
        x = x + _quant64(_fold64(sg[1].double() * q, HB)) @ _tern64(*w["o"]).t()
        _, a = _rms64(x, nw[1], sg[2], HB)
        x = x + _smfold64(a @ _tern64(*w["gate"]).t(), a @ _tern64(*w["up"]).t(), sg[3], HBF) @ _tern64(*w["down"]).t()
    xn, _ = _rms64(x, _norm_w(H, seed, 51), _signs(H, seed, 50), HB)
    return dict(x=x, xn=xn, k=ks, v=vs)


def _exact_mlp(case, seed):
    c, M = CLASSES[case["cls"]], case["M"]
    H, F = c["hidden"], c["ff"]
    w = {m: (R, C, seed, i) for i, (m, R, C) in enumerate(_mats(case))}
    xw = _rows(M, H, seed, 20).double() + _rows(M, H, seed, 21).double()
    _, a = _rms64(xw, _norm_w(H, seed, 40), _signs(H, seed, 30), c["hb"])
    h = _smfold64(a @ _tern64(*w["gate"]).t(), a @ _tern64(*w["up"]).t(), _signs(F, seed, 31), c["hbf"])
    return dict(xw=xw, y=h @ _tern64(*w["down"]).t())


def _exact_chunk(case, seed):
    c, M = CLASSES[case["cls"]], case["M"]
    H, F = c["hidden"], c["ff"]
    out = {}
    for i, (n, R, C) in enumerate(_mats(case)):
        if n in ("up", "down"):
            x = _rows(M, C, seed, 20 if n == "up" else 21)
            amax = x.abs().amax(dim=1, keepdim=True)
            out[n] = (_round_q(x, amax) * (amax.double() / 127.0)) @ _tern64(R, C, seed, i).t()
    return out


def _quant8_64(x):
    """rows rounded to int8 a 32-column block, times their fp16 scales"""
    M, C = x.shape
    x = x.float().reshape(M, C // 32, 32)
    amax = x.abs().amax(dim=2, keepdim=True)
    return (_round_q(x, amax) * _div(amax, 127.0).to(torch.float16).double()).reshape(M, C)


def _exact_moe(case, seed):
    M, E, k, H, F = (case[n] for n in ("M", "E", "k", "H", "F"))
    lg = _logits(M, E, seed).double()
    if case["score"] == "sigmoid":
        s = torch.sigmoid(lg)
        ids = (s + _bias(E, seed).double()).topk(k, dim=1).indices
        gw = s.gather(1, ids)
        gw = gw / gw.sum(dim=1, keepdim=True) * ROUTE_SCALE
    else:
        top, ids = lg.topk(k, dim=1)
        gw = torch.softmax(top, dim=1)
    x = _rows(M, H, seed, 20)
    xq, y = _quant8_64(x), x.double()
    for e in ids.unique().tolist():
        t, j = (ids == e).nonzero(as_tuple=True)
        u = (xq[t] @ _q8_64(F, H, seed, 100 + e).t()).clamp(min=0.0)
        yd = _quant8_64(u * u) @ _q8_64(H, F, seed, 400 + e).t()
        y.index_add_(0, t, gw[t, j].unsqueeze(1) * yd)
    return y


def _exact_q8(case, seed):
    R, C = case["R"], case["C"]
    return _quant8_64(_rows(case["M"], C, seed, 20)) @ _q8_64(R, C, seed, 0).t()
