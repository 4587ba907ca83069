"""Performance cases of the decode hot path: the work a program that uses `pck` has it do.

Each case is a dict of plain values.  `prepare` makes what such a program holds before the call
(weights, checkers, packed weights, a captured decode graph), `run` is one pass through the public
entry points, `work` the bytes and operations the pass cannot do without, `exact` its results in
64 bits by plain torch.  Kinds:

  gemv       one product y = W x: BF16 weights in the coalesced or the naive tree, E4M3FN weights
             with the row scales applied in the same launch; any row length
  layer      decode layers at batch 1 (q/k/v, o, gate/up, down), every output checked, captured
             in a graph as a decode loop runs them: the checks carried by later launches
             (CarriedChecker) or one standalone launch per layer (check_many)
  blayer     one decode layer for a batch of rows on the matrix cores (packed weights) with every
             output column checked, captured in a graph
  batched    one batched product and its check, called eagerly; row lengths without a packed
             route included
  member     the sampled-token membership check of a decode step's logits
  sampling   the top-k / top-p set check
"""

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "proof-carrying-kernels_amd"))

from pck import tree_height  # noqa: E402
from pck import cuda as pc  # noqa: E402
from pck.member import check_members  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # The smallest call: one k or v projection of a decode step, called eagerly; latency.
        {"name": "kv_bf16", "kind": "gemv", "dtype": "bf16", "tree": "coalesced", "m": 1024,
         "n": 4096, "threads": 256},
        # A projection whose rows are no whole number of 16-byte vectors (a pruned width).
        {"name": "ragged_bf16", "kind": "gemv", "dtype": "bf16", "tree": "coalesced", "m": 14336,
         "n": 4100, "threads": 256},
        # FP8 weights with their row scales, rows of 8-byte multiples only (no 16-byte vectors).
        {"name": "ragged_fp8", "kind": "gemv", "dtype": "fp8", "tree": "coalesced", "m": 28672,
         "n": 4104, "threads": 256},
        # The second GEMV kernel of the detection campaign.
        {"name": "naive_bf16", "kind": "gemv", "dtype": "bf16", "tree": "naive", "m": 14336,
         "n": 4096, "threads": 256},
        # The headline: batch-1 decode, BF16, checks carried by the next layer's launches.
        {"name": "layers_bf16", "kind": "layer", "dtype": "bf16", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "layers": 2, "block": 128, "check": "carried"},
        # The same with FP8 weights and row scales; one standalone check launch per layer, as a
        # caller that needs each layer's verdict before the next one asks for.
        {"name": "layers_fp8", "kind": "layer", "dtype": "fp8", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "layers": 2, "block": 128, "check": "standalone"},
        # A serving batch of 128 requests, BF16.
        {"name": "blayer_bf16_b128", "kind": "blayer", "dtype": "bf16", "hidden": 4096,
         "kv": 1024, "ffn": 14336, "block": 128, "batch": 128},
        # The largest: 256 requests, FP8 weights.
        {"name": "blayer_fp8_b256", "kind": "blayer", "dtype": "fp8", "hidden": 4096,
         "kv": 1024, "ffn": 14336, "block": 128, "batch": 256},
        # A small ragged batch and a row length without a packed route.
        {"name": "batched_ragged", "kind": "batched", "dtype": "bf16", "m": 4096, "n": 3000,
         "block": 128, "batch": 24},
        # Verifying a decode step's sampled tokens for a full serving batch.
        {"name": "member_b256", "kind": "member", "rows": 256, "vocab": 151936, "logits": "fp32",
         "top_k": True, "top_p": True, "greedy": False},
        # The same for a few requests without a top-k, some of them greedy, BF16 logits.
        {"name": "member_b4", "kind": "member", "rows": 4, "vocab": 151936, "logits": "bf16",
         "top_k": False, "top_p": True, "greedy": True},
        # A top-p sampler's selected sets, judged by the set checker.
        {"name": "sampling_topp_b64", "kind": "sampling", "rows": 64, "vocab": 151936,
         "top_p": True, "k": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _to(v, q):
    return max(q, v // q * q)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "layer", "blayer", "batched", "member", "sampling"])
    if kind == "gemv":
        dtype = rng.choice(["bf16", "fp8"])
        tree = "naive" if dtype == "bf16" and rng.random() < 0.3 else "coalesced"
        n = _to(_log(rng, 1024, 16384), rng.choice([1, 2, 4, 8, 16, 128]))
        m = _log(rng, 512, min(32768, 120_000_000 // n))
        threads = rng.choice([64, 128, 256, 256, 512, 1024])
        return {"kind": kind, "dtype": dtype, "tree": tree, "m": m, "n": n, "threads": threads}
    if kind in ("layer", "blayer"):
        hidden = _to(_log(rng, 1024, 4096), 128)
        case = {"kind": kind, "dtype": rng.choice(["bf16", "fp8"]), "hidden": hidden,
                "kv": rng.choice([256, 512, 1024]), "ffn": _to(int(hidden * rng.uniform(2.5, 3.5)), 256),
                "block": rng.choice([64, 128])}
        if kind == "layer":
            case["layers"] = rng.choice([1, 2])
            case["check"] = rng.choice(["carried", "standalone"])
        else:
            case["batch"] = _log(rng, 16, 256)
        return case
    if kind == "batched":
        n = _to(_log(rng, 1024, 3072), rng.choice([4, 8, 128]))
        m = _to(_log(rng, 512, 5_000_000 // n), 64)
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp8"]), "m": m, "n": n, "block": 64,
                "batch": _log(rng, 16, 64)}
    rows = _log(rng, 1, 256)
    vocab = rng.randint(32000, 152000)
    if kind == "member":
        top_k = rng.random() < 0.6
        return {"kind": kind, "rows": rows, "vocab": vocab, "logits": rng.choice(["fp32", "fp32", "bf16"]),
                "top_k": top_k, "top_p": not top_k or rng.random() < 0.7, "greedy": rng.random() < 0.3}
    top_p = rng.random() < 0.5
    return {"kind": kind, "rows": rows, "vocab": vocab, "top_p": top_p,
            "k": 0 if top_p else rng.choice([1, 20, 50, 200])}


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _weights(m, n, g):
    return (torch.randn((m, n), generator=g, device=DEV) * 0.02).bfloat16()


def _acts(shape, g):
    return torch.randn(shape, generator=g, device=DEV).bfloat16()


def _layer_shapes(case):
    """(rows of each grouped product, columns) of a decode layer's four launches."""
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [([h, kv, kv], h), ([h], h), ([f, f], h), ([h], f)]


def _checker(W, block, height, seed):
    cpu = torch.Generator()
    cpu.manual_seed(int(seed) + 5)
    return pc.GpuBlockedChecker(W.bfloat16(), block, height, generator=cpu)


def _draw_gemv(case, seed):
    g = _gen(seed)
    return _weights(case["m"], case["n"], g), _acts((case["n"],), g)


def _draw_layers(case, seed):
    g = _gen(seed)
    layers = []
    for _ in range(case["layers"]):
        layers.append([([_weights(m, n, g) for m in ms], _acts((n,), g)) for ms, n in _layer_shapes(case)])
    return layers


def _draw_blayer(case, seed):
    """The grouped products' weights are one matrix each, as a serving program stores them."""
    g = _gen(seed)
    return [(_weights(sum(ms), n, g), _acts((case["batch"], n), g)) for ms, n in _layer_shapes(case)]


def _draw_batched(case, seed):
    g = _gen(seed)
    return _weights(case["m"], case["n"], g), _acts((case["batch"], case["n"]), g)


def _draw_logits(case, seed):
    """N(0, 3) logits with a few hot tokens per row."""
    g = _gen(seed)
    B, V = case["rows"], case["vocab"]
    logits = torch.randn((B, V), generator=g, device=DEV) * 3
    hot = torch.randint(0, V, (B, 5), generator=g, device=DEV)
    logits.scatter_add_(1, hot, 6 + 6 * torch.rand((B, 5), generator=g, device=DEV))
    return logits, g


def _draw_member(case, seed):
    logits, g = _draw_logits(case, seed)
    B, V = logits.shape
    if case["logits"] == "bf16":
        logits = logits.bfloat16()
    # the sampler's tokens: Gumbel-max over the 20 largest, 1% replaced by tokens outside the set
    v, idx = logits.float().topk(20, dim=1)
    u = torch.rand(v.shape, generator=g, device=DEV).clamp_min(1e-20)
    pick = (v - torch.log(-torch.log(u))).argmax(1, keepdim=True)
    tokens = idx.gather(1, pick).squeeze(1)
    bad = torch.rand(B, generator=g, device=DEV) < 0.01
    tokens = torch.where(bad, torch.randint(0, V, (B,), generator=g, device=DEV), tokens)
    greedy = None
    if case["greedy"]:
        greedy = torch.arange(B, device=DEV) % 4 == 3
        tokens = torch.where(greedy, logits.argmax(1), tokens)
    top_k = torch.full((B,), 50, dtype=torch.int64, device=DEV) if case["top_k"] else None
    top_p = torch.full((B,), 0.9, dtype=torch.float64, device=DEV) if case["top_p"] else None
    return logits, tokens, top_k, top_p, greedy


def _draw_sampling(case, seed):
    logits, _ = _draw_logits(case, seed)
    if not case["top_p"]:
        return logits, logits.topk(case["k"], dim=1).indices.contiguous(), None
    # a serving sampler keeps at most 1024 candidates: the nucleus of a temperature-0.7 softmax
    order = logits.topk(1024, dim=1).indices.contiguous()
    w = (logits.double() / 0.7 - logits.double().amax(1, keepdim=True) / 0.7).exp()
    c = w.gather(1, order).cumsum(1) / w.sum(1, keepdim=True)
    lengths = ((c < 0.9).sum(1) + 1).clamp(max=1024)
    return logits, order, lengths


# ---- one pass -------------------------------------------------------------------------------


def _gemv_pass(case, s):
    if case["tree"] == "naive":
        return pc.gemv_naive(s["W"], s["x"], case["threads"])
    if case["dtype"] == "bf16":
        return pc.gemv_coalesced(s["W"], s["x"], case["threads"])
    return pc.gemv_fp8_scaled(s["W"], s["x"], s["scale"], case["threads"])


def _layer_pass(case, layers):
    fp8 = case["dtype"] == "fp8"
    carrier = pc.CarriedChecker() if case["check"] == "carried" else None
    out, pending = [], []
    for layer in layers:
        items = []
        for Ws, x, scales, checkers in layer:
            if fp8:
                triples = [(W, x, s) for W, s in zip(Ws, scales)]
                if carrier is not None:
                    zs, ys = carrier.gemv_group_fp8_scaled(triples)
                else:
                    zs, ys, _ = pc.gemv_group_fp8_scaled(triples)
                out += ys
            else:
                pairs = [(W, x) for W in Ws]
                zs = carrier.gemv_group(pairs) if carrier is not None else pc.gemv_group(pairs)
            out += zs
            items += [(ch, x, z) for ch, z in zip(checkers, zs)]
        pending += carrier.check_many(items) if carrier is not None else pc.check_many(items)
    if carrier is not None:
        carrier.flush()
        pending = [p.result() for p in pending]
    return out + _checks(pending)


def _checks(results):
    """All verdicts, rhos and taus, each kind as one flat tensor."""
    return [torch.cat([getattr(r, f).reshape(-1) for r in results]) for f in ("passed", "rho", "tau")]


def _blayer_pass(products):
    items = []
    for packed, X, checker in products:
        items.append((checker, X, pc.gemm_batched(packed, X)))
    return [Y for _, _, Y in items] + _checks(pc.check_batched(items))


def _captured(step):
    """The step run once eagerly, then captured: (graph, its output buffers)."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return {"graph": graph, "out": out}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        W, x = _draw_gemv(case, seed)
        s = {"case": case, "W": W, "x": x}
        if case["dtype"] == "fp8":
            s["W"], s["scale"] = pc.quantize_fp8(W)
        return s
    if kind == "layer":
        layers = []
        vec = 16 if case["dtype"] == "fp8" else 8
        for layer in _draw_layers(case, seed):
            launches = []
            for i, (Ws, x) in enumerate(layer):
                scales = None
                if case["dtype"] == "fp8":
                    Ws, scales = zip(*[pc.quantize_fp8(W) for W in Ws])
                height = tree_height(x.numel(), 256, vec)
                checkers = [_checker(W, case["block"], height, seed + i) for W in Ws]
                launches.append((Ws, x, scales, checkers))
            layers.append(launches)
        return {"case": case, "layers": layers, **_captured(lambda: _layer_pass(case, layers))}
    if kind in ("blayer", "batched"):
        drawn = _draw_blayer(case, seed) if kind == "blayer" else [_draw_batched(case, seed)]
        products = []
        for i, (W, X) in enumerate(drawn):
            W = pc.quantize_fp8(W)[0] if case["dtype"] == "fp8" else W
            checker = _checker(W, case["block"], pc.batched_height(W.shape[1]), seed + i)
            products.append((pc.pack_batched_weights(W), X, checker))
        s = {"case": case, "products": products}
        if kind == "blayer":
            s.update(_captured(lambda: _blayer_pass(products)))
        return s
    if kind == "member":
        logits, tokens, top_k, top_p, greedy = _draw_member(case, seed)
        host = None if top_k is None else top_k.cpu().numpy()
        return {"case": case, "args": (logits, tokens, top_k, top_p, greedy), "host": host}
    logits, selected, lengths = _draw_sampling(case, seed)
    return {"case": case, "logits": logits, "selected": selected, "lengths": lengths}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        return _gemv_pass(case, state)
    if kind in ("layer", "blayer"):
        state["graph"].replay()
        return state["out"]
    if kind == "batched":
        return _blayer_pass(state["products"])
    if kind == "member":
        return check_members(*state["args"], top_k_host=state["host"])
    if case["top_p"]:
        r = pc.check_topp_gpu(state["logits"], state["selected"], state["lengths"], 0.9, 0.7)
    else:
        r = pc.check_topk_gpu(state["logits"], state["selected"], case["k"])
    return [r.passed, r.min_selected, r.max_rejected, r.mass, r.mass_without_smallest]


# ---- what a pass cannot do without ----------------------------------------------------------


def _product(m, n, batch, fp8, scaled=False):
    b = m * n * (1 if fp8 else 2) + 2 * n * batch + 4 * m * batch + (8 * m if scaled else 0)
    return b, 2.0 * m * n * batch


def _check_work(m, n, batch, block):
    """The bank (c FP32, a BF16 per block and column), signs, activations, outputs, results."""
    nb = m // block
    b = 6 * nb * n + m + 2 * n * batch + 4 * m * batch + 17 * nb * batch
    return b, batch * (4.0 * nb * n + 4.0 * m)


def work(case):
    kind = case["kind"]
    total = [0.0, 0.0]

    def add(w):
        total[0] += w[0]
        total[1] += w[1]

    fp8 = case.get("dtype") == "fp8"
    if kind == "gemv":
        add(_product(case["m"], case["n"], 1, fp8, scaled=fp8))
    elif kind in ("layer", "blayer"):
        B = case.get("batch", 1)
        for _ in range(case.get("layers", 1)):
            for ms, n in _layer_shapes(case):
                for m in [sum(ms)] if kind == "blayer" else ms:
                    add(_product(m, n, B, fp8, scaled=fp8 and kind == "layer"))
                    add(_check_work(m, n, B, case["block"]))
    elif kind == "batched":
        add(_product(case["m"], case["n"], case["batch"], fp8))
        add(_check_work(case["m"], case["n"], case["batch"], case["block"]))
    else:
        B, V = case["rows"], case["vocab"]
        size = 2 if case.get("logits") == "bf16" else 4
        add((B * V * size + 64 * B, 3.0 * B * V))
    return {"bytes": total[0], "flops": total[1]}


def tolerance(case):
    """FP32 sums of up to 16384 products are 0.7e-7 to 1.1e-7 off the 64-bit result, and two
    orders differ by up to twice that: 1e-6.  rho is the rounding of y itself, so it compares at
    all only because the order of every y is part of the interface (the outputs equal the CPU
    model bit for bit).  The sampling checks sum FP32 exponentials in FP64: up to 1e-7 (2 ulp)
    where the few largest terms decide."""
    return {"rel": 4e-7} if case["kind"] in ("member", "sampling") else {"rel": 1e-6}


# ---- the same in 64 bits --------------------------------------------------------------------


def _quantized(W):
    """(codes as FP64 values, FP32 row scales) of W at E4M3FN."""
    amax = W.abs().amax(dim=1).float()
    s = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    return (W.float() / s[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double(), s


def _passes(outs, block):
    """Every block of honest outputs passes; rho and tau have no 64-bit value of their own."""
    count = sum(y.numel() // block for y in outs)
    return [torch.ones(count, dtype=torch.bool, device=DEV), None, None]


def exact(case, seed):
    kind = case["kind"]
    fp8 = case.get("dtype") == "fp8"
    if kind == "gemv":
        W, x = _draw_gemv(case, seed)
        if not fp8:
            return W.double() @ x.double()
        Q, s = _quantized(W)
        z = Q @ x.double()
        return z, s.double() * z
    if kind == "layer":
        out, zs = [], []
        for layer in _draw_layers(case, seed):
            for Ws, x in layer:
                if fp8:
                    pairs = [_quantized(W) for W in Ws]
                    z = [Q @ x.double() for Q, _ in pairs]
                    out += [s.double() * v for (_, s), v in zip(pairs, z)]
                else:
                    z = [W.double() @ x.double() for W in Ws]
                out += z
                zs += z
        return out + _passes(zs, case["block"])
    if kind in ("blayer", "batched"):
        drawn = _draw_blayer(case, seed) if kind == "blayer" else [_draw_batched(case, seed)]
        out = []
        for W, X in drawn:
            W64 = _quantized(W)[0] if fp8 else W.double()
            out.append(X.double() @ W64.t().contiguous())
        return out + _passes(out, case["block"])
    if kind == "member":
        logits, tokens, top_k, top_p, greedy = _draw_member(case, seed)
        l = logits.double()
        lt = l.gather(1, tokens[:, None])
        above = (l > lt).sum(1)
        limit = top_k if top_k is not None else torch.full_like(tokens, l.shape[1])
        limit = limit if greedy is None else torch.where(greedy, torch.ones_like(limit), limit)
        ok = above < limit
        mass = torch.zeros(l.shape[0], dtype=torch.float64, device=DEV)
        if top_p is not None:
            kept = l >= l.topk(50, dim=1).values[:, -1:] if top_k is not None else torch.ones_like(l, dtype=torch.bool)
            e = torch.where(kept, (l - l.amax(1, keepdim=True)).exp(), torch.zeros_like(l))
            mass = torch.where(l > lt, e, torch.zeros_like(e)).sum(1) / e.sum(1)
            within = mass < top_p + 1e-4
            ok &= within if greedy is None else within | greedy
        return {"ok": ok, "above": above, "mass_above": mass}
    logits, selected, lengths = _draw_sampling(case, seed)
    l = logits.double()
    B, L = selected.shape
    live = torch.ones_like(selected, dtype=torch.bool)
    if lengths is not None:
        live = torch.arange(L, device=DEV)[None] < lengths[:, None]
    inside = torch.zeros_like(l, dtype=torch.bool).scatter_(1, selected, live)
    inf = torch.full_like(l, math.inf)
    low = torch.where(inside, l, inf).amin(1)
    high = torch.where(inside, -inf, l).amax(1)
    ok = low >= high
    mass = torch.zeros(B, dtype=torch.float64, device=DEV)
    without = mass.clone()
    if case["top_p"]:
        e = ((l - l.amax(1, keepdim=True)) / 0.7).exp()
        z = e.sum(1)
        sel = torch.where(inside, e, torch.zeros_like(e)).sum(1)
        mass = sel / z
        without = (sel - ((low - l.amax(1)) / 0.7).exp()) / z
        ok &= (mass >= 0.9 - 1e-6) & (without < 0.9 + 1e-6)
        mass, without = torch.where(ok | (low >= high), mass, 0 * mass), torch.where(ok | (low >= high), without, 0 * without)
    return [ok, low.float(), high.float(), mass, without]
