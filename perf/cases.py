"""What this library's speed is measured on: the calls its users make, over the sizes they make them at.

Sizes are those of the repository's own benchmark and tests (hidden 2048, expert width 768, top 8 of 128 experts,
32 query / 4 kv heads of 128, vocabulary 151936) and generic odd ones around them.  Each kind of case:

  linear    prequant -> lin_pq of one to sixteen rows, over several layers' weights: the projections and the head
            of a decode step (captured in a HIP graph, as a decode loop runs them)
  forward   the one-call linear with its own activation quantization: prompts of 17 to 4096 tokens
  dropin    prequant -> moe_gateup -> moe_down -> moe_combine over host pointer lists, several layers (graph)
  batch     route_topk -> prequant -> the two-launch MoE of a batched decode or speculative-verify step (graph)
  prefill   route_topk -> moe_compute: the MoE of a prompt of one to 4096 tokens
  attn      kv_write -> attn_decode over one layer's FP8 cache after another (graph)
  stack     decode_stack: every MoE layer of a one-token step in one launch
  step      a whole decode step (embedding to logits) of a few layers, captured as its users capture it

The layers of one case take their own inputs (they are not chained), so a result shows one layer's rounding;
`stack` and `step` are chains.
"""
import math

import torch

from moe_fused_inference_amd import get_decode_ext, get_ext, moe_layer
from moe_fused_inference_amd.decode_step import DecodeStep, ModelConfig, synthetic_model

DEV = "cuda"
BLOCK = 32
MAGS = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
MIDS = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # o_proj of a one-token step: the smallest dense call, bound by latency
        {"name": "proj_one_token", "kind": "linear", "M": 1, "N": 2048, "K": 4096, "layers": 64},
        # the vocabulary head of a batch-8 step: the largest weight of a step
        {"name": "head_batch8", "kind": "linear", "M": 8, "N": 151936, "K": 2048, "layers": 2},
        # a short prompt through a layer of odd sizes
        {"name": "forward_ragged", "kind": "forward", "M": 333, "N": 1000, "K": 2080, "dtype": "float16"},
        # a long prompt through a large projection
        {"name": "forward_4096", "kind": "forward", "M": 4096, "N": 4096, "K": 2048, "dtype": "bfloat16"},
        # one token through the reference's own operators
        {"name": "dropin_one_token", "kind": "dropin", "M": 1, "E": 8, "n": 128, "H": 2048, "Mi": 768, "layers": 16},
        # speculative verify: one token and eight drafts
        {"name": "verify_9", "kind": "batch", "M": 9, "E": 8, "n": 128, "H": 2048, "Mi": 768, "zipf": 0.5, "layers": 4},
        # a short prompt: every expert is read for a handful of tokens
        {"name": "prefill_100", "kind": "prefill", "T": 100, "E": 8, "n": 128, "H": 2048, "Mi": 768, "zipf": 0.0},
        # a long prompt
        {"name": "prefill_2048", "kind": "prefill", "T": 2048, "E": 8, "n": 128, "H": 2048, "Mi": 768, "zipf": 0.0},
        # attention of a one-token step at the benchmark's context
        {"name": "attn_4k", "kind": "attn", "M": 1, "Hkv": 4, "G": 8, "ctx": 4095, "layers": 16},
        # attention of a verify step over a long document
        {"name": "attn_long_verify", "kind": "attn", "M": 9, "Hkv": 4, "G": 8, "ctx": 23001, "layers": 4},
        # all MoE layers of a one-token step whose routing is drawn ahead
        {"name": "stack_16", "kind": "stack", "layers": 16, "E": 8, "n": 128, "H": 2048, "Mi": 768, "strict": False},
        # a whole batch-8 step
        {"name": "step_batch8", "kind": "step", "M": 8, "layers": 2, "n": 128, "E": 8, "Mi": 768, "vocab": 151936,
         "ctx": 3000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    """A multiple of step, spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, _log(rng, lo, hi) // step * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "forward", "forward", "dropin", "batch", "prefill", "prefill", "attn",
                       "attn", "stack", "step"])
    if kind == "linear":
        if rng.random() < 0.3:
            return {"kind": kind, "M": rng.randint(1, 16), "N": _log(rng, 8192, 151936), "K": rng.choice([1024, 2048]),
                    "layers": 2}
        n, k = rng.choice([(5120, 2048), (2048, 4096), (128, 2048), (_log(rng, 64, 8192), _log(rng, 100, 4096))])
        return {"kind": kind, "M": rng.randint(1, 16), "N": n, "K": k, "layers": rng.choice([8, 32])}
    if kind == "forward":
        return {"kind": kind, "M": _log(rng, 17, 4096), "N": _log(rng, 128, 4096),
                "K": rng.choice([768, 2048, _log(rng, 256, 2048)]), "dtype": rng.choice(["bfloat16", "float16"])}
    E = rng.choice([8, 8, rng.randint(1, 8)])
    n = rng.choice([128, 60, rng.randint(8, 128)])
    if kind == "dropin":
        H, Mi = rng.choice([(2048, 768), (_log(rng, 256, 2048), _log(rng, 96, 1024))])
        return {"kind": kind, "M": rng.randint(1, 9), "E": E, "n": n, "H": H, "Mi": Mi, "layers": rng.randint(2, 8)}
    if kind == "batch":
        H, Mi = rng.choice([(2048, 768), (_mult(rng, 256, 4096, 128), _mult(rng, 96, 1536, 32))])
        return {"kind": kind, "M": rng.randint(1, 16), "E": E, "n": n, "H": H, "Mi": Mi,
                "zipf": rng.choice([0.0, 0.5, 1.0]), "layers": rng.randint(1, 3)}
    if kind == "prefill":
        H, Mi = rng.choice([(2048, 768), (2048, 768), (_mult(rng, 256, 2048, 32), _mult(rng, 96, 1024, 32))])
        return {"kind": kind, "T": _log(rng, 1, 2048), "E": E, "n": n, "H": H, "Mi": Mi,
                "zipf": rng.choice([0.0, 0.5, 1.0])}
    if kind == "attn":
        hkv, g = rng.choice([(4, 8), (4, 8), (8, 4), (2, 2), (1, 16), (8, 1)])
        return {"kind": kind, "M": rng.choice([1, rng.randint(2, 16)]), "Hkv": hkv, "G": g,
                "ctx": _log(rng, 20, 24000), "layers": rng.randint(1, 4)}
    if kind == "stack":
        return {"kind": kind, "layers": rng.randint(2, 12), "E": E, "n": n, "H": rng.choice([512, 1024, 2048, 2048]),
                "Mi": rng.choice([768, _mult(rng, 96, 1024, 32)]), "strict": rng.random() < 0.3}
    return {"kind": "step", "M": rng.choice([1, rng.randint(2, 16)]), "layers": rng.randint(1, 2), "n": rng.choice([32, 128]), "E": 8,
            "Mi": 768, "vocab": rng.choice([32000, 151936]), "ctx": _log(rng, 100, 4000)}


# ------------------------------------------------------------------ inputs
def _codes(x):
    """MXFP4 of rows (.., K), K a multiple of 32: E2M1 codes (.., K) and block exponents (.., K/32)."""
    b = x.reshape(*x.shape[:-1], -1, BLOCK)
    am = b.abs().amax(-1)
    m, q = torch.frexp(am)
    e = torch.where(m <= 0.75, q - 3, q - 2).clamp(-127, 127)
    e = torch.where(am > 0, e, torch.zeros_like(e))
    s = torch.ldexp(b, -e.unsqueeze(-1))
    mag = torch.bucketize(s.abs(), torch.tensor(MIDS, dtype=x.dtype, device=x.device), right=True, out_int32=True)
    code = (mag + 8 * (s < 0)).to(torch.uint8)
    return code.reshape(x.shape), e


def _pad(x):
    k = x.shape[-1]
    return torch.nn.functional.pad(x, (0, -k % BLOCK)) if k % BLOCK else x


def _pack(x):
    code, e = _codes(_pad(x))
    return code[..., 0::2] | (code[..., 1::2] << 4), (e + 127).to(torch.uint8)


def _weight(g, n, k, std=0.02):
    """Packed MXFP4 of a bf16 N(0, std) weight of n rows."""
    kp = (k + BLOCK - 1) // BLOCK * BLOCK
    wp = torch.empty((n, kp // 2), dtype=torch.uint8, device=DEV)
    ws = torch.empty((n, kp // BLOCK), dtype=torch.uint8, device=DEV)
    step = max(1, (64 << 20) // kp)
    for r in range(0, n, step):
        c = min(step, n - r)
        wp[r:r + c], ws[r:r + c] = _pack((torch.randn((c, k), generator=g, device=DEV) * std).bfloat16().float())
    return wp, ws


def _experts(g, c):
    p = {}
    for nm, (n, k) in (("gate", (c["Mi"], c["H"])), ("up", (c["Mi"], c["H"])), ("down", (c["H"], c["Mi"]))):
        wp, ws = _weight(g, c["n"] * n, k)
        p[nm + "_wp"], p[nm + "_ws"] = wp.view(c["n"], n, -1), ws.view(c["n"], n, -1)
    return p


def _rows(g, m, k, dtype=torch.bfloat16):
    """Normed activations: N(0, 1) with a few outliers."""
    x = torch.randn((m, k), generator=g, device=DEV)
    x[torch.rand((m, k), generator=g, device=DEV) < 0.005] *= 4.0
    return x.to(dtype)


def _logits(g, c, m):
    """Router logits of m tokens: N(0, 1), with `zipf` times a skewed preference of the experts."""
    order = torch.randperm(c["n"], generator=g, device=DEV)
    skew = -1.1 * torch.log(torch.arange(1, c["n"] + 1, device=DEV, dtype=torch.float32))
    return torch.randn((m, c["n"]), generator=g, device=DEV) + c.get("zipf", 0.0) * skew[order]


def _inputs(c, seed):
    """The inputs of a case, from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    kind, d = c["kind"], {}
    L = range(c.get("layers", 1))
    c = dict(c, E=min(c["E"], c["n"])) if "n" in c else c
    if kind == "linear":
        d["w"] = [_weight(g, c["N"], c["K"]) for _ in L]
        d["x"] = [_rows(g, c["M"], c["K"]) for _ in L]
    elif kind == "forward":
        d["w"] = _weight(g, c["N"], c["K"])
        d["x"] = _rows(g, c["M"], c["K"], getattr(torch, c["dtype"]))
    elif kind in ("dropin", "stack"):
        m = c.get("M", 1)
        d["experts"] = [_experts(g, c) for _ in L]
        d["x"] = [_rows(g, m, c["H"]) for _ in L]
        pr = [torch.softmax(_logits(g, c, m), -1).topk(c["E"], -1) for _ in L]
        d["ids"] = [p.indices for p in pr]
        d["w"] = [(p.values / p.values.sum(-1, keepdim=True)).contiguous() for p in pr]
    elif kind in ("batch", "prefill"):
        m = c["M"] if kind == "batch" else c["T"]
        d["experts"] = [_experts(g, c) for _ in L]
        d["x"] = [_rows(g, m, c["H"]) for _ in L]
        d["logits"] = [_logits(g, c, m) for _ in L]
    elif kind == "attn":
        M, hkv, hq = c["M"], c["Hkv"], c["Hkv"] * c["G"]
        d["max_pos"] = mp = (c["ctx"] + M + 255) // 256 * 256
        d["q"] = [(torch.randn((M, hq, 128), generator=g, device=DEV)).bfloat16() for _ in L]
        for nm in ("k", "v"):
            d[nm] = [torch.randn((M, hkv, 128), generator=g, device=DEV).bfloat16() for _ in L]
            cache = []
            for _ in L:   # the context's rows as an earlier step's conversion left them; the rest zero
                kv = torch.zeros((mp, hkv, 128), dtype=torch.uint8, device=DEV)
                kv[:c["ctx"]] = torch.randn((c["ctx"], hkv, 128), generator=g, device=DEV).to(
                    torch.float8_e4m3fn).view(torch.uint8)
                cache.append(kv)
            d["kv" + nm] = cache
        d["dpos"] = torch.tensor([c["ctx"]], dtype=torch.int32, device=DEV)
    return d, c


# ------------------------------------------------------------------ the calls
def _captured(fn):
    """fn's launches as a HIP graph, after one eager call."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return {"graph": graph, "out": out}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        cfg = ModelConfig(n_layers=case["layers"], n_experts=case["n"], top_k=case["E"], moe_inter=case["Mi"],
                          vocab=case["vocab"])
        step = DecodeStep(synthetic_model(cfg, seed=seed), cfg, M=case["M"], max_pos=4096)
        step.fill_cache(case["ctx"], seed=seed + 1)
        g = torch.Generator(device=DEV)
        g.manual_seed(seed + 2)
        ids = torch.randint(0, cfg.vocab, (case["M"],), generator=g, device=DEV, dtype=torch.int32)
        step.set_state(ids, case["ctx"])
        graph = step.capture()
        return {"kind": kind, "step": step, "graph": graph, "ids": ids, "ctx": case["ctx"]}
    d, c = _inputs(case, seed)
    st = {"kind": kind, "d": d, "c": c}
    if kind == "forward":
        st["ext"] = get_ext()
        return st
    if kind == "stack":
        st["stack"] = stack = moe_layer.LayerStack([moe_layer.StackedExperts(**e) for e in d["experts"]])
        ids = torch.cat(d["ids"]).int()
        w = torch.cat(d["w"]).contiguous()
        st["ws"] = moe_layer.stack_workspace(c["E"], c["H"], c["Mi"])
        L = len(stack)
        out = [torch.empty(c["H"], dtype=torch.bfloat16, device=DEV),
               torch.empty((L, c["H"]), dtype=torch.bfloat16, device=DEV),
               torch.empty((L, c["H"]), dtype=torch.float32, device=DEV)]
        st["call"] = moe_layer.DecodeStackCall(d["x"][0].reshape(-1), ids, w, stack, out[0], st["ws"], out[1], out[2],
                                               strict=c["strict"])
        st["out"] = out
        return st
    if kind == "prefill":
        st["experts"] = moe_layer.StackedExperts(**d["experts"][0])
        st["ws"] = moe_layer.prefill_workspace(c["T"], c["E"], c["n"], c["H"], c["Mi"])
        return st
    ext = get_decode_ext()
    L = range(c["layers"])
    if kind == "linear":
        def fn():
            out = []
            for l in L:
                xq, xs = ext.prequant(d["x"][l])
                out.append(ext.lin_pq(xq, xs, d["w"][l][0], d["w"][l][1], c["M"], c["N"], c["K"]))
            return out
    elif kind == "dropin":
        M, E, H, Mi = c["M"], c["E"], c["H"], c["Mi"]
        tabs = []
        for l in L:
            p, ids = d["experts"][l], d["ids"][l].tolist()
            gu = [[p[nm + s][e] for m in range(M) for nm in ("gate", "up") for e in ids[m]] for s in ("_wp", "_ws")]
            dn = [[p["down" + s][e] for m in range(M) for e in ids[m]] for s in ("_wp", "_ws")]
            tabs.append((gu, dn))

        def fn():
            out = []
            for l in L:
                gu, dn = tabs[l]
                xq, xs = ext.prequant(d["x"][l])
                h = ext.moe_gateup(xq, xs, gu[0], gu[1], E, M, Mi, H)
                yd = ext.moe_down(h, dn[0], dn[1], E, M, H, Mi)
                out.append(ext.moe_combine(yd, d["w"][l], M))
            return out
    elif kind == "batch":
        st["experts"] = ex = [moe_layer.StackedExperts(**e) for e in d["experts"]]

        def fn():
            out = []
            for l in L:
                ids, w = moe_layer.route_topk(d["logits"][l], c["E"])
                xq, xs = ext.prequant(d["x"][l])
                out.append(moe_layer.decode_batch(xq, xs, ids, w, ex[l]))
            return out
    else:
        hq = c["Hkv"] * c["G"]
        sc = torch.empty((c["M"], hq, d["max_pos"]), dtype=torch.float32, device=DEV)

        def fn():
            out = []
            for l in L:
                ext.kv_write(d["k"][l], d["v"][l], d["kvk"][l], d["kvv"][l], d["dpos"], c["M"])
                out.append(ext.attn_decode(d["q"][l], d["kvk"][l], d["kvv"][l], d["dpos"], sc, c["M"]))
            return out + d["kvk"] + d["kvv"]
    st.update(_captured(fn))
    return st


def run(state):
    kind = state["kind"]
    if kind == "step":
        state["step"].set_state(state["ids"], state["ctx"])
        state["graph"].replay()
        b = state["step"].b
        return [b.logits, b.kvk, b.kvv]
    if kind == "forward":
        return state["ext"].forward(state["d"]["x"], *state["d"]["w"])
    if kind == "stack":
        state["call"]()
        return state["out"]
    if kind == "prefill":
        d = state["d"]
        _, w, topi = moe_layer.route_topk(d["logits"][0], state["c"]["E"], want_int64=True)
        return moe_layer.moe_compute(d["x"][0], topi, w, state["experts"], ws=state["ws"])
    state["graph"].replay()
    return state["out"]


# ------------------------------------------------------------------ what a pass cannot do without
def _wbytes(n, k):
    kp = (k + BLOCK - 1) // BLOCK * BLOCK
    return n * (kp // 2 + kp // BLOCK)


def _distinct(c, tokens):
    """Expected distinct experts of evenly routed tokens (an upper bound where the routing is skewed)."""
    return c["n"] * (1.0 - (1.0 - min(c["E"], c["n"]) / c["n"]) ** tokens)


def _moe_work(c, tokens, experts, abytes, obytes):
    H, Mi, E = c["H"], c["Mi"], min(c["E"], c["n"])
    return {"bytes": experts * (2 * _wbytes(Mi, H) + _wbytes(H, Mi)) + tokens * H * (abytes + obytes),
            "flops": 6.0 * tokens * E * H * Mi}


def work(case):
    c, kind, L = case, case["kind"], case.get("layers", 1)
    if kind in ("linear", "forward"):
        w = {"bytes": _wbytes(c["N"], c["K"]) + c["M"] * (2 * c["K"] + 4 * c["N"]),
             "flops": 2.0 * c["M"] * c["N"] * c["K"]}
    elif kind == "attn":
        M, hkv, hq = c["M"], c["Hkv"], c["Hkv"] * c["G"]
        # the cache once, q, k, v in, the raw scores and o out
        w = {"bytes": 2 * c["ctx"] * hkv * 128 + M * 128 * (2 * hq + 6 * hkv + 4 * hq) + 4 * M * hq * c["ctx"],
             "flops": 4.0 * M * hq * 128 * c["ctx"]}
    elif kind == "step":
        m = dict(c, H=2048)
        w = _moe_work(m, c["M"], _distinct(c, c["M"]), 2, 2)
        w["bytes"] += _wbytes(5120, 2048) + _wbytes(2048, 4096) + _wbytes(c["n"], 2048) + 2 * c["ctx"] * 4 * 128
        w["flops"] += 2.0 * c["M"] * (5120 * 2048 + 2048 * 4096 + c["n"] * 2048) + 4.0 * c["M"] * 32 * 128 * c["ctx"]
        return {"bytes": L * w["bytes"] + _wbytes(c["vocab"], 2048) + 4 * c["M"] * c["vocab"],
                "flops": L * w["flops"] + 2.0 * c["M"] * c["vocab"] * 2048}
    else:
        tokens = c.get("T", c.get("M", 1))
        w = _moe_work(c, tokens, _distinct(c, tokens), 2, 2 if kind == "prefill" else 4)
    return {k: L * v for k, v in w.items()}


def tolerance(case):
    """About four times what measuring against `exact` shows, and no less than what one rounding that falls the other
    way does."""
    return {
        # fp32 sums of exact products: measured 0
        "linear": {"rel": 1e-6},
        "forward": {"rel": 1e-6},
        # measured 1e-7; h is quantized to 4 bits inside, and one h of a token's 6144 that lies beside a threshold and
        # takes the other code moves that token's result by 2e-3
        "dropin": {"rel": 2e-3},
        "batch": {"rel": 2e-3},
        # bf16 results (measured 2.9e-3), h through fp16 and 4 bits
        "prefill": {"rel": 1.2e-2},
        # measured 2e-6
        "attn": {"rel": 1e-5},
        # bf16 activations carried from layer to layer: measured 4.2e-3
        "stack": {"rel": 1.7e-2},
        # MoE outputs moved by one part in a million give the same logits bit for bit; moved further, a bf16 rounding
        # goes the other way and the 4-bit activations of the next layer amplify it
        "step": {"rel": 3e-2, "differ": 1e-3},
    }[case["kind"]]


# ------------------------------------------------------------------ the same in 64 bits
def _value(code, e):
    v = torch.tensor(MAGS, dtype=torch.float64, device=code.device)[(code & 7).long()]
    v = torch.where(code >= 8, -v, v).reshape(*e.shape, BLOCK)
    return torch.ldexp(v, e.unsqueeze(-1)).reshape(code.shape)


def _snap(x):
    """Rows rounded to MXFP4, as float64 (columns padded to a multiple of 32)."""
    return _value(*_codes(_pad(x.double())))


def _deq(wp, ws):
    code = torch.stack((wp & 15, wp >> 4), -1).reshape(*wp.shape[:-1], -1)
    return _value(code, ws.int() - 127)


def _moe64(x, ids, w, p, snap=True, half=False):
    """The routed experts of rows x (float64, K padded), weighted and summed."""
    out = torch.zeros((x.shape[0], p["down_wp"].shape[1]), dtype=torch.float64, device=DEV)
    for e in ids.unique().tolist():
        t, s = torch.where(ids == e)
        g, u = (x[t] @ _deq(p[nm + "_wp"][e], p[nm + "_ws"][e]).T for nm in ("gate", "up"))
        h = g / (1.0 + torch.exp(-g)) * u
        h = _snap(h.half() if half else h) if snap else _pad(h)
        out.index_add_(0, t, (h @ _deq(p["down_wp"][e], p["down_ws"][e]).T) * w[t, s].double().unsqueeze(1))
    return out


def _route64(logits, k):
    pr = torch.softmax(logits.double(), -1)
    v, i = torch.sort(pr, dim=-1, descending=True, stable=True)
    return i[:, :k], v[:, :k] / v[:, :k].sum(-1, keepdim=True)


def _cache_encode(v):
    """Rounding of the cache write: E4M3, mantissa half away from zero, 0x7F from 248 up, m * 2^-6 below 2^-6."""
    v = v.double()
    a = v.abs()
    m, q = torch.frexp(a)
    eb, mant = q.long() + 6, torch.floor((2.0 * m - 1.0) * 8.0 + 0.5).long()
    eb, mant = torch.where(mant == 8, eb + 1, eb), torch.where(mant == 8, torch.zeros_like(mant), mant)
    code = torch.where(eb >= 15, torch.full_like(eb, 0x7F), (eb << 3) | mant)
    code = torch.where(eb <= 0, torch.floor(a * 64.0 + 0.5).long().clamp(0, 7), code)
    code = torch.where(a == 0, torch.zeros_like(code), code)
    return (code + 128 * (v < 0)).to(torch.uint8)


def _cache_decode(b):
    b = b.long()
    e, m = (b >> 3) & 15, (b & 7).double()
    v = torch.where(e == 0, m * 2.0 ** -6, torch.ldexp(1.0 + m / 8.0, e - 7))
    v = torch.where(e == 15, 56.0 * (8.0 + m), v)
    return torch.where(b >= 128, -v, v)


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return None
    d, c = _inputs(case, seed)
    if kind == "linear":
        return [_snap(x) @ _deq(*w).T for x, w in zip(d["x"], d["w"])]
    if kind == "forward":
        return _snap(d["x"].half()) @ _deq(*d["w"]).T
    if kind == "dropin":
        return [_moe64(_snap(x), i, w, p) for x, i, w, p in zip(d["x"], d["ids"], d["w"], d["experts"])]
    if kind == "batch":
        return [_moe64(_snap(x), *_route64(lg, c["E"]), p) for x, lg, p in zip(d["x"], d["logits"], d["experts"])]
    if kind == "prefill":
        ids, w = _route64(d["logits"][0], c["E"])
        return _moe64(_snap(d["x"][0].half()), ids, w.bfloat16(), d["experts"][0], half=True)
    if kind == "stack":
        x, xs, ys = d["x"][0], [], []
        for l in range(c["layers"]):
            ys.append(_moe64(x.double(), d["ids"][l], d["w"][l], d["experts"][l], snap=False)[0])
            x = (x.double() + ys[-1].bfloat16().double()).bfloat16()
            xs.append(x[0].double())
        return [xs[-1], torch.stack(xs), torch.stack(ys)]
    scale = float(torch.tensor(1.0) / torch.tensor(128.0).sqrt())
    o, ks, vs = [], [], []
    for l in range(c["layers"]):
        kvk, kvv = d["kvk"][l], d["kvv"][l]
        rows = slice(c["ctx"], c["ctx"] + c["M"])
        kvk[rows], kvv[rows] = _cache_encode(d["k"][l]), _cache_encode(d["v"][l])
        n = c["ctx"] + c["M"]
        k64, v64 = _cache_decode(kvk[:n]).permute(1, 0, 2), _cache_decode(kvv[:n]).permute(1, 0, 2)
        q = d["q"][l].double().view(c["M"], c["Hkv"], c["G"], 128).permute(1, 2, 0, 3)
        s = torch.matmul(q.reshape(c["Hkv"], -1, 128), k64.transpose(1, 2).contiguous()) * scale
        s = s.view(c["Hkv"], c["G"], c["M"], n)
        seen = torch.arange(n, device=DEV) <= c["ctx"] + torch.arange(c["M"], device=DEV).unsqueeze(1)
        pr = torch.softmax(s.masked_fill(~seen, -math.inf), -1).view(c["Hkv"], -1, n)
        r = torch.matmul(pr, v64.contiguous()).view(c["Hkv"], c["G"], c["M"], 128)
        o.append(r.permute(2, 0, 1, 3).reshape(c["M"], -1, 128))
        ks.append(kvk)
        vs.append(kvv)
    return o + ks + vs
