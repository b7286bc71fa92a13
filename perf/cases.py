"""The work this library is measured on: MoE layers, stacks of them and the expert products alone,
called through flashrt_amd as an engine calls them, on seeded inputs made on the GPU.

listed() names the cases, draw() gives more of the same ranges. A case is one call: `tokens` rows
through one layer ("layer"), one token through a stack ("stack"), the expert GEMVs of a decode window
("hits") or the grouped expert products of a prefill chunk ("q2"). Two layer shapes run through all of
them: hidden 2048 with 512-wide experts (the benchmark's) and hidden 2560 with 640-wide ones (the
model's, whose shared expert comes in its GGUF type).

exact() restates the call in float64 with plain torch: Q2_0 weights dequantized, activations and the
experts' hidden values rounded to Q8_0 codes, every sum in float64. The input's codes are whole numbers
that the call defines in float32 operations, and bf16 inputs often lie on a tie (half of a block's
largest value), so they are formed in float32 here too; the hidden values' codes come from float64.
"""
import math

import torch

import flashrt_amd as F

GGML = {"f32": 0, "f16": 1, "q8_0": 8, "bf16": 30}
BENCH = dict(n=2048, ff=512, E=512, K=10)
MODEL = dict(n=2560, ff=640, E=512, K=10)


def listed():
    return [
        # one decoded token through one layer, the smallest call: launches and latency
        dict(name="decode1", kind="layer", tokens=1, shared="q2_0", norm=False, resid=False, skew="flat", corr=0.0, **BENCH),
        # the same on the model's own layer: RMS norm, residual and a Q8_0 shared expert
        dict(name="decode1_model", kind="layer", tokens=1, shared="q8_0", norm=True, resid=True, skew="zipf", corr=0.0, **MODEL),
        # a speculative-verify window: one token and two drafts, partly the same experts
        dict(name="verify3", kind="layer", tokens=3, shared="q2_0", norm=False, resid=False, skew="flat", corr=0.8, **BENCH),
        # the widest verify window
        dict(name="verify8", kind="layer", tokens=8, shared="q2_0", norm=True, resid=True, skew="flat", corr=0.8, **BENCH),
        # a whole decode step: one token through the 48 layers in one call
        dict(name="stack48", kind="stack", tokens=1, layers=48, shared="q2_0", norm=True, skew="zipf", **BENCH),
        # the expert GEMVs alone, as an engine with its own router calls them in a window
        dict(name="hits4", kind="hits", tokens=4, corr=0.8, **MODEL),
        # decode of 37 sequences at once
        dict(name="batch37", kind="layer", tokens=37, shared="q2_0", norm=True, resid=True, skew="zipf", corr=0.0, **BENCH),
        # a short prompt on the model's layer, shared expert in BF16
        dict(name="prompt200_model", kind="layer", tokens=200, shared="bf16", norm=True, resid=True, skew="zipf", corr=0.3, **MODEL),
        # a prefill chunk on the model's layer, shared expert in Q8_0
        dict(name="chunk1024_model", kind="layer", tokens=1024, shared="q8_0", norm=True, resid=True, skew="zipf", corr=0.3, **MODEL),
        # the grouped expert products alone, 64-wide activation blocks and bf16 results, a ragged count
        dict(name="q2_777", kind="q2", tokens=777, block64=True, yd="bf16", **MODEL),
        # the benchmark's prefill chunk: 2048 tokens under skewed expert popularity
        dict(name="prefill2048", kind="layer", tokens=2048, shared="q2_0", norm=False, resid=False, skew="zipf", corr=0.0, **BENCH),
        # the largest call: an 8192-token chunk with 16 decoding sequences, 16 experts far ahead of the rest
        dict(name="mixed8208", kind="layer", tokens=8208, shared="q2_0", norm=False, resid=False, skew="hot", corr=0.0, **BENCH),
    ]


def draw(rng):
    def tokens(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))
    shape = dict(rng.choice([BENCH, BENCH, MODEL, MODEL, dict(n=1024, ff=1024, E=128, K=8)]))
    if rng.random() < 0.25:
        shape["K"] = rng.randint(4, 12)
    kind = rng.choice(["layer"] * 6 + ["stack", "hits", "q2"])
    if kind == "stack":
        return dict(kind="stack", tokens=1, layers=rng.randint(2, 48), shared="q2_0", norm=True,
                    skew=rng.choice(["flat", "zipf"]), **dict(BENCH, K=shape["K"]))
    if kind == "hits":
        return dict(kind="hits", tokens=rng.randint(1, 8), corr=rng.choice([0.0, 0.8]), **shape)
    if kind == "q2":
        return dict(kind="q2", tokens=tokens(9, 2048), block64=rng.random() < 0.5, yd=rng.choice(["f32", "bf16"]), **shape)
    size = rng.choice(["window", "batch", "prefill", "prefill"])
    n_tok = rng.randint(1, 8) if size == "window" else tokens(9, 128) if size == "batch" else tokens(129, 4096)
    return dict(kind="layer", tokens=n_tok, shared=rng.choice(["q2_0", "q2_0", "q2_0", "q8_0", "q8_0", "bf16", "f16", "f32"]),
                norm=rng.random() < 0.5, resid=rng.random() < 0.5, skew=rng.choice(["flat", "zipf", "hot"]),
                corr=rng.choice([0.0, 0.3, 0.8]), **shape)


# ---------------------------------------------------------------- inputs, from the seed alone

def _expert_bytes(n, ff):
    return 3 * n * (ff // 64) * 18


def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + what) & 0x7FFFFFFF)
    return g


def _normal(shape, g, sd=1.0):
    return torch.randn(shape, generator=g, device="cuda") * sd


def _blobs(count, stride, n, ff, g):
    """`count` expert blobs (gate | up | down, planar Q2_0): uniform codes, scales |N(0, 1)| * 0.02 in fp16."""
    out = torch.randint(-2**31, 2**31, (count * stride // 4,), generator=g, device="cuda", dtype=torch.int32)
    out = out.view(torch.uint8).view(count, stride)
    mat = n * (ff // 64) * 18
    for m in range(3):
        lo, size = m * mat + n * ff // 4, n * ff // 64
        out[:, lo:lo + 2 * size].view(torch.float16).copy_(_normal((count, size), g, 0.02).abs_())
    return out


def _stride(case):
    return (_expert_bytes(case["n"], case["ff"]) + 4095) // 4096 * 4096


def _dense(kind, rows, cols, g):
    """A [rows][cols] weight matrix N(0, 0.02) in ggml's layout of the type, as raw bytes."""
    w = _normal((rows, cols), g, 0.02)
    if kind == "q8_0":
        blk = w.view(-1, 32)
        d = (blk.abs().amax(1, keepdim=True) / 127).half()
        q = torch.round(blk / d.float()).clamp_(-127, 127).to(torch.int8)
        return torch.cat([d.view(torch.uint8).view(-1, 2), q.view(torch.uint8)], 1).reshape(-1).contiguous()
    return w.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]).view(torch.uint8).reshape(-1)


def _bias(case, g):
    """The router's prior: none, a Zipf popularity over a random order, or 16 experts far ahead."""
    E = case["E"]
    order = torch.randperm(E, generator=g, device="cuda")
    bias = torch.zeros(E, device="cuda")
    if case["skew"] == "zipf":
        strength = 1.1 if case["tokens"] <= 64 else 0.5   # (a lone token's prior; a chunk's, softened)
        bias[order] = -strength * torch.log(torch.arange(1, E + 1, device="cuda").float())
    elif case["skew"] == "hot":
        bias[order[:16]] = 2.8
    return bias


def _tokens(case, g):
    """[tokens][n] N(0, 1) rows with pairwise cosine `corr`; a prefill chunk's arrive rounded to bf16."""
    T, n, c = case["tokens"], case["n"], case.get("corr", 0.0)
    x = math.sqrt(1 - c) * _normal((T, n), g) + math.sqrt(c) * _normal((1, n), g)
    return x.bfloat16().float() if T > 64 else x


def _layer_weights(case, seed, layer):
    n, ff, E = case["n"], case["ff"], case["E"]
    g = _gen(seed, 10 + layer)
    w = dict(router=_normal((E, n), g, 0.02), gate=_normal((n,), g, 0.02), bias=_bias(case, g))
    if case["shared"] == "q2_0":
        w["shared"] = _blobs(1, _stride(case), n, ff, g)
    else:
        w["shared"] = [_dense(case["shared"], r, c, g) for r, c in ((ff, n), (ff, n), (n, ff))]
    return w


def _ids(case, g):
    """[tokens][K] distinct experts of each token, as a router with the case's overlap picks them."""
    T, E, c = case["tokens"], case["E"], case.get("corr", 0.0)
    lg = math.sqrt(1 - c) * _normal((T, E), g) + math.sqrt(c) * _normal((1, E), g)
    if case["kind"] == "q2":
        order = torch.randperm(E, generator=g, device="cuda")
        lg[:, order] -= 0.5 * torch.log(torch.arange(1, E + 1, device="cuda").float())
    return torch.topk(lg, case["K"], dim=1).indices.to(torch.int32).contiguous()


def _inputs(case, seed):
    """(experts [layers * E][stride] bytes, per-layer weights, x, extra) of the case."""
    layers = case.get("layers", 1)
    g = _gen(seed, 1)
    experts = torch.empty((layers * case["E"], _stride(case)), dtype=torch.uint8, device="cuda")
    for l in range(layers):
        experts[l * case["E"]:(l + 1) * case["E"]] = _blobs(case["E"], _stride(case), case["n"], case["ff"], g)
    g = _gen(seed, 2)
    x = _tokens(case, g)
    if case["kind"] in ("layer", "stack"):
        weights = [_layer_weights(case, seed, l) for l in range(layers)]
        resid = _normal(x.shape, g) if case.get("resid") else None
        return experts, weights, x, resid
    return experts, None, x, _ids(case, g)


# ---------------------------------------------------------------- the call

def prepare(case, seed):
    kind, T, n, ff, E, K = (case[k] for k in ("kind", "tokens", "n", "ff", "E", "K"))
    experts, weights, x, extra = _inputs(case, seed)
    stride = _stride(case)
    s = dict(case=dict(case), x=x, keep=(experts, weights, extra))
    if kind in ("layer", "stack"):
        layers = []
        for l, w in enumerate(weights):
            q2 = case["shared"] == "q2_0"
            ml = F.MoeLayer(experts[l * E].data_ptr(), stride, E, w["shared"].data_ptr() if q2 else 0, w["router"], w["gate"],
                            n, ff, K, router_bias=w["bias"], norm_input=case["norm"])
            if not q2:
                ml.set_shared_dense(GGML[case["shared"]], *w["shared"], ff)
            layers.append(ml)
        s["ids"] = torch.empty((len(layers) * T, K), dtype=torch.int32, device="cuda")
        s["wts"] = torch.empty((len(layers) * T, K), dtype=torch.float32, device="cuda")
        s["out"] = torch.empty((T, n), dtype=torch.float32, device="cuda")
        if kind == "stack":
            for l, ml in enumerate(layers):
                ml.set_next_router(weights[(l + 1) % len(layers)]["router"])
            s["call"] = F.MoeStack(layers)
            s["ws"] = s["call"].workspace()
        else:
            s["call"] = layers[0]
            s["ws"] = layers[0].workspace(T)
            s["resid"] = extra
    elif kind == "hits":
        s["hit_ptr"] = (experts.data_ptr() + extra.to(torch.int64) * stride).contiguous()
        s["hit_n"] = torch.full((T,), K, dtype=torch.int32, device="cuda")
        s["ws"] = torch.empty(F.moe_hits_scratch_bytes(K, ff, T), dtype=torch.uint8, device="cuda")
        s["out"] = torch.empty((T, K, n), dtype=torch.float32, device="cuda")
    else:
        s["ids"] = extra
        s["experts"], s["stride"] = experts.data_ptr(), stride
        s["ws_bytes"] = F.moe_q2.workspace_bytes(T, K, n, ff, E)
        s["ws"] = torch.empty(s["ws_bytes"], dtype=torch.uint8, device="cuda")
        s["out"] = torch.empty((T * K, n), dtype=torch.bfloat16 if case["yd"] == "bf16" else torch.float32, device="cuda")
    return s


def run(s):
    case, out = s["case"], s["out"]
    kind, T, n, ff, E, K = (case[k] for k in ("kind", "tokens", "n", "ff", "E", "K"))
    if kind == "layer":
        s["call"].forward(s["x"], out, T=T, resid=s["resid"], ids=s["ids"], wts=s["wts"], ws=s["ws"])
    elif kind == "stack":
        s["call"].forward(s["x"], out, ids=s["ids"], wts=s["wts"], ws=s["ws"])
    elif kind == "hits":
        F.moe_hits(s["hit_ptr"], s["hit_n"], K, s["x"], n, ff, s["ws"], out, T=T)
        return {"out": out}
    else:
        F.moe_q2.run(s["experts"], s["stride"], E, n, ff, s["x"], s["ids"], T, K, out, s["ws"], s["ws_bytes"],
                     block64=case["block64"], yd_bf16=case["yd"] == "bf16")
        return {"out": out}
    return {"out": out, "ids": s["ids"], "wts": s["wts"]}


# ---------------------------------------------------------------- what a pass cannot do without

def _distinct(case):
    """The number of experts that a call of the case's tokens is expected to read."""
    E, slots = case["E"], case["tokens"] * case["K"]
    skew = case.get("skew", "zipf" if case["kind"] == "q2" else "flat")
    if skew == "zipf":
        a = 1.1 if case["tokens"] <= 64 else 0.5
        p = [r ** -a for r in range(1, E + 1)]
    elif skew == "hot":
        p = [9.0 / 16] * 16 + [1.0 / (E - 16)] * (E - 16)
    else:
        p = [1.0] * E
    if case.get("corr"):   # the tokens' common part counts as fewer tokens
        slots = case["K"] * (1 + (case["tokens"] - 1) * (1 - case["corr"]))
    tot = sum(p)
    return max(case["K"], min(slots, sum(1 - (1 - q / tot) ** slots for q in p)))


def work(case):
    T, n, ff, E, K = (case[k] for k in ("tokens", "n", "ff", "E", "K"))
    eb = _expert_bytes(n, ff)
    b, f = _distinct(case) * eb, 2.0 * T * K * 3 * n * ff
    if case["kind"] in ("layer", "stack"):
        per = {"q2_0": 18 / 64, "q8_0": 34 / 32, "f16": 2, "bf16": 2, "f32": 4}[case["shared"]]
        b += 3 * n * ff * per + 4 * (E + 1) * n
        f += 2.0 * T * 3 * n * ff + 2.0 * T * (E + 1) * n
        b, f = b * case.get("layers", 1), f * case.get("layers", 1)
        b += T * n * 4 * (3 if case.get("resid") else 2)
    else:
        b += T * n * 4 + T * K * n * (2 if case.get("yd") == "bf16" else 4)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Relative 2-norm errors, about four times what the calls show against exact(). A sum in another
    order moves some Q8_0 codes of the experts' hidden values by one step (3e-4 for a lone token); in a
    stack the moved values reach the routers of the layers above. Prefill also holds the hidden values
    and a layer's per-expert outputs in fp16 (5e-4 measured), or gives them out in bf16 (1.8e-3)."""
    if case["kind"] == "stack":
        return {"rel": 5e-3, "differ": 0.01}
    if case.get("yd") == "bf16":
        return {"rel": 7e-3}
    return {"rel": 1e-3 if case["tokens"] <= 8 else 2e-3, "differ": 0.002}


# ---------------------------------------------------------------- the same in float64, plain torch

def _mat(b, rows, cols):
    """[rows][cols] float64 values of a planar Q2_0 matrix: element j of a 64-block in byte j % 16, bits 2 (j / 16)."""
    nb = cols // 64
    codes = b[:rows * nb * 16].view(rows, nb, 1, 16)
    shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device).view(1, 1, 4, 1)
    q = ((codes >> shift) & 3).double() - 1
    d = b[rows * nb * 16:rows * nb * 18].view(torch.float16).view(rows, nb, 1, 1).double()
    return (q * d).view(rows, cols)


def _q8(v, block):
    """v rounded to Q8_0, in its own precision: codes round(v * (1 / d)), half away from zero, with
    d = amax / 127; the value is the code times d held in fp16, as float64."""
    r = v.reshape(-1, block)
    d = r.abs().amax(1, keepdim=True) / 127
    code = r * torch.where(d == 0, torch.zeros_like(d), 1 / d)
    code = torch.sign(code) * torch.floor(code.abs().double() + 0.5)
    return (code.double() * d.half().double()).view(v.shape)


def _ffn(g, u, d, x, block):
    h = x @ g.T
    h = h / (1 + torch.exp(-h)) * (x @ u.T)
    return (_q8(h, block) if block else h) @ d.T


def _blob_ffn(blob, n, ff, x, block):
    m = n * (ff // 64) * 18
    return _ffn(_mat(blob[:m], ff, n), _mat(blob[m:2 * m], ff, n), _mat(blob[2 * m:3 * m], n, ff), x, block)


def _routed(case, experts, x, ids, block):
    """[tokens][K][n] per-slot expert outputs."""
    y = torch.empty((*ids.shape, case["n"]), dtype=torch.float64, device="cuda")
    xq = _q8(x.float(), block)
    for e in torch.unique(ids).tolist():
        t, k = torch.nonzero(ids == e, as_tuple=True)
        y[t, k] = _blob_ffn(experts[e], case["n"], case["ff"], xq[t], block)
    return y


def _dense_values(kind, raw, rows, cols):
    if kind == "q8_0":
        blk = raw.view(-1, 34)
        d = blk[:, :2].contiguous().view(torch.float16).double()
        return (blk[:, 2:].contiguous().view(torch.int8).double() * d).view(rows, cols)
    return raw.view({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]).double().view(rows, cols)


def _moe(case, experts, w, x):
    """(the layer's output without the residual, ids, weights)."""
    n, ff, K = case["n"], case["ff"], case["K"]
    if case["norm"]:   # (the input proper, in float32: its codes and the router's operand)
        x = (x.float() * (1 / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6)).float()).double()
    top = torch.sort(x @ w["router"].double().T + w["bias"].double(), dim=1, descending=True, stable=True)
    ids = top.indices[:, :K].to(torch.int32)
    p = torch.softmax(top.values, 1)[:, :K]
    wts = p / p.sum(1, keepdim=True).clamp_min(2.0 ** -14)
    y = (_routed(case, experts, x, ids, 32) * wts[:, :, None]).sum(1)
    if case["shared"] == "q2_0":
        sh = _blob_ffn(w["shared"][0], n, ff, _q8(x.float(), 32), 32)
    else:
        q8 = case["shared"] == "q8_0"
        g, u, d = (_dense_values(case["shared"], r, *s) for r, s in zip(w["shared"], ((ff, n), (ff, n), (n, ff))))
        sh = _ffn(g, u, d, _q8(x.float(), 32) if q8 else x, 32 if q8 else 0)
    return y + sh * torch.sigmoid(x @ w["gate"].double())[:, None], ids, wts


def exact(case, seed):
    experts, weights, x, extra = _inputs(case, seed)
    x = x.double()
    E = case["E"]
    if case["kind"] == "layer":
        y, ids, wts = _moe(case, experts, weights[0], x)
        return {"out": y if extra is None else y + extra.double(), "ids": ids, "wts": wts}
    if case["kind"] == "stack":
        ids, wts = [], []
        for l, w in enumerate(weights):
            y, i, p = _moe(case, experts[l * E:(l + 1) * E], w, x)
            x = x + y
            ids.append(i)
            wts.append(p)
        return {"out": x, "ids": torch.cat(ids), "wts": torch.cat(wts)}
    y = _routed(case, experts, x, extra, 64 if case.get("block64") else 32)
    return {"out": y if case["kind"] == "hits" else y.view(-1, case["n"])}
