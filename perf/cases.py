"""The work that a user of the quantized-weight path has it do, as cases that can be timed and checked.

listed() names the cases, draw() gives more of the same ranges, prepare() builds
what a program holds before a call (weights in device memory, activations, a
captured decode step), run() is one pass through the public entry points,
work() the bytes and operations no pass can do without, exact() the results in
64 bits by plain torch, tolerance() how far another correct implementation of
the same precision may be from them.

The models are the three of the benchmark's decode workloads.  Weights are block
data as quantizers write them (codes near a bell, block scales that vary by a
factor of two, minima that centre the block) with the variance of a trained
projection; activations are normal with a few channels eight times larger.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "edgexpu-llm_amd"))
import edgexpu_amd as E  # noqa: E402

DEV = "cuda"
EPS = 1e-5
TYPES = {"q8_0": E.Q8_0, "q4_k": E.Q4_K, "q6_k": E.Q6_K}

MODELS = {
    "smollm2-135m": dict(layers=30, hidden=576, qdim=576, kv=192, ffn=1536, vocab=49152,
                         wtype="q8_0", down="q8_0", logits="q8_0"),
    "hybrid-4b": dict(layers=36, hidden=2560, qdim=4096, kv=1024, ffn=9728, vocab=151936,
                      wtype="q4_k", down="q6_k", logits="q6_k"),
    "llama3-8b": dict(layers=32, hidden=4096, qdim=4096, kv=1024, ffn=14336, vocab=128256,
                      wtype="q4_k", down="q4_k", logits="q4_k"),
}


def _model(case):
    """The case's model, with a vocabulary of the case's own where it has one (fine-tuned models extend or cut it)."""
    c = MODELS[case["model"]]
    return dict(c, vocab=case["vocab"]) if "vocab" in case else c


def listed():
    return [
        # one token's q/k/v projections of the smallest model: the smallest call, where latency is all
        dict(name="qkv_smollm_m1", kind="linear", type="q8_0", n_in=576, n_outs="576,192,192", m=1, bias=False),
        # a whole decode step of the smallest model as a serving loop replays it: 123 dependent launches
        dict(name="step_smollm_m1", kind="step", model="smollm2-135m", layers=30),
        # one token through a layer of the largest model: single-user decoding
        dict(name="layer_8b_m1", kind="layer", model="llama3-8b", m=1),
        # four tokens through a layer of mixed formats: a few users, or a drafted continuation being verified
        dict(name="layer_hybrid_m4", kind="layer", model="hybrid-4b", m=4),
        # eight users decoding at once
        dict(name="layer_8b_m8", kind="layer", model="llama3-8b", m=8),
        # a short prompt of odd length
        dict(name="layer_hybrid_m45", kind="layer", model="hybrid-4b", m=45),
        # a full prefill chunk of the largest model
        dict(name="layer_8b_m512", kind="layer", model="llama3-8b", m=512),
        # a ragged prompt through the smallest model
        dict(name="layer_smollm_m131", kind="layer", model="smollm2-135m", m=131),
        # the end of a greedy decode step: scores of the whole vocabulary and the best token
        dict(name="logits_hybrid_m1", kind="logits", model="hybrid-4b", m=1),
        # the same for four sequences
        dict(name="logits_8b_m4", kind="logits", model="llama3-8b", m=4),
        # the end of a sampled decode step: temperature, softmax, top-p, one draw
        dict(name="sample_128k", kind="sample", n=128256, temperature=0.8, top_p=0.9),
        # one tensor expanded to f32 (a program that wants plain weights)
        dict(name="dequant_q6k_ffn", kind="dequant", type="q6_k", n=4096 * 14336),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "linear", "linear", "step", "logits", "sample", "dequant"])
    if kind == "layer":
        return dict(kind=kind, model=rng.choice(sorted(MODELS)), m=_log_int(rng, 1, 512))
    if kind == "linear":
        qt = rng.choice(sorted(TYPES))
        unit = E.BLOCK[TYPES[qt]][0]
        n_in = unit * max(1, round(_log_int(rng, 256, 14336) / unit))
        outs = [_log_int(rng, 32, 14336) for _ in range(rng.randint(1, 3))]
        # at most the operations of one [14336 x 4096] projection of a full prefill chunk
        m = min(_log_int(rng, 1, 512), max(1, 512 * 14336 * 4096 // (n_in * sum(outs))))
        return dict(kind=kind, type=qt, n_in=n_in, n_outs=",".join(map(str, outs)), m=m, bias=rng.random() < 0.3)
    if kind == "step":
        return dict(kind=kind, model="smollm2-135m", layers=rng.randint(4, 29), vocab=_log_int(rng, 8000, 49152))
    if kind == "logits":
        c = rng.choice(sorted(MODELS))
        return dict(kind=kind, model=c, m=rng.randint(1, 8), vocab=_log_int(rng, 8000, MODELS[c]["vocab"]))
    if kind == "sample":
        return dict(kind=kind, n=_log_int(rng, 32000, 262144), temperature=round(rng.uniform(0.5, 1.3), 3),
                    top_p=rng.choice([0.5, 0.8, 0.9, 0.95, 1.0]))
    qt = rng.choice(sorted(TYPES))
    return dict(kind=kind, type=qt, n=256 * _log_int(rng, 64, 4096 * 14336 // 256))


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _f16b(t):
    return t.to(torch.float16).view(torch.uint8)


def _normal(shape, g):
    return torch.randn(shape, generator=g, device=DEV)


def _weights_piece(qt, rows, n, std, g):
    if qt == "q8_0":
        nb = n // 32
        q = (_normal((rows, nb, 32), g) * 42).round_().clamp_(-127, 127).to(torch.int8)
        d = std / 42 * (0.7 + 0.7 * torch.rand((rows, nb, 1), generator=g, device=DEV))
        return torch.cat([_f16b(d), q.view(torch.uint8)], 2).view(rows, -1)
    nb = n // 256
    if qt == "q4_k":
        sc = torch.randint(24, 64, (rows, nb, 8), generator=g, device=DEV)
        mn = (sc + torch.randint(-4, 5, (rows, nb, 8), generator=g, device=DEV)).clamp_(0, 63)
        q = (_normal((rows, nb, 4, 2, 32), g) * 2.9 + 7.5).round_().clamp_(0, 15).to(torch.uint8)
        d = std / (2.9 * 43) * (0.7 + 0.7 * torch.rand((rows, nb, 1), generator=g, device=DEV))
        lo = sc[..., :4] | (sc[..., 4:] >> 4 << 6)
        mid = mn[..., :4] | (mn[..., 4:] >> 4 << 6)
        hi = (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)
        return torch.cat([_f16b(d), _f16b(7.5 * d), torch.cat([lo, mid, hi], 2).to(torch.uint8),
                          (q[:, :, :, 0] | (q[:, :, :, 1] << 4)).view(rows, nb, 128)], 2).view(rows, -1)
    sc = torch.randint(40, 128, (rows, nb, 16), generator=g, device=DEV)
    sc = sc * (1 - 2 * torch.randint(0, 2, (rows, nb, 16), generator=g, device=DEV))
    q = ((_normal((rows, nb, 2, 4, 32), g) * 10).round_().clamp_(-32, 31) + 32).to(torch.uint8)
    d = std / (10 * 87) * (0.7 + 0.7 * torch.rand((rows, nb, 1), generator=g, device=DEV))
    ql = torch.cat([(q[:, :, :, 0] & 15) | (q[:, :, :, 2] << 4), (q[:, :, :, 1] & 15) | (q[:, :, :, 3] << 4)], 3)
    qh = (q[:, :, :, 0] >> 4) | (q[:, :, :, 1] >> 4 << 2) | (q[:, :, :, 2] >> 4 << 4) | (q[:, :, :, 3] >> 4 << 6)
    return torch.cat([ql.reshape(rows, nb, 128), qh.reshape(rows, nb, 64), sc.to(torch.int8).view(torch.uint8),
                      _f16b(d)], 2).view(rows, -1)


def _weights(qt, rows, n, g):
    out = torch.empty((rows, E.row_bytes(TYPES[qt], n)), dtype=torch.uint8, device=DEV)
    step = max(1, (1 << 26) // n)
    for r in range(0, rows, step):
        k = min(step, rows - r)
        out[r:r + k] = _weights_piece(qt, k, n, 1 / math.sqrt(n), g)
    return out


def _activations(m, n, g):
    big = (torch.rand((1, n), generator=g, device=DEV) < 0.01).float() * 7 + 1
    return _normal((m, n), g) * big


def _layer_shapes(c):
    h, q, kv, f, t = c["hidden"], c["qdim"], c["kv"], c["ffn"], c["wtype"]
    return dict(q=(t, q, h), k=(t, kv, h), v=(t, kv, h), o=(t, h, q), gate=(t, f, h), up=(t, f, h),
                down=(c["down"], h, f))


def _layer_weights(c, g):
    w = {name: _weights(t, rows, n, g) for name, (t, rows, n) in _layer_shapes(c).items()}
    w["attn_norm"] = 1 + 0.1 * _normal((c["hidden"],), g)
    w["ffn_norm"] = 1 + 0.1 * _normal((c["hidden"],), g)
    return w


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        outs = [int(v) for v in case["n_outs"].split(",")]
        return dict(case=case, outs=outs, w=[_weights(case["type"], r, case["n_in"], g) for r in outs],
                    bias=[0.1 * _normal((r,), g) for r in outs] if case["bias"] else None,
                    x=_activations(case["m"], case["n_in"], g))
    if kind == "layer":
        c, m = _model(case), case["m"]
        gate = _normal((m, c["ffn"]), g)
        return dict(case=case, c=c, w=_layer_weights(c, g), x=_activations(m, c["hidden"], g),
                    attn=0.3 * _normal((m, c["qdim"]), g), mid=_activations(m, c["hidden"], g),
                    act=torch.nn.functional.silu(gate) * _normal((m, c["ffn"]), g))
    if kind == "step":
        return _prepare_step(case, g)
    if kind == "logits":
        c = _model(case)
        return dict(case=case, c=c, w=_weights(c["logits"], c["vocab"], c["hidden"], g),
                    hidden=_normal((case["m"], c["hidden"]), g))
    if kind == "sample":
        # a language model's scores: a broad body and a few dozen candidates above it
        s = 2.5 * _normal((case["n"],), g)
        top = torch.randint(0, case["n"], (40,), generator=g, device=DEV)
        s[top] += 6 + 8 * torch.rand((40,), generator=g, device=DEV)
        return dict(case=case, scores=s, work=torch.empty_like(s), rng=(seed * 2654435761 + 12345) & (2 ** 63 - 1))
    n = case["n"]
    return dict(case=case, src=_weights(case["type"], n // 256, 256, g).view(-1))


def _prepare_step(case, g):
    """The decode step captured once in a HIP graph, as a serving loop keeps it."""
    c = _model(case)
    s = dict(case=case, c=c, layers=[_layer_weights(c, g) for _ in range(case["layers"])],
             embd=_weights(c["logits"], c["vocab"], c["hidden"], g),  # tied: also the output matrix
             norm=1 + 0.1 * _normal((c["hidden"],), g),
             ids=torch.randint(0, c["vocab"], (1,), generator=g, device=DEV, dtype=torch.int32),
             scores=torch.empty((1, c["vocab"]), device=DEV), best=torch.empty(1, dtype=torch.int32, device=DEV))
    E.hip().check(E.hip().init(torch.cuda.current_device()), "init")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(s)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        _step(s)
    return s


def _step(s):
    """Embedding, layers, final norm, logits.  Attention is not on this path: o reads q, which keeps the order of
    the launches."""
    c, t = s["c"], TYPES[s["c"]["wtype"]]
    h = E.embed_rows(s["embd"], TYPES[c["logits"]], c["vocab"], c["hidden"], s["ids"])
    for w in s["layers"]:
        q, _, _ = E.layer_linear([w["q"], w["k"], w["v"]], t, h, [c["qdim"], c["kv"], c["kv"]], c["hidden"],
                                 norm_weight=w["attn_norm"], eps=EPS)
        E.layer_linear([w["o"]], t, q, [c["hidden"]], c["qdim"], residuals=[h], outs=[h])
        act = E.gate_up_silu(w["gate"], w["up"], t, h, c["ffn"], c["hidden"], norm_weight=w["ffn_norm"], eps=EPS)
        E.layer_linear([w["down"]], TYPES[c["down"]], act, [c["hidden"]], c["ffn"], residuals=[h], outs=[h])
    hn = E.rmsnorm(h, s["norm"], EPS)
    L = E.hip()
    L.check(L.logits_noalloc_dev(s["scores"].data_ptr(), s["best"].data_ptr(), hn.data_ptr(), s["embd"].data_ptr(),
                                 TYPES[c["logits"]], None, 1, c["vocab"], c["hidden"], 0,
                                 torch.cuda.current_stream().cuda_stream), "logits_noalloc")


# ------------------------------------------------------------------ a pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        return E.linear_quant_group(s["w"], TYPES[case["type"]], s["x"], s["outs"], case["n_in"], biases=s["bias"])
    if kind == "layer":
        # the four calls of a layer, each on what its place in the layer reads (so that every result has an exact value)
        c, w, t = s["c"], s["w"], TYPES[s["c"]["wtype"]]
        q, k, v = E.layer_linear([w["q"], w["k"], w["v"]], t, s["x"], [c["qdim"], c["kv"], c["kv"]], c["hidden"],
                                 norm_weight=w["attn_norm"], eps=EPS)
        o, = E.layer_linear([w["o"]], t, s["attn"], [c["hidden"]], c["qdim"], residuals=[s["x"]])
        act = E.gate_up_silu(w["gate"], w["up"], t, s["mid"], c["ffn"], c["hidden"], norm_weight=w["ffn_norm"], eps=EPS)
        h, = E.layer_linear([w["down"]], TYPES[c["down"]], s["act"], [c["hidden"]], c["ffn"], residuals=[s["mid"]])
        return dict(q=q, k=k, v=v, o=o, act=act, h=h)
    if kind == "step":
        s["graph"].replay()
        return dict(scores=s["scores"])  # of which the token is the largest
    if kind == "logits":
        c = s["c"]
        scores, best = E.logits(s["w"], TYPES[c["logits"]], s["hidden"], c["vocab"], c["hidden"])
        return dict(scores=scores, best=best)
    if kind == "sample":
        p = s["work"].copy_(s["scores"])  # the entry points work in place; a step's scores are new each time
        E.div_scalar(p, case["temperature"])
        token, _ = E.sample_softmax(p, case["top_p"], s["rng"])
        return dict(p=p, token=token)
    return E.dequantize(s["src"], TYPES[case["type"]], case["n"])


# ------------------------------------------------------------------ what a pass cannot do without


def _linear_work(t, rows, n, m):
    return rows * E.row_bytes(TYPES[t], n) + 4 * m * rows, 2 * m * rows * n


def work(case):
    kind = case["kind"]
    if kind == "linear":
        parts = [_linear_work(case["type"], int(r), case["n_in"], case["m"]) for r in case["n_outs"].split(",")]
        return {"bytes": sum(p[0] for p in parts) + 4 * case["m"] * case["n_in"], "flops": sum(p[1] for p in parts)}
    if kind in ("layer", "step"):
        c, m = _model(case), case.get("m", 1)
        parts = {k: _linear_work(*v, m) for k, v in _layer_shapes(c).items()}
        # gate and up leave as their product
        b = sum(p[0] for p in parts.values()) - 4 * m * c["ffn"] + 8 * c["hidden"]
        f = sum(p[1] for p in parts.values())
        if kind == "layer":
            return {"bytes": b + 4 * m * (2 * c["hidden"] + c["qdim"] + c["ffn"]), "flops": f}
        lb, lf = _linear_work(c["logits"], c["vocab"], c["hidden"], 1)
        return {"bytes": case["layers"] * b + lb, "flops": case["layers"] * f + lf}
    if kind == "logits":
        c, m = _model(case), case["m"]
        b, f = _linear_work(c["logits"], c["vocab"], c["hidden"], m)
        return {"bytes": b + 4 * m * c["hidden"], "flops": f}
    if kind == "sample":
        return {"bytes": 8 * case["n"], "flops": 6 * case["n"]}
    return {"bytes": E.row_bytes(TYPES[case["type"]], case["n"]) + 4 * case["n"], "flops": 2 * case["n"]}


# ------------------------------------------------------------------ the results in 64 bits


def _unpack(qt, w, n):
    """[rows, n] float64 weights of uint8 rows."""
    rows = w.shape[0]

    def f16(b):
        return b.contiguous().view(torch.float16).to(torch.float64)

    if qt == "q8_0":
        b = w.view(rows, n // 32, 34)
        return (f16(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).to(torch.float64)).view(rows, n)
    nb = n // 256
    if qt == "q4_k":
        b = w.view(rows, nb, 144)
        s = b[..., 4:16]
        lo, mid, hi = s[..., :4], s[..., 4:8], s[..., 8:]
        sc = torch.cat([lo & 63, (hi & 15) | (lo >> 6 << 4)], 2).to(torch.float64)
        mn = torch.cat([mid & 63, (hi >> 4) | (mid >> 6 << 4)], 2).to(torch.float64)
        qs = b[..., 16:].view(rows, nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).view(rows, nb, 8, 32).to(torch.float64)
        d, dm = f16(b[..., :2]), f16(b[..., 2:4])
        return ((d * sc).unsqueeze(3) * q - (dm * mn).unsqueeze(3)).view(rows, n)
    b = w.view(rows, nb, 210)
    ql, qh = b[..., :128].view(rows, nb, 2, 2, 32), b[..., 128:192].view(rows, nb, 2, 32)
    q = torch.stack([(ql[:, :, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, :, 1] & 15) | ((qh >> 2 & 3) << 4),
                     (ql[:, :, :, 0] >> 4) | ((qh >> 4 & 3) << 4), (ql[:, :, :, 1] >> 4) | (qh >> 6 << 4)], 3)
    q = q.reshape(rows, nb, 16, 16).to(torch.float64) - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).to(torch.float64)
    return ((f16(b[..., 208:]) * sc).unsqueeze(3) * q).view(rows, n)


def _codes(qt, x):
    """The activation as the product sees it, in float64: 8-bit codes times the block's scale.  The codes are decided
    in 32 bits by the format's definition."""
    m, n = x.shape
    x = x.to(torch.float32).cpu()
    if qt == "q8_0":
        b = x.view(m, n // 32, 32)
        top = b.abs().amax(2, keepdim=True)
        q = torch.where(top > 0, (b * (127.0 / top)).round(), torch.zeros_like(b)).clamp(-127, 127)
        return (q.to(torch.float64) * (top / 127.0).to(torch.float16).to(torch.float64)).view(m, n).to(DEV)
    b = x.view(m, n // 256, 256)
    top = b.abs().amax(2, keepdim=True)
    inv = 127.0 / top
    q = torch.where(top > 0, (b * inv).round(), torch.zeros_like(b)).clamp(-127, 127)
    d = torch.where(top > 0, 1.0 / inv, torch.zeros_like(inv))
    return (q.to(torch.float64) * d.to(torch.float64)).view(m, n).to(DEV)


def _product(qt, w, n, a):
    step = max(1, (1 << 26) // n)
    return torch.cat([a @ _unpack(qt, w[r:r + step], n).t() for r in range(0, w.shape[0], step)], 1)


def _rmsnorm(x, weight):
    """In the 32-bit steps whose rounding decides the codes: the mean of squares in 64 bits, then the scale, x times
    it, times the weight, each rounded."""
    x, weight = x.to(torch.float32).cpu(), weight.cpu()
    mean = x.to(torch.float64).square().mean(1, keepdim=True).to(torch.float32)
    return x * (1.0 / torch.sqrt(mean + EPS)) * weight


def _silu(x):
    return x / (1 + torch.exp(-x))


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    s = prepare(case, seed)
    if kind == "linear":
        a = _codes(case["type"], s["x"])
        outs = [_product(case["type"], w, case["n_in"], a) for w in s["w"]]
        return outs if s["bias"] is None else [o + b.to(torch.float64) for o, b in zip(outs, s["bias"])]
    if kind == "layer":
        c, w = s["c"], s["w"]
        t, h = c["wtype"], c["hidden"]
        a = _codes(t, _rmsnorm(s["x"], w["attn_norm"]))
        r = {k: _product(t, w[k], h, a) for k in ("q", "k", "v")}
        r["o"] = s["x"].to(torch.float64) + _product(t, w["o"], c["qdim"], _codes(t, s["attn"]))
        a = _codes(t, _rmsnorm(s["mid"], w["ffn_norm"]))
        r["act"] = _silu(_product(t, w["gate"], h, a)) * _product(t, w["up"], h, a)
        r["h"] = s["mid"].to(torch.float64) + _product(c["down"], w["down"], c["ffn"], _codes(c["down"], s["act"]))
        return r
    if kind == "logits":
        t, n = s["c"]["logits"], s["c"]["hidden"]
        scores = _product(t, s["w"], n, _codes(t, s["hidden"]) if t == "q8_0" else s["hidden"].to(torch.float64))
        return dict(scores=scores, best=scores.argmax(1).to(torch.int32))
    if kind == "sample":
        # the token is a place in a sum and has no value of its own in 64 bits
        return dict(p=torch.softmax(s["scores"].to(torch.float64) / case["temperature"], 0), token=None)
    return _unpack(case["type"], s["src"].view(-1, E.row_bytes(TYPES[case["type"]], 256)), 256).view(-1)


def _exact_step(case, seed):
    s = prepare(case, seed)
    c = s["c"]
    t, n = c["wtype"], c["hidden"]
    h = _unpack(c["logits"], s["embd"][s["ids"].long()], n)
    for w in s["layers"]:
        q = _product(t, w["q"], n, _codes(t, _rmsnorm(h, w["attn_norm"])))
        h = h + _product(t, w["o"], c["qdim"], _codes(t, q))
        a = _codes(t, _rmsnorm(h, w["ffn_norm"]))
        h = h + _product(c["down"], w["down"], c["ffn"],
                         _codes(c["down"], _silu(_product(t, w["gate"], n, a)) * _product(t, w["up"], n, a)))
    scores = _product(c["logits"], s["embd"], n, _codes(c["logits"], _rmsnorm(h, s["norm"])))
    return dict(scores=scores)


# Each about four times what the path shows against exact(), which another order of its 32-bit sums shows too.
TOLERANCE = {
    "linear": {"rel": 1e-6},   # 1e-7 to 2e-7
    "layer": {"rel": 1e-4},    # 2e-7, but 3e-5 where a last bit of the norm's scale moves codes of the activation
    "step": {"rel": 3e-2},     # 1.6e-2: thirty layers carry every moved code on
    "logits": {"rel": 2e-6},   # 4e-7
    "sample": {"rel": 3e-6},   # 6e-7
    "dequant": "exact",
}


def tolerance(case):
    return TOLERANCE[case["kind"]]
