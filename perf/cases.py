"""The calls this package is timed on, and their float64 results.

Three kinds of call, each through a public entry point:

  layer  one pass of a compiled decoder layer (compile_decoder + run_layer): prefill
         (context 0) or a decode step of `sequence` new tokens per sequence over
         `context` cached ones, dense or MoE FFN, fp32 / bf16 / int8 weights;
  moe    the MoE block alone through the C ABI: route, expert GEMMs, weighted combine;
  paged  paged attention alone through the C ABI, every sequence with its own length.

Whole MoE layers run from a routing trace: their router input carries the rounding of
everything before it, so a near tie between two experts could go either way.  The
`moe` kind routes on the device from fp32 rows given exactly.
"""
from __future__ import annotations

import ctypes
import math
import zlib

import numpy as np
import torch

from schedforge_amd import _abi
from schedforge_amd.configs import DecoderConfig
from schedforge_amd.layer import DecoderData, compile_decoder, run_layer

WEIGHT_STD = 0.02   # projection, expert and router weights
EPS, THETA = 1e-5, 10000.0

# (hidden, intermediate, query heads, kv heads, head dim): the realistic profiles'
# tiny / medium / large models and the bf16 decode benchmark's
TINY = (512, 1376, 8, 2, 64)
MEDIUM = (1024, 2816, 16, 4, 64)
BASE = (2048, 5632, 16, 4, 128)
LARGE = (4096, 11008, 32, 8, 128)
# expert width of the MoE configurations at hidden 2048
MOE_BASE = (2048, 1408, 16, 4, 128)


def _layer(model, dtype, batch, sequence, context=0, experts=0, name=None):
    h, i, hq, hkv, d = model
    c = {"kind": "layer", "dtype": dtype, "batch": batch, "sequence": sequence, "context": context,
         "hidden": h, "intermediate": i, "query_heads": hq, "kv_heads": hkv, "head_dim": d,
         "experts": experts, "top_k": 2 if experts else 0}
    return {"name": name, **c} if name else c


def _moe(model, dtype, tokens, experts=8, name=None):
    c = {"kind": "moe", "dtype": dtype, "tokens": tokens, "hidden": model[0], "intermediate": model[1],
         "experts": experts, "top_k": 2}
    return {"name": name, **c} if name else c


def _paged(batch, hq, hkv, d, longest, seq_q=1, dtype="bf16", name=None):
    c = {"kind": "paged", "dtype": dtype, "batch": batch, "query_heads": hq, "kv_heads": hkv,
         "head_dim": d, "longest": longest, "seq_q": seq_q, "page_tokens": 16}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the fp32 parity configuration: a short prompt through a small layer, the smallest call
        _layer((256, 688, 4, 2, 64), "f32", 1, 128, name="f32-prefill-128"),
        # fp32 is the operator interface's own type: a 2048-token prompt of the medium profile
        _layer(MEDIUM, "f32", 1, 2048, name="f32-prefill-2048"),
        # the headline prefill: one 8192-token prompt, the largest call
        _layer((4096, 14336, 32, 8, 128), "bf16", 1, 8192, name="bf16-prefill-8192"),
        # an ordinary prompt: the large profile at 512 tokens
        _layer(LARGE, "bf16", 1, 512, name="bf16-prefill-512"),
        # int8 weights under prefill: two prompts of an odd length
        _layer(LARGE, "w8", 2, 777, name="w8-prefill-2x777"),
        # the MoE prefill configuration, eight experts, top-2
        _layer(MOE_BASE, "bf16", 4, 512, experts=8, name="bf16-moe-prefill-4x512"),
        # the MoE block of an int8 model on a ragged batch of tokens, routed on the device
        _moe(MOE_BASE, "w8", 500, name="w8-moe-block-500"),
        # the bf16 decode configuration: 16 sequences at 4096 cached tokens
        _layer(BASE, "bf16", 16, 1, 4096, name="bf16-decode-16"),
        # one user's decode step of the large profile at 4096 cached tokens
        _layer(LARGE, "bf16", 1, 1, 4096, name="bf16-decode-1"),
        # the int8 MoE decode configuration: 64 sequences at 8192 cached tokens
        _layer((4096, 14336, 32, 8, 128), "w8", 64, 1, 8192, experts=8, name="w8-moe-decode-64"),
        # a step of several tokens per sequence over a ragged cache (drafted tokens, the
        # tail of a prompt)
        _layer(BASE, "bf16", 8, 5, 3000, name="bf16-decode-8x5"),
        # decode attention over a serving batch whose sequences have lengths 1 .. 8192
        _paged(32, 32, 8, 128, 8192, name="bf16-paged-32-ragged"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("prefill", "prefill", "prefill", "decode", "decode", "chunk", "moe-prefill",
                       "moe-decode", "moe", "paged"))
    if kind == "prefill":
        dtype = rng.choice(("f32", "bf16", "w8"))
        model = rng.choice((TINY, MEDIUM, BASE, LARGE))
        batch = _log(rng, 1, 8)
        # fp32 products cost more per FLOP: their rows are held to what the listed
        # 2048-row medium layer takes
        rows = _log(rng, 64, 4096 if dtype != "f32" else max(96, 2048 * 1024 * 1024 // (model[0] * model[0])))
        return _layer(model, dtype, batch, max(24, min(2500, rows // batch)))
    if kind == "decode":
        return _layer(rng.choice((TINY, MEDIUM, BASE, LARGE)), rng.choice(("f32", "bf16", "bf16", "w8")),
                      _log(rng, 1, 64), 1, _log(rng, 64, 6000))
    if kind == "chunk":
        return _layer(rng.choice((TINY, MEDIUM, BASE)), rng.choice(("bf16", "w8")), _log(rng, 1, 8),
                      rng.randint(2, 8), _log(rng, 64, 3000))
    if kind == "moe-prefill":
        return _layer(MOE_BASE, rng.choice(("bf16", "w8")), _log(rng, 1, 4), _log(rng, 64, 700), experts=8)
    if kind == "moe-decode":
        return _layer(MOE_BASE, rng.choice(("bf16", "w8")), _log(rng, 1, 64), 1, _log(rng, 64, 6000), experts=8)
    if kind == "moe":
        return _moe(MOE_BASE, rng.choice(("bf16", "w8")), _log(rng, 16, 3000))
    return _paged(_log(rng, 1, 40), 32, 8, 128, _log(rng, 128, 8192), rng.choice((1, 1, 1, 4)))


# ---------------------------------------------------------------- inputs
def _gen(seed, name):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))


def _normal(seed, name, shape, std=1.0):
    return torch.empty(shape, device="cuda").normal_(0.0, std, generator=_gen(seed, name))


def _bf16(t):
    return t.to(torch.bfloat16).to(torch.float32)


def _trace(case, seed):
    """Routing trace [rows][k]: distinct experts per token under a moderate skew, weights summing to 1."""
    rows = case["batch"] * case["sequence"]
    logits = _normal(seed, "route", (rows, case["experts"])) + _normal(seed, "skew", (case["experts"],), 0.5)
    top = torch.topk(logits, case["top_k"], dim=1)
    return top.indices.to(torch.int32), torch.softmax(top.values, dim=1)


def _layer_data(case, seed):
    h, i, d = case["hidden"], case["intermediate"], case["head_dim"]
    kvd = case["kv_heads"] * d
    rows = case["batch"] * case["sequence"]
    low = case["dtype"] != "f32"
    data = DecoderData()
    data.input = _normal(seed, "x", (rows, h))
    data.rms1_weight = 1.0 + 0.1 * _normal(seed, "rms1", (h,))
    data.rms2_weight = 1.0 + 0.1 * _normal(seed, "rms2", (h,))
    data.query_weight = _normal(seed, "wq", (h, h), WEIGHT_STD)
    data.key_weight = _normal(seed, "wk", (h, kvd), WEIGHT_STD)
    data.value_weight = _normal(seed, "wv", (h, kvd), WEIGHT_STD)
    data.output_weight = _normal(seed, "wo", (h, h), WEIGHT_STD)
    if case["experts"]:
        data.router_weight = _normal(seed, "router", (h, case["experts"]), WEIGHT_STD)
        data.w1 = lambda e: _normal(seed, f"w1.{e}", (h, i), WEIGHT_STD)
        data.w3 = lambda e: _normal(seed, f"w3.{e}", (h, i), WEIGHT_STD)
        data.w2 = lambda e: _normal(seed, f"w2.{e}", (i, h), WEIGHT_STD)
        data.routing_trace = _trace(case, seed)
    else:
        data.gate_weight = _normal(seed, "wg", (h, i), WEIGHT_STD)
        data.up_weight = _normal(seed, "wu", (h, i), WEIGHT_STD)
        data.down_weight = _normal(seed, "wd", (i, h), WEIGHT_STD)
    if case["context"]:
        shape = (case["batch"], case["kv_heads"], case["context"], d)
        data.cached_key = _normal(seed, "k", shape)
        data.cached_value = _normal(seed, "v", shape)
    if low:
        data.input = _bf16(data.input)
    return data


def _prepare_layer(case, seed):
    cfg = DecoderConfig(
        batch=case["batch"], sequence=case["sequence"], hidden=case["hidden"],
        intermediate=case["intermediate"], query_heads=case["query_heads"], kv_heads=case["kv_heads"],
        head_dim=case["head_dim"], rms_epsilon=EPS, rope_theta=THETA, ffn="moe" if case["experts"] else "dense",
        experts=case["experts"] or 4, top_k=case["top_k"] or 2, context_sequence=case["context"],
        dtype=case["dtype"])
    data = _layer_data(case, seed)
    perm = None
    if case["context"]:
        pages = case["batch"] * ((case["context"] + cfg.page_tokens - 1) // cfg.page_tokens)
        perm = np.random.RandomState(seed % (1 << 32)).permutation(pages).astype(np.int32)
    plan = compile_decoder(cfg, data, "cuda", page_permutation=perm)
    x = data.input.contiguous()
    return {"kind": "layer", "plan": plan, "x": x, "out": torch.empty_like(x)}


def _moe_weight(case, seed, name, e):
    shape = (case["intermediate"], case["hidden"]) if name == "w2" else (case["hidden"], case["intermediate"])
    return _normal(seed, f"{name}.{e}", shape, WEIGHT_STD)


def _prepare_moe(case, seed):
    lib = _abi.load()
    t, h, i, e, k = (case[n] for n in ("tokens", "hidden", "intermediate", "experts", "top_k"))
    i8 = case["dtype"] == "w8"
    stream = torch.cuda.current_stream().cuda_stream
    tiled = all(lib.sfg_hip_preferred_weight_layout_v1(t * k, kk, 1) == _abi.LAYOUT_TILED for kk in (h, i))
    layout = _abi.LAYOUT_TILED if tiled else _abi.LAYOUT_NK

    def pack(names, rows, depth):
        w = torch.empty((e, rows, depth), dtype=torch.int8 if i8 else torch.int16, device="cuda")
        s = torch.empty((e, rows), device="cuda") if i8 else None
        for g in range(e):
            at = 0
            for name in names:
                src = _moe_weight(case, seed, name, g)
                n = src.shape[1]
                if i8:
                    _abi.check(lib.sfg_hip_quantize_weight_v1(src.data_ptr(), depth, n, w[g, at].data_ptr(),
                                                              s[g, at:].data_ptr(), layout, stream))
                else:
                    _abi.check(lib.sfg_hip_pack_weight_v1(src.data_ptr(), depth, n, n, w[g, at].data_ptr(),
                                                          _abi.BF16, layout, stream))
                torch.cuda.synchronize()
                at += n
        return w, s

    s = {"kind": "moe", "lib": lib, "case": case, "layout": layout, "dtype": _abi.I8 if i8 else _abi.BF16}
    s["x"] = _bf16(_normal(seed, "x", (t, h)))
    s["x16"] = s["x"].to(torch.bfloat16)
    s["residual"] = _normal(seed, "residual", (t, h))
    s["router"] = _normal(seed, "router", (h, e), WEIGHT_STD)
    s["bias"] = _normal(seed, "bias", (e,), 0.5)
    s["w13"], s["s13"] = pack(("w1", "w3"), 2 * i, h)
    s["w2"], s["s2"] = pack(("w2",), h, i)
    new = lambda *shape, dtype=torch.int32: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
    s["ids"], s["wts"] = new(t, k), new(t, k, dtype=torch.float32)
    s["counts"], s["offsets"] = new(e), new(e + 1)
    s["token_ids"], s["slots"], s["position"] = new(t * k), new(t * k), new(t, k)
    s["rweights"] = new(t * k, dtype=torch.float32)
    s["act"], s["y"] = new(t * k, i, dtype=torch.int16), new(t * k, h, dtype=torch.float32)
    s["out"] = new(t, h, dtype=torch.float32)
    route = lib.sfg_hip_moe_route_workspace_v1(t, e, k)
    experts = lib.sfg_hip_moe_expert_workspace_v1(t, h, i, e, k)
    s["ws"] = new(max(1, route, experts), dtype=torch.uint8)
    return s


def _lengths(case, seed):
    lo = case["seq_q"]
    g = np.random.RandomState((seed * 7 + 1) % (1 << 32))
    lens = g.randint(lo, case["longest"] + 1, case["batch"])
    lens[g.randint(case["batch"])] = case["longest"]
    return lens.astype(np.int32)


def _paged_inputs(case, seed):
    """Pools, page table, lengths and queries of the paged call (bf16 values)."""
    b, hkv, d, pt = case["batch"], case["kv_heads"], case["head_dim"], case["page_tokens"]
    per = (case["longest"] + pt - 1) // pt
    perm = np.random.RandomState((seed * 5 + 3) % (1 << 32)).permutation(b * per).astype(np.int32)
    return {"table": torch.from_numpy(perm.reshape(b, per)).cuda(),
            "lens": torch.from_numpy(_lengths(case, seed)).cuda(),
            "k": _normal(seed, "k", (b * per, hkv, pt, d)).to(torch.bfloat16),
            "v": _normal(seed, "v", (b * per, hkv, d, pt)).to(torch.bfloat16),
            "q": _normal(seed, "q", (b, case["query_heads"], case["seq_q"], d))}


def _prepare_paged(case, seed):
    lib = _abi.load()
    s = {"kind": "paged", "lib": lib, "case": case, **_paged_inputs(case, seed)}
    s["out"] = torch.empty_like(s["q"])
    n = lib.sfg_hip_attn_paged_workspace_v1(case["batch"], case["query_heads"], case["kv_heads"], case["seq_q"],
                                            case["head_dim"], _abi.BF16, case["longest"], case["page_tokens"], 0)
    s["ws"] = torch.empty(max(1, n), dtype=torch.uint8, device="cuda")
    return s


def prepare(case, seed):
    return {"layer": _prepare_layer, "moe": _prepare_moe, "paged": _prepare_paged}[case["kind"]](case, seed)


# ---------------------------------------------------------------- one pass
def run(s):
    if s["kind"] == "layer":
        run_layer(s["plan"], s["x"], s["out"])
        return s["out"]
    lib, case, stream = s["lib"], s["case"], torch.cuda.current_stream().cuda_stream
    p = lambda name: s[name].data_ptr() if s[name] is not None else None  # noqa: E731
    if s["kind"] == "moe":
        t, h, i, e, k = (case[n] for n in ("tokens", "hidden", "intermediate", "experts", "top_k"))
        _abi.check(lib.sfg_hip_moe_route_v1(p("x"), p("router"), p("bias"), t, h, e, k, p("ids"), p("wts"),
                                            p("counts"), p("offsets"), p("token_ids"), p("slots"), p("rweights"),
                                            p("position"), p("ws"), s["ws"].numel(), stream))
        _abi.check(lib.sfg_hip_moe_experts_v1(p("x16"), p("offsets"), p("token_ids"), p("w13"), p("s13"), p("w2"),
                                              p("s2"), s["dtype"], s["layout"], p("act"), p("y"), t, h, i, e, k,
                                              p("ws"), s["ws"].numel(), stream))
        _abi.check(lib.sfg_hip_moe_combine_v1(p("y"), p("position"), p("wts"), p("residual"), p("out"), t, h, k,
                                              stream))
        return {"out": s["out"], "ids": s["ids"], "weights": s["wts"], "counts": s["counts"]}
    per = s["table"].shape[1]
    _abi.check(lib.sfg_hip_attn_paged_v1(
        p("q"), p("k"), p("v"), _abi.BF16, p("table"), p("lens"), p("out"), _abi.F32, case["batch"],
        case["query_heads"], case["kv_heads"], case["seq_q"], case["head_dim"], case["page_tokens"], per,
        s["k"].shape[0], case["longest"], 1, 0, ctypes.c_float(0.0), 0, p("ws"), s["ws"].numel(), stream))
    return s["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def _pairs(s, keys):
    """Allowed (query, key) pairs of s queries over `keys` keys, query i seeing keys up to keys - s + i."""
    return sum(max(0, keys - s + i + 1) for i in range(s))


def work(case):
    wb = {"f32": 4, "bf16": 2, "w8": 1}[case["dtype"]]
    if case["kind"] == "paged":
        b, hq, hkv, d, s = (case[n] for n in ("batch", "query_heads", "kv_heads", "head_dim", "seq_q"))
        mean = (s + case["longest"]) / 2.0   # lengths are even over [seq_q, longest]
        return {"bytes": b * (2 * hkv * mean * d * wb + 2 * hq * s * d * 4),
                "flops": 4.0 * b * hq * d * s * mean}
    h, i, e, k = case["hidden"], case["intermediate"], case["experts"], case["top_k"]
    if case["kind"] == "moe":
        t = case["tokens"]
        return {"bytes": e * 3 * h * i * wb + h * e * 4 + t * h * 4 * 3,
                "flops": 6.0 * t * k * h * i + 2.0 * t * h * e}
    b, s, d, hq, hkv = (case[n] for n in ("batch", "sequence", "head_dim", "query_heads", "kv_heads"))
    rows, kvd, ctx = b * s, hkv * d, case["context"]
    # a decode step attends over the cache alone and discards its own K / V: Q columns only
    proj = h * (h if ctx else h + 2 * kvd) + h * h
    flops = 2.0 * rows * proj + 4.0 * d * hq * b * _pairs(s, ctx or s)
    nbytes = proj * wb + rows * h * 4 * 2
    if ctx:
        nbytes += 2 * b * hkv * ctx * d * (4 if case["dtype"] == "f32" else 2)
    if e:
        flops += 6.0 * rows * k * h * i
        nbytes += min(e, rows * k) * 3 * h * i * wb
    else:
        flops += 6.0 * rows * h * i
        nbytes += 3 * h * i * wb
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times what each kind is off its float64 result by (2-norm, worst case seen):
    # paged 1.8e-3, the MoE block 4.5e-4, 16-bit layers 3.8e-3, fp32 layers 2.9e-6
    if case["kind"] == "paged":
        return {"rel": 7e-3}
    if case["kind"] == "moe":
        return {"rel": 2e-3, "differ": 0.001}
    return {"rel": 1e-5} if case["dtype"] == "f32" else {"rel": 1.5e-2}


# ---------------------------------------------------------------- float64 results
def _w64(w, dtype):
    """An fp32 weight [K][N] as the device holds it -- rounded to bf16, or int8 times its column's scale."""
    if dtype == "bf16":
        w = _bf16(w)
    if dtype != "w8":
        return w.double()
    top = w.abs().amax(dim=0)
    s = torch.where(top > 0, top / 127.0, torch.ones_like(top))
    v = w / s
    q = torch.clamp(torch.sign(v) * torch.floor(v.abs() + 0.5), -127, 127)
    return q.double() * s.double()


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * w.double()


def _rope64(x):
    """Rotates x [..., S, D] at positions 0 .. S - 1; angles are float32 products, as the package defines them."""
    s, d = x.shape[-2:]
    freq = np.array([math.pow(THETA, -2.0 * i / d) for i in range(d // 2)]).astype(np.float32)
    ang = torch.from_numpy((np.arange(s, dtype=np.float32)[:, None] * freq[None, :]).astype(np.float64)).cuda()
    c, n = torch.cos(ang), torch.sin(ang)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * n, a * n + b * c), dim=-1).reshape(x.shape)


def _attend64(q, k, v):
    """q [R, S, D] of one K/V head against k, v [L, D]; query i sees keys up to L - S + i."""
    r, s, d = q.shape
    keys = k.shape[0]
    hidden = None
    if s > 1:
        hidden = torch.arange(keys, device="cuda")[None, :] > (keys - s + torch.arange(s, device="cuda"))[:, None]
    out = torch.empty_like(q)
    for i in range(r):
        a = q[i] @ k.T / math.sqrt(d)
        if hidden is not None:
            a.masked_fill_(hidden, -math.inf)
        out[i] = torch.softmax(a, dim=1) @ v
    return out


def _experts64(case, x, ids, wts, w1, w3, w2):
    """sum over a token's experts of weight * W2 ((x W1) * silu(x W3))."""
    out = torch.zeros_like(x)
    for e in range(case["experts"]):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if not tok.numel():
            continue
        a = x[tok]
        act = (a @ _w64(w1(e), case["dtype"])) * torch.nn.functional.silu(a @ _w64(w3(e), case["dtype"]))
        out.index_add_(0, tok, (act @ _w64(w2(e), case["dtype"])) * wts[tok, slot].double()[:, None])
    return out


def exact(case, seed):
    if case["kind"] == "paged":
        t = _paged_inputs(case, seed)
        b, hq, hkv, d, s = (case[n] for n in ("batch", "query_heads", "kv_heads", "head_dim", "seq_q"))
        out = torch.empty((b, hq, s, d), dtype=torch.float64, device="cuda")
        g = hq // hkv
        for n in range(b):
            keys = int(t["lens"][n])
            pages = t["table"][n].long()
            k = t["k"][pages].double().permute(1, 0, 2, 3).reshape(hkv, -1, d)[:, :keys]
            v = t["v"][pages].double().permute(1, 0, 3, 2).reshape(hkv, -1, d)[:, :keys]
            for j in range(hkv):
                out[n, j * g:(j + 1) * g] = _attend64(t["q"][n, j * g:(j + 1) * g].double(), k[j], v[j])
        return out
    if case["kind"] == "moe":
        t, h, e, k = (case[n] for n in ("tokens", "hidden", "experts", "top_k"))
        x = _bf16(_normal(seed, "x", (t, h))).double()
        logits = x @ _normal(seed, "router", (h, e), WEIGHT_STD).double() + _normal(seed, "bias", (e,), 0.5).double()
        top = torch.topk(logits, k, dim=1)
        wts = torch.softmax(top.values, dim=1)
        out = _experts64(case, x, top.indices, wts, *(lambda g, n=n: _moe_weight(case, seed, n, g)
                                                     for n in ("w1", "w3", "w2")))
        ids = top.indices.to(torch.int32)
        return {"out": out + _normal(seed, "residual", (t, h)).double(), "ids": ids, "weights": wts,
                "counts": torch.bincount(top.indices.reshape(-1), minlength=e).to(torch.int32)}
    data = _layer_data(case, seed)
    dt = case["dtype"]
    b, s, d, hq, hkv, h = (case[n] for n in ("batch", "sequence", "head_dim", "query_heads", "kv_heads", "hidden"))
    g = hq // hkv
    x = data.input.double()
    xn = _rms64(x, data.rms1_weight)

    def heads(w, n):
        return (xn @ _w64(w, dt)).reshape(b, s, n, d).transpose(1, 2)

    q = _rope64(heads(data.query_weight, hq))
    if case["context"]:
        low = _bf16 if dt != "f32" else (lambda t: t)
        key, value = (lambda n, j: low(data.cached_key[n, j]).double()), (lambda n, j: low(data.cached_value[n, j]).double())
    else:
        kk, vv = _rope64(heads(data.key_weight, hkv)), heads(data.value_weight, hkv)
        key, value = (lambda n, j: kk[n, j]), (lambda n, j: vv[n, j])
    attn = torch.empty((b, hq, s, d), dtype=torch.float64, device="cuda")
    for n in range(b):
        for j in range(hkv):
            attn[n, j * g:(j + 1) * g] = _attend64(q[n, j * g:(j + 1) * g], key(n, j), value(n, j))
    r1 = attn.transpose(1, 2).reshape(b * s, h) @ _w64(data.output_weight, dt) + x
    xn2 = _rms64(r1, data.rms2_weight)
    if case["experts"]:
        ids, wts = data.routing_trace
        return r1 + _experts64(case, xn2, ids, wts, data.w1, data.w3, data.w2)
    act = torch.nn.functional.silu(xn2 @ _w64(data.gate_weight, dt)) * (xn2 @ _w64(data.up_weight, dt))
    return r1 + act @ _w64(data.down_weight, dt)
