"""The work that programs built on this library have it do, as measurable cases.

Every case is a dict of plain values; `kind` says which path it takes:

  gemv         one Q4_0 / Q8_0 Linear with a few rows, called eagerly (the smallest call: a single projection of a decode token)
  decode       a decode step through some decoder layers: the quantized projections with RMSNorm, SiLU * up and the residual adds
               between them (the attention core is not this library's), captured once in a HIP graph and replayed per token
  linear       a Q4_0 / Q8_0 / Q4_K / Q6_K Linear over a prompt
  w8a8         per-token dynamic int8 activations x int8 weights, from a decode token to a prompt
  w4a16        bf16 activations x group-quantized uint4 weights, from a decode token to a prompt
  moe_prefill  the expert FFN of an MoE layer over a prompt, experts of Zipf popularity
  moe_decode   a decode step through MoE layers (RMSNorm, router gate, expert FFN, residual add), captured as above
  attention    the activation matmuls of an attention layer with the softmax between them: prompt or decode token
  sampling     softmax and top-k over rows of a vocabulary's logits

Sizes are those of the Qwen3-4B, Qwen3-32B and Qwen3-30B-A3B shaped layers that the benchmark and the tests use, or generic.
"""
import math
import types

import numpy as np
import torch

from mllm_amd import _lib, qlinear as ql, synth

BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}  # weights and bytes of a block
QTYPE = {"q4_0": ql.Q4_0, "q8_0": ql.Q8_0, "q4_k": ql.Q4_K, "q6_k": ql.Q6_K}
LARGEST = 2048 * 9728 * 2560  # multiply-adds of the largest prompt case


def listed():
    return [
        # one projection of a decode token through the eager call: launch latency and host path
        {"name": "gemv_q4_0_1x6144x2048", "kind": "gemv", "scheme": "q4_0", "rows": 1, "n": 6144, "k": 2048, "x": "f32", "bias": False},
        # a decode token of one sequence through a Q4_0 model
        {"name": "decode_q4_0_1", "kind": "decode", "scheme": "q4_0", "rows": 1, "layers": 6, "hidden": 2560, "attn": 4096, "kv": 1024, "inter": 9728},
        # a few sequences (or a speculative run of five tokens) through the shipped K-quant recipe: down projections in Q6_K
        {"name": "decode_kq_5", "kind": "decode", "scheme": "kq", "rows": 5, "layers": 6, "hidden": 2560, "attn": 4096, "kv": 1024, "inter": 9728},
        # a long prompt through a Q4_0 projection
        {"name": "linear_q4_0_2048x9728x2560", "kind": "linear", "scheme": "q4_0", "rows": 2048, "n": 9728, "k": 2560, "x": "bf16", "bias": False},
        # a short prompt of a ragged length through a K-quant down projection
        {"name": "linear_q6_k_131x2560x9728", "kind": "linear", "scheme": "q6_k", "rows": 131, "n": 2560, "k": 9728, "x": "f32", "bias": True},
        # prompts through the int8 and the 4-bit weight-only checkpoints
        {"name": "w8a8_2048x6144x2048", "kind": "w8a8", "rows": 2048, "n": 6144, "k": 2048, "x": "bf16", "bias": False},
        {"name": "w4a16_2048x9728x2560", "kind": "w4a16", "rows": 2048, "n": 9728, "k": 2560, "group": 128, "bias": False},
        # a chunk of a few dozen tokens, a ragged count
        {"name": "w4a16_93x2048x6144", "kind": "w4a16", "rows": 93, "n": 2048, "k": 6144, "group": 128, "bias": True},
        # a prompt through the experts of an MoE layer
        {"name": "moe_prefill_q4_0_512", "kind": "moe_prefill", "scheme": "q4_0", "tokens": 512, "hidden": 2048, "inter": 768, "experts": 128, "top": 8},
        # a decode token of eight sequences through two MoE layers of the shipped K-quant recipe
        {"name": "moe_decode_kq_8", "kind": "moe_decode", "scheme": "kq", "tokens": 8, "layers": 2, "hidden": 2048, "inter": 768, "experts": 128, "top": 8},
        # a prompt's attention (8 KV heads, four query heads each), a ragged length
        {"name": "attention_f32_777", "kind": "attention", "x": "f32", "kv_heads": 8, "group": 4, "queries": 777, "keys": 777, "head": 128},
        # the next token of eight sequences
        {"name": "sampling_8x151936", "kind": "sampling", "rows": 8, "vocab": 151936, "top": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, of):
    return max(1, round(_log(rng, lo, hi) / of)) * of


def _rows_under_largest(rows, n, k):
    return max(1, min(rows, LARGEST // (n * k)))


def draw(rng):
    kind = rng.choice(["gemv", "decode", "linear", "linear", "w8a8", "w8a8", "w4a16", "w4a16", "moe_prefill", "moe_decode", "attention", "sampling"])
    if kind == "gemv":
        return {"kind": kind, "scheme": rng.choice(["q4_0", "q8_0"]), "rows": _log(rng, 1, 8), "n": _multiple(rng, 256, 9728, 8),
                "k": _multiple(rng, 256, 9728, 32), "x": rng.choice(["f32", "bf16"]), "bias": rng.random() < 0.3}
    if kind == "decode":
        scheme = rng.choice(["q4_0", "q8_0", "kq"])
        return {"kind": kind, "scheme": scheme, "rows": _log(rng, 1, 8 if scheme == "kq" else 32), "layers": rng.randint(2, 4 if scheme == "q8_0" else 6),
                "hidden": rng.choice([1024, 2048, 2560]), "attn": rng.choice([2048, 4096]), "kv": rng.choice([512, 1024]),
                "inter": rng.choice([3072, 6144, 9728])}
    if kind == "linear":
        scheme = rng.choice(["q4_0", "q8_0", "q4_k", "q6_k"])
        n, k = _multiple(rng, 1024, 9728, 8), _multiple(rng, 1024, 9728, BLOCK[scheme][0])
        return {"kind": kind, "scheme": scheme, "rows": _rows_under_largest(_log(rng, 49, 2048), n, k), "n": n, "k": k, "x": rng.choice(["f32", "bf16"]),
                "bias": rng.random() < 0.3}
    if kind == "w8a8":
        n, k = _multiple(rng, 1024, 9728, 8), _multiple(rng, 1024, 9728, 64)
        return {"kind": kind, "rows": _rows_under_largest(_log(rng, 1, 2048), n, k), "n": n, "k": k, "x": rng.choice(["f32", "bf16"]), "bias": rng.random() < 0.3}
    if kind == "w4a16":
        group = rng.choice([64, 128, 128])
        n, k = _multiple(rng, 1024, 9728, 8), _multiple(rng, 1024, 9728, group)
        return {"kind": kind, "rows": _rows_under_largest(_log(rng, 1, 2048), n, k), "n": n, "k": k, "group": group, "bias": rng.random() < 0.3}
    if kind == "moe_prefill":
        return {"kind": kind, "scheme": rng.choice(["q4_0", "q8_0", "kq"]), "tokens": _log(rng, 96, 768), "hidden": rng.choice([1024, 2048]),
                "inter": rng.choice([512, 768]), "experts": rng.choice([64, 128]), "top": rng.choice([4, 8])}
    if kind == "moe_decode":
        return {"kind": kind, "scheme": rng.choice(["q4_0", "q8_0", "kq"]), "tokens": _log(rng, 1, 32), "layers": rng.randint(1, 2),
                "hidden": rng.choice([1024, 2048]), "inter": rng.choice([512, 768]), "experts": rng.choice([64, 128]), "top": rng.choice([4, 8])}
    if kind == "attention":
        kv, head = rng.choice([4, 8]), rng.choice([64, 128])
        if rng.random() < 0.5:  # a decode token against a cache
            queries, keys = 1, _log(rng, 256, 8192)
        else:
            queries = keys = _log(rng, 64, 1024)
        return {"kind": kind, "x": rng.choice(["f32", "bf16"]), "kv_heads": kv, "group": rng.choice([1, 4]), "queries": queries, "keys": keys, "head": head}
    return {"kind": kind, "rows": _log(rng, 1, 16), "vocab": _multiple(rng, 32000, 151936, 8), "top": rng.randint(1, 64)}


# ----------------------------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(shape, g, dtype="f32"):
    t = torch.randn(shape, device="cuda", generator=g)
    return t.to(torch.bfloat16) if dtype == "bf16" else t


def _weight(scheme, n, k, g, layout="gemv"):
    if scheme in ("q4_k", "q6_k"):
        return ql.PackedKWeight.synthetic(QTYPE[scheme], n, k, g, layout=layout)
    return ql.PackedQWeight.synthetic(QTYPE[scheme], n, k, g, layout=layout)


def _bytes(nbytes):
    return torch.empty(max(1, nbytes), dtype=torch.uint8, device="cuda")


def _experts(scheme, e, n, k, g, layout="gemv"):
    if scheme in ("q4_k", "q6_k"):
        return ql.PackedKExperts.synthetic(QTYPE[scheme], e, n, k, g)
    return ql.PackedExperts.synthetic(QTYPE[scheme], e, n, k, g, layout=layout)


def _schemes(scheme):
    """formats of (all other projections, the down projection)"""
    return ("q4_k", "q6_k") if scheme == "kq" else (scheme, scheme)


def _captured(step):
    """a program's decode loop: one eager step, then the step as a graph"""
    _lib.check(_lib.lib().mllm_hip_init(torch.cuda.current_device()), "mllm_hip_init")
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = step()
    return graph, outputs


def _prepare_decode(c, s, g):
    rows, h, a, kv, inter = c["rows"], c["hidden"], c["attn"], c["kv"], c["inter"]
    main, down = _schemes(c["scheme"])
    kq = c["scheme"] == "kq"
    layers = []
    for _ in range(c["layers"]):
        layers.append(types.SimpleNamespace(
            q=_weight(main, a, h, g), k=_weight(main, kv, h, g), v=_weight(main, kv, h, g), o=_weight(main, h, a, g),
            gate=_weight(main, inter, h, g), up=_weight(main, inter, h, g), down=_weight(down, h, inter, g),
            norm1=1 + 0.1 * _randn((h,), g), norm2=1 + 0.1 * _randn((h,), g)))
    s.token = _randn((rows, h), g)
    s.x = torch.empty_like(s.token)
    new = lambda n: torch.empty((rows, n), dtype=torch.float32, device="cuda")  # noqa: E731
    outs = [[new(a), new(kv), new(kv)] for _ in layers]
    o, x1, gu, d = new(h), new(h), [new(inter), new(inter)], new(h)
    if kq:
        ws = {n: ql.kq_workspace(rows, k, n) for n, k in ((a + 2 * kv, h), (h, a), (2 * inter, h))}
        ws_down = ql.kq_workspace(rows, inter, h)
    elif rows >= 3:
        ws = {n: ql.gemv_workspace(rows, k, n) for n, k in ((a + 2 * kv, h), (h, a), (2 * inter, h))}
        ws_down = ql.gemv_workspace(rows, inter, h)
    else:
        ws, ws_down = {}, None

    def step():
        x = s.x
        for layer, qkv in zip(layers, outs):
            if kq:
                ql.linear_kq_multi([layer.q, layer.k, layer.v], ql.rmsnorm(x, layer.norm1, 1e-6), None, qkv, workspace=ws[a + 2 * kv])
                ql.linear_kq_multi([layer.o], qkv[0], None, [o], workspace=ws[h])
                y = ql.add(o, x)
                ql.linear_kq_multi([layer.gate, layer.up], ql.rmsnorm(y, layer.norm2, 1e-6), None, gu, workspace=ws[2 * inter])
                ql.linear_kq_multi([layer.down], ql.silu_mul(gu[0], gu[1]), None, [d], workspace=ws_down)
                x = ql.add(d, y)
            elif rows <= 8:
                _, image = ql.rmsnorm(x, layer.norm1, 1e-6, want_image=True)
                ql.linear_q_gemv_fused([layer.q, layer.k, layer.v], image, M=rows, image=True, outs=qkv, workspace=ws.get(a + 2 * kv))
                ql.linear_q_gemv_fused([layer.o], qkv[0], residuals=[x], outs=[x1], workspace=ws.get(h))
                _, image = ql.rmsnorm(x1, layer.norm2, 1e-6, want_image=True)
                image = ql.mlp_gate_up(layer.gate, layer.up, image, M=rows, image=True, want_h=False, want_image=True)
                x = ql.linear_q_gemv_fused([layer.down], image, M=rows, image=True, residuals=[x1], workspace=ws_down)[0]
            else:
                ql.linear_q_gemv_multi([layer.q, layer.k, layer.v], ql.rmsnorm(x, layer.norm1, 1e-6), outs=qkv, workspace=ws[a + 2 * kv])
                y = ql.add(ql.linear_q_gemv_multi([layer.o], qkv[0], outs=[o], workspace=ws[h])[0], x)
                ql.linear_q_gemv_multi([layer.gate, layer.up], ql.rmsnorm(y, layer.norm2, 1e-6), outs=gu, workspace=ws[2 * inter])
                x = ql.add(ql.linear_q_gemv_multi([layer.down], ql.silu_mul(gu[0], gu[1]), outs=[d], workspace=ws_down)[0], y)
        return {"x": x, "qkv": outs}

    s.keep = (layers, ws, ws_down)
    s.graph, s.outputs = _captured(step)


def _prepare_moe_decode(c, s, g):
    t, h, inter, e, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top"]
    main, down = _schemes(c["scheme"])
    layers = []
    for _ in range(c["layers"]):
        layers.append(types.SimpleNamespace(gate=_experts(main, e, inter, h, g), up=_experts(main, e, inter, h, g), down=_experts(down, e, h, inter, g),
                                            norm=1 + 0.1 * _randn((h,), g), router=0.05 * _randn((e, h), g)))
    L = _lib.lib()
    s.token = _randn((t, h), g)
    s.x = torch.empty_like(s.token)
    ws = _bytes((L.mllm_hip_moe_kq_workspace_bytes if c["scheme"] == "kq" else L.mllm_hip_moe_workspace_bytes)(t, h, inter, e, k))
    scores = torch.empty((t, e), dtype=torch.float32, device="cuda")
    ffn = ql.moe_ffn_kq if c["scheme"] == "kq" else ql.moe_ffn_q

    def step():
        x, routes = s.x, []
        for layer in layers:
            y = ql.rmsnorm(x, layer.norm, 1e-6)
            ids, weights = ql.moe_gate(y, layer.router, k, scores=scores)
            x = ql.add(ffn(layer.gate, layer.up, layer.down, y, ids, weights, workspace=ws), x)
            routes.append((ids, weights))
        return {"x": x, "routes": routes}

    s.keep = (layers, ws, scores)
    s.graph, s.outputs = _captured(step)


def prepare(case, seed):
    c, s, g = case, types.SimpleNamespace(), _gen(seed)
    s.case, kind = c, case["kind"]
    L = _lib.lib()
    if kind == "gemv":
        s.w = _weight(c["scheme"], c["n"], c["k"], g)
        s.x = _randn((c["rows"], c["k"]), g, c["x"])
        s.bias = _randn((c["n"],), g) if c["bias"] else None
        s.y = torch.empty((c["rows"], c["n"]), dtype=torch.float32, device="cuda")
        s.ws = ql.gemv_workspace(c["rows"], c["k"], c["n"]) if c["rows"] >= 3 else None
    elif kind == "decode":
        _prepare_decode(c, s, g)
    elif kind == "linear":
        s.w = _weight(c["scheme"], c["n"], c["k"], g, layout="gemm")
        s.x = _randn((c["rows"], c["k"]), g, c["x"])
        s.bias = _randn((c["n"],), g) if c["bias"] else None
        s.y = torch.empty((c["rows"], c["n"]), dtype=torch.float32, device="cuda")
        size = L.mllm_hip_linear_q_gemm_short_workspace_bytes if c["scheme"] in ("q4_0", "q8_0") else L.mllm_hip_linear_kq_gemm_short_workspace_bytes
        s.ws = _bytes(size(c["rows"], c["n"], c["k"]))
    elif kind == "w8a8":
        s.w = ql.w8a8_prepack(torch.randint(-127, 128, (c["n"], c["k"]), dtype=torch.int8, device="cuda", generator=g))
        s.scale = (torch.rand(c["n"], device="cuda", generator=g) + 0.01) * 0.01
        x = torch.randn((c["rows"], c["k"]), device="cuda", generator=g)
        x = torch.where(torch.rand(x.shape, device="cuda", generator=g) < 0.01, x * 20, x)  # outlier channels
        s.x = x.to(torch.bfloat16) if c["x"] == "bf16" else x
        s.bias = _randn((c["n"],), g) if c["bias"] else None
        s.y = torch.empty((c["rows"], c["n"]), dtype=torch.bfloat16, device="cuda")
        s.ws = _bytes(L.mllm_hip_w8a8_workspace_bytes(c["rows"], c["k"]))
    elif kind == "w4a16":
        groups = c["k"] // c["group"]
        qw = torch.randint(0, 256, (c["n"], c["k"] // 2), dtype=torch.uint8, device="cuda", generator=g)
        scale = (torch.randn((c["n"], groups), device="cuda", generator=g).abs() * 0.01).to(torch.float16)
        zeros = torch.randint(0, 256, (c["n"], (groups + 1) // 2), dtype=torch.uint8, device="cuda", generator=g)
        s.w = ql.w4a16_prepack(qw, scale, zeros, c["group"])
        s.x = _randn((c["rows"], c["k"]), g, "bf16")
        s.bias = _randn((c["n"],), g, "bf16") if c["bias"] else None
        s.y = torch.empty((c["rows"], c["n"]), dtype=torch.bfloat16, device="cuda")
    elif kind == "moe_prefill":
        t, h, inter, e, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top"]
        main, down = _schemes(c["scheme"])
        s.gate, s.up = _experts(main, e, inter, h, g, "gemm"), _experts(main, e, inter, h, g, "gemm")
        s.down = _experts(down, e, h, inter, g, "gemm")
        ids, weights = synth.make_moe_routing(np.random.default_rng(int(seed)), t, e, k)
        s.ids, s.weights = torch.from_numpy(ids).cuda(), torch.from_numpy(weights).cuda()
        s.x = _randn((t, h), g, "bf16")
        s.y = torch.empty((t, h), dtype=torch.float32, device="cuda")
        s.ws = _bytes((L.mllm_hip_moe_kq_workspace_bytes if c["scheme"] == "kq" else L.mllm_hip_moe_gemm_workspace_bytes)(t, h, inter, e, k))
    elif kind == "moe_decode":
        _prepare_moe_decode(c, s, g)
    elif kind == "attention":
        heads, head = c["kv_heads"], c["head"]
        s.q = _randn((heads, c["group"] * c["queries"], head), g, c["x"]) * (head ** -0.5)  # the query heads of a KV head are rows of one product
        s.k, s.v = _randn((heads, c["keys"], head), g, c["x"]), _randn((heads, c["keys"], head), g, c["x"])
        s.scores = torch.empty((heads, c["group"] * c["queries"], c["keys"]), dtype=s.q.dtype, device="cuda")
        s.o = torch.empty_like(s.q)
    else:
        s.logits = 3 * _randn((c["rows"], c["vocab"]), g)
    return s


# -------------------------------------------------------------------------------------------------------------------- run
def run(s):
    c = s.case
    kind = c["kind"]
    if kind in ("decode", "moe_decode"):
        s.x.copy_(s.token)
        s.graph.replay()
        return s.outputs
    if kind == "gemv":
        if s.ws is None:
            return ql.linear_q_gemv(s.w, s.x, s.bias, out=s.y)
        return ql.linear_q_gemv_multi([s.w], s.x, [s.bias], outs=[s.y], workspace=s.ws)[0]
    if kind == "linear":
        if c["scheme"] in ("q4_0", "q8_0"):
            return ql.linear_q_gemm(s.w, s.x, s.bias, workspace=s.ws, out=s.y, short=True)
        return ql.linear_kq_gemm(s.w, s.x, s.bias, out=s.y, workspace=s.ws, short=True)
    if kind == "w8a8":
        return ql.w8a8_linear_packed(s.x, s.w, c["n"], s.scale, s.bias, workspace=s.ws, out=s.y)
    if kind == "w4a16":
        return ql.w4a16_gemm_packed(s.x, s.w, c["n"], s.bias, c["group"], out=s.y)
    if kind == "moe_prefill":
        ffn = ql.moe_ffn_kq if c["scheme"] == "kq" else ql.moe_ffn_q_gemm
        return ffn(s.gate, s.up, s.down, s.x, s.ids, s.weights, workspace=s.ws, out=s.y)
    if kind == "attention":
        scores = ql.matmul(s.q, s.k, transpose_b=True, out=s.scores)
        p = ql.softmax(scores if c["x"] == "f32" else scores.float())
        return ql.matmul(p if c["x"] == "f32" else p.to(torch.bfloat16), s.v, out=s.o)
    probs = ql.softmax(s.logits)
    values, ids = ql.topk(probs, c["top"])
    return {"probs": probs, "values": values, "ids": ids}


# ------------------------------------------------------------------------------------------------------ work and tolerance
def _linear_work(scheme, rows, n, k, x_bytes, y_bytes):
    per, size = BLOCK[scheme]
    return n * k / per * size + rows * (k * x_bytes + n * y_bytes), 2.0 * rows * n * k


def work(case):
    c, kind = case, case["kind"]
    x_bytes = 2 if c.get("x") == "bf16" else 4
    if kind in ("gemv", "linear"):
        nbytes, flops = _linear_work(c["scheme"], c["rows"], c["n"], c["k"], x_bytes, 4)
    elif kind == "decode":
        main, down = _schemes(c["scheme"])
        h, nbytes, flops = c["hidden"], 0.0, 0.0
        for scheme, n, k in ((main, c["attn"], h), (main, 2 * c["kv"], h), (main, h, c["attn"]), (main, 2 * c["inter"], h), (down, h, c["inter"])):
            per, size = BLOCK[scheme]
            nbytes += c["layers"] * n * k / per * size
            flops += c["layers"] * 2.0 * c["rows"] * n * k
        nbytes += c["rows"] * 4 * (2 * h + c["layers"] * (c["attn"] + 2 * c["kv"])) + c["layers"] * 8 * h
    elif kind == "w8a8":
        nbytes = c["n"] * c["k"] + 4 * c["n"] + c["rows"] * (c["k"] * x_bytes + c["n"] * 2)
        flops = 2.0 * c["rows"] * c["n"] * c["k"]
    elif kind == "w4a16":
        groups = c["k"] // c["group"]
        nbytes = c["n"] * (c["k"] / 2 + groups * 2.5) + c["rows"] * 2 * (c["k"] + c["n"])
        flops = 2.0 * c["rows"] * c["n"] * c["k"]
    elif kind in ("moe_prefill", "moe_decode"):
        main, down = _schemes(c["scheme"])
        t, h, inter, e, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top"]
        layers = c.get("layers", 1)
        active = e * (1 - (1 - k / e) ** t)  # experts with a token, for even routing
        nbytes = active * h * inter * (2 * BLOCK[main][1] / BLOCK[main][0] + BLOCK[down][1] / BLOCK[down][0])
        nbytes = layers * (nbytes + t * k * 8) + t * h * (4 + (2 if kind == "moe_prefill" else 4))
        flops = layers * 6.0 * t * k * h * inter
        if kind == "moe_decode":
            nbytes, flops = nbytes + layers * (4 * e * h + 4 * h), flops + layers * 2.0 * t * e * h
    elif kind == "attention":
        rows = c["kv_heads"] * c["group"] * c["queries"]
        nbytes = x_bytes * c["head"] * 2 * (rows + c["kv_heads"] * c["keys"])
        flops = 4.0 * rows * c["keys"] * c["head"]
    else:
        nbytes, flops = c["rows"] * (c["vocab"] * 8 + c["top"] * 8), 5.0 * c["rows"] * c["vocab"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """about four times what two forms of the same path, or the path and its 64-bit restatement, were measured apart"""
    kind = case["kind"]
    if kind == "gemv":
        return {"rel": 1e-5}  # exact integer block sums, fp32 sums in another order: 1e-7
    if kind == "decode":
        return {"rel": 1e-3}  # sums in another order move activations over a rounding edge of the next quantization: 1.8e-4 after six layers
    if kind == "linear":
        return {"rel": 1.2e-3, "max": 8e-3}  # fp16 operands against the fp32 block arithmetic: 2e-4 to 3e-4, single values 1.7e-3
    if kind in ("w8a8", "w4a16"):
        return {"rel": 3e-4, "max": 1.6e-2}  # a sum next to a rounding edge of bf16 falls the other way: 1.5e-5 to 5e-5, single values one bf16 step
    if kind == "moe_prefill":
        return {"rel": 5e-4, "max": 3e-2}  # as decode, through one re-quantization: 8e-5, single values 6e-3
    if kind == "moe_decode":
        return {"rel": 5e-4, "max": 3e-2}
    if kind == "attention":
        return {"rel": 1e-5} if case["x"] == "f32" else {"rel": 3e-3, "max": 3e-2}  # fp32 sums: 6e-7; bf16 scores and probabilities
    return {"rel": 2e-6, "differ": 0.005}  # fp32 sums: 1.5e-7; equal probabilities
