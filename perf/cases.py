"""Workloads of the packed runtime, as a program that serves a packed model calls it.

A case is a dict of plain values. ``prepare`` builds what such a program holds
before the call (packed layers, a decoder, inputs), ``run`` makes one pass
through the public entry points, ``exact`` computes the same outputs in 64 bits
with plain torch. Five kinds:

* ``linear``: packed linears on ``HipPackedBackend``, one alone (``linear``) or
  several sharing one launch per phase (``linear_batch``): one decode token up
  to a 2048-token prompt;
* ``attention``: the prompt rows' q/k norm, RoPE, cache append and causal
  attention;
* ``decode_attention``: one token's attention over a filled cache;
* ``prompt``: a decoder's whole prompt pass, ids to logits;
* ``step``: a decoder's one-token step (the captured graph), id to logits.
"""

from __future__ import annotations

import math

import torch

from nanoquant_amd.runtime import (
    PACKED_LAYOUT_VERSION,
    DecoderLayerWeights,
    DecoderShellConfig,
    DecoderShellWeights,
    HipPackedBackend,
    PackedDecoder,
    PackedLayerState,
    QuantizedLinearSpec,
)
from nanoquant_amd.runtime import shell_ops as ops
from nanoquant_amd.runtime.row_sidecar import OutputRowSidecar, RowSidecarLayerState

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EPS = 1e-6
ROPE_THETA = 1_000_000.0

# in:out:rank of the projections that the benchmark and the tests use.
QKV_QWEN = "4096:4096:2048,4096:1024:819,4096:1024:819"
GATE_UP_QWEN = "4096:12288:3072,4096:12288:3072"
DOWN_QWEN = "12288:4096:3072"
QKV_LLAMA = "4096:4096:1638,4096:1024:655,4096:1024:655"
O_LLAMA = "4096:4096:1638"
GATE_UP_LLAMA = "4096:14336:2549,4096:14336:2549"
DOWN_LLAMA = "14336:4096:2549"
GATE_GEMMA_1B = "1152:6912:768"
DOWN_GEMMA_4B = "10240:2560:1536"
QWEN_LAYER = (4096, 12288, 32, 8, 128)  # hidden, intermediate, q heads, kv heads, head_dim


def _linear(name, linears, tokens, *, x="bf16", operands="fp16", sidecar="none", bias=False):
    return {"name": name, "kind": "linear", "linears": linears, "tokens": tokens, "x": x, "operands": operands,
            "sidecar": sidecar, "bias": bias}


def _attention(name, tokens, start, rows, *, q_heads=32, kv_heads=8, head_dim=128, cache="bf16", out="bf16"):
    return {"name": name, "kind": "attention", "tokens": tokens, "start": start, "rows": rows, "q_heads": q_heads,
            "kv_heads": kv_heads, "head_dim": head_dim, "cache": cache, "out": out}


def _decode_attention(name, position, rows, *, q_heads=32, kv_heads=8, head_dim=128, cache="bf16", out="bf16"):
    return {"name": name, "kind": "decode_attention", "position": position, "rows": rows, "q_heads": q_heads,
            "kv_heads": kv_heads, "head_dim": head_dim, "cache": cache, "out": out}


def _decoder(name, kind, layers, tokens, *, rows=640, vocab=151936):
    return {"name": name, "kind": kind, "layers": layers, "tokens": tokens, "rows": rows, "vocab": vocab}


def listed():
    return [
        # The smallest call: one decode token through one small projection, launched eagerly.
        _linear("gate_1152_m1", GATE_GEMMA_1B, 1),
        # One decode token through an attention block's three projections in one launch pair.
        _linear("qkv_m1", QKV_QWEN, 1),
        # A few sequences decoded together; the layer keeps its salient input columns in int8.
        _linear("down_salient_m8", DOWN_GEMMA_4B, 8, sidecar="columns"),
        # The largest token count of the decode kernels: a small server batch through an MLP's wide half.
        _linear("gate_up_m16", GATE_UP_QWEN, 16),
        # A short prompt (a chat turn), odd length, one projection on its own.
        _linear("o_m61", O_LLAMA, 61),
        # An ordinary prompt through the widest pair of a layer.
        _linear("gate_up_m512", GATE_UP_LLAMA, 512),
        # A long prompt through the projection with the longest rows.
        _linear("down_m2048", DOWN_LLAMA, 2048),
        # A prompt in fp32: operands carried as a value and its remainder.
        _linear("qkv_split_m300", QKV_QWEN, 300, x="f32", operands="split"),
        # The second chunk of a long prompt: attention against the chunk and what the cache already holds.
        _attention("attention_1531", 1531, 517, 2048),
        # One token far into a long conversation.
        _decode_attention("decode_attention_4k", 3900, 4096),
        # A whole prompt through a decoder: the time to the first token.
        _decoder("prompt_512", "prompt", 12, 512),
        # A whole decode step: the time per token.
        _decoder("step", "step", 12, 600),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    pick = rng.random()
    if pick < 0.64:
        x = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        decode = pick < 0.32
        tokens = rng.randint(1, 16) if decode else _log_int(rng, 17, 2048)
        if rng.random() < 0.3:
            # A projection of no particular model: any widths, ragged ones among them.
            i, o = _log_int(rng, 200, 9000), _log_int(rng, 200, 9000)
            linears = f"{i}:{o}:{max(8, round(rng.uniform(0.6, 1.0) * i * o / (i + o)))}"
        else:
            linears = rng.choice([QKV_QWEN, GATE_UP_QWEN, DOWN_QWEN, QKV_LLAMA, O_LLAMA, GATE_UP_LLAMA, DOWN_LLAMA,
                                  GATE_GEMMA_1B, DOWN_GEMMA_4B])
        sidecar = rng.choice(["none", "none", "none", "columns", "rows"])
        case = _linear("", linears, tokens, x=x, operands="split" if x == "f32" and rng.random() < 0.7 else "fp16",
                       sidecar=sidecar, bias=rng.random() < 0.2)
    elif pick < 0.84:
        geometry = rng.choice([(32, 8, 128), (32, 8, 128), (16, 4, 128), (16, 8, 128), (8, 4, 256), (4, 4, 64)])
        tokens = _log_int(rng, 17, 1531)
        start = rng.choice([0, 0, rng.randint(1, 1000)])
        rows = start + tokens + rng.randint(0, 200)
        case = _attention("", tokens, start, rows, q_heads=geometry[0], kv_heads=geometry[1], head_dim=geometry[2],
                          cache=rng.choice(["bf16", "bf16", "bf16", "f16", "f32"]), out=rng.choice(["bf16", "f32"]))
    elif pick < 0.92:
        geometry = rng.choice([(32, 8, 128), (16, 8, 128), (64, 8, 128), (8, 8, 64)])
        position = _log_int(rng, 40, 16000)
        case = _decode_attention("", position, position + rng.randint(1, 700), q_heads=geometry[0],
                                 kv_heads=geometry[1], head_dim=geometry[2], cache=rng.choice(["bf16", "f16"]),
                                 out=rng.choice(["bf16", "f32"]))
    else:
        kind = rng.choice(["prompt", "step"])
        tokens = _log_int(rng, 17, 512) if kind == "prompt" else _log_int(rng, 20, 900)
        case = _decoder("", kind, rng.randint(2, 10), tokens, rows=tokens + rng.randint(8, 200),
                        vocab=rng.choice([32000, 128256, 151936]))
    del case["name"]
    return case


# -- inputs --------------------------------------------------------------------


def _shapes(case):
    return [tuple(int(v) for v in part.split(":")) for part in case["linears"].split(",")]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _words(g, rows, cols):
    words = torch.randint(-(2**31), 2**31, (rows, -(-cols // 32)), generator=g, dtype=torch.int64, device="cuda")
    words = words.to(torch.int32)
    if cols % 32:
        words[:, -1] &= (1 << (cols % 32)) - 1
    return words


def _layer_tensors(g, i, o, r, sidecar="none", bias=False):
    """One packed layer's tensors: random signs, log-normal scales sized so that
    unit activations give unit outputs, and the optional sidecars."""

    t = {
        "v": _words(g, r, i),
        "u": _words(g, o, r),
        "s_in": torch.exp(0.25 * _randn(g, i)).half(),
        "s_mid": (torch.exp(0.25 * _randn(g, r)) * i**-0.5).half(),
        "s_out": (torch.exp(0.25 * _randn(g, o)) * r**-0.5).half(),
    }
    if bias:
        t["bias"] = (0.1 * _randn(g, o)).half()
    if sidecar == "columns":
        columns = torch.randperm(i, generator=g, device="cuda")[:26].sort().values
        t["s_in"][columns] = 0
        t["columns"] = columns.to(torch.int32)
        t["column_values"] = torch.randint(-127, 128, (o, 26), generator=g, device="cuda").to(torch.int8)
        t["column_scales"] = (torch.exp(0.25 * _randn(g, 26)) / 127).half()
    elif sidecar == "rows":
        t["rows"] = torch.randperm(o, generator=g, device="cuda")[:26].sort().values.to(torch.int32)
        t["row_values"] = torch.randint(-127, 128, (26, i), generator=g, device="cuda").to(torch.int8)
        t["row_scales"] = (torch.exp(0.25 * _randn(g, 26)) * i**-0.5 / 127).half()
    return t


def _state(name, i, o, r, t):
    columns = "columns" in t
    spec = QuantizedLinearSpec(name, "nanoquant-v1", i, o, r, "float32", "float16",
                               outlier_count=26 if columns else 0, outlier_value_dtype="int8" if columns else None,
                               has_outlier_scales=columns, has_bias="bias" in t)
    state = PackedLayerState(spec, PACKED_LAYOUT_VERSION, t["u"], t["v"], t["s_in"], t["s_mid"], t["s_out"],
                             t.get("bias"), t.get("columns"), t.get("column_values"), t.get("column_scales"))
    if "rows" in t:
        return RowSidecarLayerState(state, OutputRowSidecar(t["rows"], t["row_values"], t["row_scales"]))
    return state


def _linear_inputs(case, seed):
    g = _generator(seed)
    shapes = _shapes(case)
    tensors = [_layer_tensors(g, i, o, r, case["sidecar"], case["bias"]) for i, o, r in shapes]
    # Hidden states: normal, some channels several times as large as others.
    x = _randn(g, case["tokens"], shapes[0][0]) * torch.exp(0.5 * _randn(g, shapes[0][0]))
    return shapes, tensors, x.to(DTYPES[case["x"]])


def _rope(rows, head_dim, dtype=torch.float32):
    inv = 1.0 / (ROPE_THETA ** (torch.arange(0, head_dim, 2, dtype=torch.float) / head_dim))
    angles = torch.arange(rows, dtype=torch.float)[:, None] * inv[None, :]
    return angles.cos().to("cuda", dtype), angles.sin().to("cuda", dtype)


def _attention_inputs(case, seed):
    g = _generator(seed)
    qh, kvh, d, rows = case["q_heads"], case["kv_heads"], case["head_dim"], case["rows"]
    tokens = case.get("tokens", 1)
    dtype = DTYPES[case["cache"]]
    t = {
        "q": _randn(g, tokens, qh * d), "k": _randn(g, tokens, kvh * d), "v": _randn(g, tokens, kvh * d),
        "q_norm": 1.0 + 0.2 * _randn(g, d), "k_norm": 1.0 + 0.2 * _randn(g, d),
        "k_cache": _randn(g, kvh, rows, d).to(dtype), "v_cache": _randn(g, kvh, rows, d).to(dtype),
    }
    # Queries and keys share a direction, so that the softmax has heavy and light rows.
    t["q"].view(tokens, qh, d).add_(_randn(g, d))
    t["cos"], t["sin"] = _rope(rows, d)
    t["position"] = torch.tensor([case.get("start", case.get("position"))], dtype=torch.int32, device="cuda")
    return t


def _decoder_inputs(case, seed):
    g = _generator(seed)
    hidden, inter, qh, kvh, d = QWEN_LAYER
    config = DecoderShellConfig(case["layers"], hidden, inter, qh, kvh, d, case["vocab"], EPS, ROPE_THETA)
    dims = config.linear_dims()

    def norm(n):
        return 1.0 + 0.1 * _randn(g, n)

    layers = []
    for _ in range(case["layers"]):
        linears = {}
        for role, (i, o) in dims.items():
            r = round(i * o / (i + o))
            linears[role] = (i, o, r, _layer_tensors(g, i, o, r))
        layers.append((norm(hidden), norm(hidden), norm(d), norm(d), linears))
    dense = {name: (0.02 * _randn(g, case["vocab"], hidden)).to(torch.bfloat16) for name in ("embed", "lm_head")}
    dense["final_norm"] = norm(hidden)
    ids = torch.randint(0, case["vocab"], (case["tokens"],), generator=g, device="cuda")
    cache = None
    if case["kind"] == "step":
        shape = (case["layers"], kvh, case["rows"], d)
        cache = [_randn(g, *shape).to(torch.bfloat16) for _ in range(2)]
    return config, layers, dense, ids, cache


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        shapes, tensors, x = _linear_inputs(case, seed)
        backend = HipPackedBackend(prefill_operands=case["operands"])
        layers = [backend.prepare(_state(f"blocks.0.linear_{n}", *shape, t), "cuda")
                  for n, (shape, t) in enumerate(zip(shapes, tensors))]
        return {"kind": kind, "backend": backend, "layers": layers, "x": x}
    if kind in ("attention", "decode_attention"):
        t = _attention_inputs(case, seed)
        shared = {name: t[name] for name in ("cos", "sin", "position", "k_cache", "v_cache", "q_norm", "k_norm")}
        shared.update(q_heads=case["q_heads"], kv_heads=case["kv_heads"], head_dim=case["head_dim"], eps=EPS)
        if kind == "attention":
            need = ops.attention_workspace_bytes(case["tokens"], case["q_heads"], case["head_dim"], case["rows"])
        else:
            need = ops.decode_attention_workspace_bytes(case["q_heads"], case["kv_heads"], case["head_dim"],
                                                        DTYPES[case["cache"]], case["rows"])
        return {"kind": kind, "qkv": (t["q"], t["k"], t["v"]), "shared": shared, "out": DTYPES[case["out"]],
                "scaling": case["head_dim"] ** -0.5,
                "workspace": torch.empty(need, dtype=torch.uint8, device="cuda")}
    config, layers, dense, ids, cache = _decoder_inputs(case, seed)
    weights = DecoderShellWeights(dense["embed"], dense["lm_head"], dense["final_norm"], [
        DecoderLayerWeights(*norms, {role: _state(f"blocks.{n}.{role}", i, o, r, t)
                                     for role, (i, o, r, t) in linears.items()})
        for n, (*norms, linears) in enumerate(layers)])
    decoder = PackedDecoder(config, weights, max_positions=case["rows"])
    state = {"kind": kind, "decoder": decoder, "ids": ids}
    if kind == "step":
        p = case["tokens"]
        decoder.k_cache.copy_(cache[0])
        decoder.v_cache.copy_(cache[1])
        state["step"] = {
            "input_ids": ids[-1:].view(1, 1), "attention_mask": torch.ones(1, p + 1, dtype=torch.bool, device="cuda"),
            "position_ids": torch.tensor([[p]], device="cuda"), "cache_position": torch.tensor([p], device="cuda"),
            "cache": decoder, "max_cache_length": case["rows"], "workload": "decode", "deterministic": True,
        }
    return state


def run(state):
    kind = state["kind"]
    if kind == "linear":
        if len(state["layers"]) == 1:
            return state["backend"].linear(state["x"], state["layers"][0])
        return state["backend"].linear_batch([state["x"]] * len(state["layers"]), state["layers"])
    if kind == "attention":
        shared = state["shared"]
        rotated = ops.launch_qk_norm_rope_cache(*state["qkv"], **shared)
        out = ops.launch_attention(rotated, shared["k_cache"], shared["v_cache"], position=shared["position"],
                                   scaling=state["scaling"], out_dtype=state["out"], workspace=state["workspace"])
        return out, rotated, shared["k_cache"], shared["v_cache"]
    if kind == "decode_attention":
        shared = state["shared"]
        out = ops.launch_decode_attention(*state["qkv"], **shared, scaling=state["scaling"], out_dtype=state["out"],
                                          workspace=state["workspace"])
        return out, shared["k_cache"], shared["v_cache"]
    decoder = state["decoder"]
    if kind == "prompt":
        logits = decoder.prefill(state["ids"])
    else:
        logits = decoder.forward_step(**state["step"]).logits
    return logits, decoder.k_cache, decoder.v_cache


# -- what a pass cannot do without ----------------------------------------------


def _linear_work(shapes, tokens, x_bytes, y_bytes):
    words = sum(4 * r * -(-i // 32) + 4 * o * -(-r // 32) + 2 * (i + r + o) for i, o, r in shapes)
    moved = words + x_bytes * tokens * shapes[0][0] + y_bytes * tokens * sum(o for _, o, _ in shapes)
    return moved, sum(2 * tokens * r * (i + o) for i, o, r in shapes)


def _attention_work(tokens, start, q_heads, kv_heads, head_dim, cache_bytes):
    """Cache rows read, new rows written, and the products over the causal pairs."""

    pairs = sum(start + t + 1 for t in range(tokens))
    moved = 2 * kv_heads * head_dim * cache_bytes * (start + tokens)
    return moved, 4 * pairs * q_heads * head_dim


def work(case):
    kind = case["kind"]
    size = {"bf16": 2, "f16": 2, "f32": 4}
    if kind == "linear":
        shapes = _shapes(case)
        moved, flops = _linear_work(shapes, case["tokens"], size[case["x"]], 4)
        if case["sidecar"] == "columns":
            moved += sum(26 * o for _, o, _ in shapes)
            flops += sum(2 * 26 * o * case["tokens"] for _, o, _ in shapes)
        elif case["sidecar"] == "rows":
            moved += sum(26 * i for i, _, _ in shapes)
            flops += sum(2 * 26 * i * case["tokens"] for i, _, _ in shapes)
        return {"bytes": moved, "flops": flops}
    if kind in ("attention", "decode_attention"):
        tokens = case.get("tokens", 1)
        qh, kvh, d = case["q_heads"], case["kv_heads"], case["head_dim"]
        moved, flops = _attention_work(tokens, case.get("start", case.get("position")), qh, kvh, d, size[case["cache"]])
        moved += tokens * d * (4 * (qh + 2 * kvh) + size[case["out"]] * qh)
        if kind == "attention":
            moved += 4 * tokens * d * qh  # the rotated queries
        return {"bytes": moved, "flops": flops}
    hidden, inter, qh, kvh, d = QWEN_LAYER
    tokens, start = (case["tokens"], 0) if kind == "prompt" else (1, case["tokens"])
    dims = [(hidden, qh * d), (hidden, kvh * d), (hidden, kvh * d), (qh * d, hidden), (hidden, inter), (hidden, inter),
            (inter, hidden)]
    shapes = [(i, o, round(i * o / (i + o))) for i, o in dims]
    moved, flops = _linear_work(shapes, tokens, 0, 0)
    more = _attention_work(tokens, start, qh, kvh, d, 2)
    moved, flops = case["layers"] * (moved + more[0]), case["layers"] * (flops + more[1])
    head = case["vocab"] * hidden
    return {"bytes": moved + 2 * head + 2 * tokens * hidden + 4 * case["vocab"], "flops": flops + 2 * head}


# -- tolerances and 64-bit results ------------------------------------------------


def tolerance(case):
    """About four times the distance to the 64-bit result that was measured over the ranges."""

    kind = case["kind"]
    if kind == "linear":
        if case["tokens"] <= 16:
            return {"rel": 1e-4}  # activations as 24-bit integers, fp32 sums
        return {"rel": 3e-6 if case["operands"] == "split" else 1.2e-3}  # 22 or 11 bits an operand
    if kind in ("attention", "decode_attention"):
        # The result's own rounding; for fp32, cache rows that round the other way.
        return {"rel": 7e-3 if case["out"] == "bf16" else 1e-4}
    return {"rel": 5e-2 if kind == "prompt" else 2.5e-2}  # bf16 activations and cache through every layer


def _signs(words, cols):
    bits = (words[:, :, None] >> torch.arange(32, device=words.device, dtype=torch.int32)) & 1
    return 1.0 - 2.0 * bits.reshape(words.shape[0], -1)[:, :cols].double()


def _exact_linear(x, i, r, t):
    x = x.double()
    y = (x * t["s_in"].double()) @ _signs(t["v"], i).t()
    y = (y * t["s_mid"].double()) @ _signs(t["u"], r).t() * t["s_out"].double()
    if "columns" in t:
        y += x[:, t["columns"].long()] @ (t["column_values"].double() * t["column_scales"].double()).t()
    if "bias" in t:
        y += t["bias"].double()
    if "rows" in t:
        y[:, t["rows"].long()] += x @ t["row_values"].double().t() * t["row_scales"].double()
    return y


def _exact_norm(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _exact_rotate(x, weight, cos, sin):
    """q/k RMSNorm and rotate-half RoPE of [tokens, heads, head_dim]."""

    a, b = _exact_norm(x, weight).chunk(2, dim=-1)
    cos, sin = cos[:, None, :], sin[:, None, :]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _exact_attention(q, k_cache, v_cache, start):
    """Causal grouped-query attention of [tokens, q_heads, d] over [kv_heads, rows, d]."""

    tokens, qh, d = q.shape
    group = qh // k_cache.shape[0]
    end = start + tokens
    future = torch.arange(end, device=q.device)[None, :] > (start + torch.arange(tokens, device=q.device))[:, None]
    out = torch.empty_like(q)
    for h in range(qh):
        scores = q[:, h] @ k_cache[h // group, :end].t() * d**-0.5
        scores.masked_fill_(future, -math.inf)
        out[:, h] = torch.softmax(scores, dim=-1) @ v_cache[h // group, :end]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        shapes, tensors, x = _linear_inputs(case, seed)
        outs = [_exact_linear(x, i, r, t) for (i, _, r), t in zip(shapes, tensors)]
        return outs[0] if len(outs) == 1 else outs
    if kind in ("attention", "decode_attention"):
        t = _attention_inputs(case, seed)
        tokens, start = case.get("tokens", 1), case.get("start", case.get("position"))
        qh, kvh, d = case["q_heads"], case["kv_heads"], case["head_dim"]
        at = slice(start, start + tokens)
        cos, sin = t["cos"][at].double(), t["sin"][at].double()
        q = _exact_rotate(t["q"].double().view(tokens, qh, d), t["q_norm"], cos, sin)
        k = _exact_rotate(t["k"].double().view(tokens, kvh, d), t["k_norm"], cos, sin)
        kc, vc = t["k_cache"].clone(), t["v_cache"].clone()
        # The caller's cache type holds the new rows, as it holds the old ones.
        kc[:, at] = k.transpose(0, 1).to(kc.dtype)
        vc[:, at] = t["v"].view(tokens, kvh, d).transpose(0, 1).to(vc.dtype)
        out = _exact_attention(q, kc.double(), vc.double(), start)
        if kind == "attention":
            return out.reshape(tokens, qh * d), q, kc.double(), vc.double()
        return out.reshape(qh * d), kc.double(), vc.double()
    _, layers, dense, ids, cache = _decoder_inputs(case, seed)
    hidden, inter, qh, kvh, d = QWEN_LAYER
    start = 0 if kind == "prompt" else case["tokens"]
    ids = ids if kind == "prompt" else ids[-1:]
    tokens = ids.numel()
    shape = (case["layers"], kvh, case["rows"], d)
    kc, vc = [c.double() for c in cache] if cache else [torch.zeros(shape, dtype=torch.float64, device="cuda")
                                                        for _ in range(2)]
    at = slice(start, start + tokens)
    cos, sin = (table[at] for table in _rope(case["rows"], d, torch.float64))
    h = dense["embed"][ids].double()
    for n, (in_norm, post_norm, q_norm, k_norm, linears) in enumerate(layers):
        def linear(role, value):
            i, _, r, t = linears[role]
            return _exact_linear(value, i, r, t)

        xn = _exact_norm(h, in_norm)
        q = _exact_rotate(linear("q_proj", xn).view(tokens, qh, d), q_norm, cos, sin)
        k = _exact_rotate(linear("k_proj", xn).view(tokens, kvh, d), k_norm, cos, sin)
        kc[n, :, at] = k.transpose(0, 1)
        vc[n, :, at] = linear("v_proj", xn).view(tokens, kvh, d).transpose(0, 1)
        h = h + linear("o_proj", _exact_attention(q, kc[n], vc[n], start).reshape(tokens, qh * d))
        xn = _exact_norm(h, post_norm)
        gate = linear("gate_proj", xn)
        h = h + linear("down_proj", gate * torch.sigmoid(gate) * linear("up_proj", xn))
    logits = _exact_norm(h[-1], dense["final_norm"]) @ dense["lm_head"].double().t()
    return (logits if kind == "prompt" else logits.view(1, 1, -1)), kc, vc
