"""The work this package is timed on: cases, their inputs, one pass of each through the public
entry points, and what each pass computes in 64 bits.

Kinds of case:

    linear   one 4-bit projection, `hip_native.matmul` (what a module of the native plan calls)
             or, with `path` "library", the forward of a plain `QuantizedLinear`; from one row
             (a decode step of one request) through 32 (a batched step) to a long prompt
    moe      one expert projection of a mixture-of-experts layer, `hip_native.gather_matmul`:
             gate/up (a token's row shared by its experts) or down (a row per pair)
    stream   a chain of independent one-row projections in one launch of the streaming engine
    attend   the decode step's attention of one layer over long contexts
    decode   a whole decode step: the staged program for one request, else a captured
             `decode_step`; every request at its own position
    prefill  a whole prompt through `decode.prefill`

Weights are zero-mean (each group's bias is about -7.5 of its scales) with a standard deviation of
about 1/sqrt(K), and in a model of L layers the projections that add to the residual stream (o and
down) are scaled by a further 1/sqrt(2 L), as decoders are initialised: a layer changes the stream by
a part of itself.
"""

import math
from types import SimpleNamespace

import torch

from ironmule_amd import _native, decode, hip_native
from ironmule_amd.quantized import QuantizedLinear

DEVICE = "cuda"
GROUP = 64

#: A Qwen3-4B-shaped decoder, the repository's own default configuration.
MODEL = dict(hidden=2560, layers=36, heads=32, kv_heads=8, intermediate=9728, vocab=151936)


def listed():
    return [
        # one token through the smallest projection of a decode step: latency
        dict(name="linear_1", kind="linear", path="native", rows=1, n=2560, k=2560),
        # a few requests, odd rows and an odd width
        dict(name="linear_7_ragged", kind="linear", path="native", rows=7, n=8200, k=1024),
        # a full batch of requests on the shared-weight sweep's own size
        dict(name="linear_32", kind="linear", path="native", rows=32, n=15360, k=3840),
        # a short chat prompt through a module that was not installed, long K
        dict(name="prompt_77_library", kind="linear", path="library", rows=77, n=2560, k=9728),
        # a long prompt through a gate or up projection
        dict(name="prompt_1024", kind="linear", path="native", rows=1024, n=9728, k=2560),
        # a small decode batch on an expert layer's gate or up projection
        dict(name="moe_decode_4x8", kind="moe", form="gate_up", tokens=4, top=8, experts=32, n=768, k=2560),
        # a prompt on the same layer's down projection
        dict(name="moe_prompt_128x8", kind="moe", form="down", tokens=128, top=8, experts=32, n=2560, k=768),
        # the bandwidth chain: every projection of the model once, one row
        dict(name="stream_36", kind="stream", layers=36, hidden=2560, heads=32, kv_heads=8, intermediate=9728),
        # four long conversations, one layer's attention
        dict(name="attend_4x8192", kind="attend", batch=4, context=8192, heads=32, kv_heads=8),
        # one conversation, a token at a time
        dict(name="decode_1", kind="decode", batch=1, context=512, **MODEL),
        # a serving batch
        dict(name="decode_32", kind="decode", batch=32, context=512, **MODEL),
        # a prompt before its decode steps
        dict(name="prefill_512", kind="prefill", tokens=512, **MODEL),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, layers):
    """A decoder of the ranges the repository's configurations and tests span."""
    return dict(hidden=rng.choice((1024, 2048, 2560)), layers=rng.randint(2, layers),
                heads=rng.choice((16, 24, 32)), kv_heads=8, intermediate=256 * rng.randint(8, 38),
                vocab=64 * _log(rng, 64, 2374))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "moe", "moe", "stream", "attend", "decode", "decode", "prefill"))
    if kind == "linear":
        rows = _log(rng, 1, 1024)
        return dict(kind=kind, path=rng.choice(("native", "native", "library")), rows=rows,
                    n=_log(rng, 256, 16384), k=GROUP * _log(rng, 4, 160))
    if kind == "moe":
        return dict(kind=kind, form=rng.choice(("gate_up", "down")), tokens=_log(rng, 1, 128),
                    top=rng.choice((2, 4, 8)), experts=rng.choice((8, 16, 32, 64)),
                    n=_log(rng, 256, 2048), k=GROUP * _log(rng, 8, 32))
    if kind == "stream":
        s = _shape(rng, 36)
        return dict(kind=kind, layers=s["layers"], hidden=s["hidden"], heads=s["heads"],
                    kv_heads=s["kv_heads"], intermediate=s["intermediate"])
    if kind == "attend":
        batch = _log(rng, 1, 32)
        return dict(kind=kind, batch=batch, context=_log(rng, 16, 32768 // batch),
                    heads=rng.choice((16, 32)), kv_heads=8)
    if kind == "decode":
        return dict(kind=kind, batch=rng.choice((1, 1, 2, 3, 4, 6, 8, 13, 16, 24, 32)),
                    context=_log(rng, 16, 512), **_shape(rng, 12))
    return dict(kind=kind, tokens=_log(rng, 4, 512), **_shape(rng, 12))


# ------------------------------------------------------------------ inputs

def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return gen


def _quant(gen, n, k, gain=1.0):
    """A zero-mean 4-bit weight of (n, k) with a standard deviation of about gain / sqrt(k)."""
    w = torch.randint(-2**31, 2**31, (n, k // 8), dtype=torch.int32, device=DEVICE, generator=gen)
    s = torch.empty((n, k // GROUP), device=DEVICE).uniform_(0.7, 1.3, generator=gen)
    s *= gain / (4.61 * math.sqrt(k))
    b = torch.empty((n, k // GROUP), device=DEVICE).uniform_(0.95, 1.05, generator=gen) * s * -7.5
    return w, s.to(torch.bfloat16), b.to(torch.bfloat16)


def _normal(gen, *shape):
    return torch.randn(shape, device=DEVICE, generator=gen).to(torch.bfloat16)


def _norm_weight(gen, n):
    return torch.empty(n, device=DEVICE).uniform_(0.9, 1.1, generator=gen).to(torch.bfloat16)


def _config(case):
    return decode.DecoderConfig(hidden=case["hidden"], layers=case["layers"], heads=case["heads"],
                                kv_heads=case["kv_heads"], intermediate=case["intermediate"],
                                vocab=case["vocab"])


def _weights(gen, config):
    weights, into_h = decode.DecoderWeights(config), 1.0 / math.sqrt(2 * config.layers)
    for _ in range(config.layers):
        layer = {name: _quant(gen, n, k, gain=into_h if name in ("o", "down") else 1.0)
                 for name, (n, k) in config.projections.items()}
        layer.update(input_norm=_norm_weight(gen, config.hidden), post_norm=_norm_weight(gen, config.hidden),
                     q_norm=_norm_weight(gen, config.head_dim), k_norm=_norm_weight(gen, config.head_dim))
        weights.layers.append(layer)
    weights.embed = _quant(gen, config.vocab, config.hidden, gain=0.5 * math.sqrt(config.hidden))
    weights.norm = _norm_weight(gen, config.hidden)
    return weights


def _positions(case):
    """Every request's position: spread over the upper half of the context."""
    c = case["context"]
    return [c - 1 - (29 * i) % (c // 2 + 1) for i in range(case["batch"])]


def _indices(gen, case):
    """Each token's `top` distinct experts."""
    order = torch.rand((case["tokens"], case["experts"]), device=DEVICE, generator=gen).argsort(dim=-1)
    return order[:, :case["top"]].to(torch.int32).contiguous()


def _state(config, batch, capacity):
    """A DecodeState whose layers' KV pools are slices of one tensor each."""
    state = decode.DecodeState(config, batch=batch, slots=batch, capacity=capacity, max_len=capacity, device=DEVICE)
    shape = (config.layers, batch, config.kv_heads, capacity, config.head_dim)
    keys = torch.zeros(shape, dtype=torch.bfloat16, device=DEVICE)
    values = torch.zeros(shape, dtype=torch.bfloat16, device=DEVICE)
    state.k_pool, state.v_pool = list(keys.unbind(0)), list(values.unbind(0))
    return state, keys, values


def _stages(gen, case):
    """(weights, x, output views) per stage of the chain, and the tensor the outputs lie in."""
    config = decode.DecoderConfig(hidden=case["hidden"], layers=case["layers"], heads=case["heads"],
                                  kv_heads=case["kv_heads"], intermediate=case["intermediate"])
    sizes = config.projections
    groups = (("q", "k", "v"), ("o",), ("gate", "up"), ("down",))
    rows = [_normal(gen, sizes[names[0]][1]) for names in groups]
    total = sum(n for n, _ in sizes.values())
    out = torch.empty(case["layers"] * total, dtype=torch.bfloat16, device=DEVICE)
    stages, at = [], 0
    for _ in range(case["layers"]):
        for names, x in zip(groups, rows):
            outs = []
            for name in names:
                outs.append(out[at:at + sizes[name][0]])
                at += sizes[name][0]
            stages.append(([_quant(gen, *sizes[name]) for name in names], x, outs))
    return stages, out


def prepare(case, seed):
    gen, kind = _generator(seed), case["kind"]
    if kind == "linear":
        quant, x = _quant(gen, case["n"], case["k"]), _normal(gen, case["rows"], case["k"])
        module = QuantizedLinear(*quant) if case["path"] == "library" else None
        return SimpleNamespace(kind=kind, quant=quant, x=x, module=module)
    if kind == "moe":
        w, s, b = _quant(gen, case["experts"] * case["n"], case["k"])
        quant = tuple(t.view(case["experts"], case["n"], -1) for t in (w, s, b))
        per = case["top"] if case["form"] == "down" else 1
        return SimpleNamespace(kind=kind, quant=quant, x=_normal(gen, case["tokens"], per, 1, case["k"]),
                               indices=_indices(gen, case))
    if kind == "stream":
        stages, out = _stages(gen, case)
        program = _native.stream_program([(weights, x, outs, False) for weights, x, outs in stages])
        return SimpleNamespace(kind=kind, stages=stages, out=out, program=program)
    if kind == "attend":
        b, hq, hkv, cap = case["batch"], case["heads"], case["kv_heads"], case["context"] + 8
        return SimpleNamespace(
            kind=kind, q=_normal(gen, b, hq * 128), k=_normal(gen, b, hkv * 128), v=_normal(gen, b, hkv * 128),
            q_norm=_norm_weight(gen, 128), k_norm=_norm_weight(gen, 128),
            k_pool=_normal(gen, b, hkv, cap, 128), v_pool=_normal(gen, b, hkv, cap, 128),
            positions=torch.tensor(_positions(case), dtype=torch.int32, device=DEVICE),
            slots=torch.arange(b, dtype=torch.int32, device=DEVICE),
            out=torch.empty((b, hq * 128), dtype=torch.bfloat16, device=DEVICE), max_len=cap,
            workspace=torch.empty(_native.attention_workspace(b, hq, cap), dtype=torch.float32, device=DEVICE),
            counters=torch.zeros(b * hkv, dtype=torch.int32, device=DEVICE))
    config = _config(case)
    weights = _weights(gen, config)
    if kind == "prefill":
        tokens = torch.randint(0, config.vocab, (case["tokens"],), device=DEVICE, generator=gen).tolist()
        state, keys, values = _state(config, 1, case["tokens"] + 8)
        return SimpleNamespace(kind=kind, weights=weights, state=state, tokens=tokens, keys=keys, values=values)
    state, keys, values = _state(config, case["batch"], case["context"] + 8)
    for pool in (*state.k_pool, *state.v_pool):
        pool.copy_(_normal(gen, *pool.shape))
    tokens = torch.randint(0, config.vocab, (case["batch"],), device=DEVICE, generator=gen).tolist()
    state.set_requests(tokens, list(range(case["batch"])), _positions(case))
    made = SimpleNamespace(kind=kind, weights=weights, state=state, tokens=tokens, keys=keys, values=values,
                           program=None, graph=None)
    if case["batch"] == 1:
        made.program = decode.PersistentDecode(weights, state, staged=True)
        return made
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    decode.decode_step(weights, state, stream=stream)  # workspaces, before the capture
    stream.synchronize()
    made.graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(made.graph, stream=stream):
        decode.decode_step(weights, state, stream=stream)
    torch.cuda.current_stream().wait_stream(stream)
    return made


# ------------------------------------------------------------------ one pass

def run(state):
    kind = state.kind
    if kind == "linear":
        if state.module is not None:
            return state.module(state.x)
        return hip_native.matmul(state.x, *state.quant)
    if kind == "moe":
        return hip_native.gather_matmul(state.x, *state.quant, state.indices)
    if kind == "stream":
        state.program.launch()
        return state.out
    if kind == "attend":
        out = _native.attention_fused(state.q, state.k, state.v, state.q_norm, state.k_norm, state.positions,
                                      state.slots, state.k_pool, state.v_pool, state.out, state.max_len,
                                      1e6, 1e-6, state.workspace, state.counters)
        return {"out": out, "keys": state.k_pool, "values": state.v_pool}
    if kind == "prefill":
        logits = decode.prefill(state.weights, state.state, state.tokens, 0)
        return {"logits": logits, "keys": state.keys, "values": state.values}
    if state.program is not None:
        logits = state.program.step()
    else:
        state.graph.replay()
        logits = state.state.logits
    return {"logits": logits, "h": state.state.h, "keys": state.keys, "values": state.values}


# ------------------------------------------------------------------ what a pass cannot do without

def _quant_bytes(n, k):
    return n * k // 2 + n * (k // GROUP) * 4


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": _quant_bytes(n, k) + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "moe":
        t, p, n, k = case["tokens"], case["tokens"] * case["top"], case["n"], case["k"]
        rows = p if case["form"] == "down" else t
        return {"bytes": min(case["experts"], p) * _quant_bytes(n, k) + 2 * rows * k + 2 * p * n + 4 * p,
                "flops": 2 * p * n * k}
    if kind == "attend":
        keys = sum(p + 1 for p in _positions(case))
        return {"bytes": keys * case["kv_heads"] * 128 * 2 * 2 + case["batch"] * (2 * case["heads"] + 4 * case["kv_heads"]) * 256,
                "flops": 4 * keys * case["heads"] * 128}
    config = decode.DecoderConfig(**{k: case[k] for k in ("hidden", "layers", "heads", "kv_heads", "intermediate")})
    layer = sum(_quant_bytes(n, k) for n, k in config.projections.values())
    macs = sum(n * k for n, k in config.projections.values())
    if kind == "stream":
        rows = 2 * sum(n for n, _ in config.projections.values())
        return {"bytes": case["layers"] * (layer + rows) + 4 * 2 * config.hidden, "flops": 2 * case["layers"] * macs}
    head, head_macs = _quant_bytes(case["vocab"], case["hidden"]), case["vocab"] * case["hidden"]
    kv_row = case["kv_heads"] * 128 * 2 * 2
    if kind == "decode":
        keys, b = sum(p + 1 for p in _positions(case)), case["batch"]
        return {"bytes": case["layers"] * (layer + keys * kv_row) + head + 4 * b * case["vocab"],
                "flops": 2 * b * (case["layers"] * macs + head_macs) + 4 * case["layers"] * keys * case["heads"] * 128}
    t = case["tokens"]
    return {"bytes": case["layers"] * (layer + t * kv_row) + head + 4 * case["vocab"],
            "flops": 2 * t * case["layers"] * macs + 2 * head_macs + 2 * case["layers"] * t * (t + 1) * case["heads"] * 128}


def tolerance(case):
    # One rounding to bf16 leaves about 1.7e-3; `attend` reads keys and queries that were
    # rounded once more.  Through a whole model every layer's activations are rounded, and
    # what one layer rounds otherwise travels on: 4e-3 against 64 bits.
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 1.5e-2, "max": 0.1}
    if case["kind"] == "attend":
        return {"rel": 8e-3, "max": 4e-2}
    return {"rel": 6e-3, "max": 2e-2}


# ------------------------------------------------------------------ the same in 64 bits

def _dense(quant):
    w, s, b = quant
    shifts = 4 * torch.arange(8, dtype=torch.int32, device=w.device)
    q = ((w[..., None] >> shifts) & 15).to(torch.float64).view(*s.shape, GROUP)
    return (q * s.double()[..., None] + b.double()[..., None]).view(*w.shape[:-1], -1)


def _rms(x, weight, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + eps) * weight.double()


def _rope(x, positions, theta=1e6):
    """(rows, heads, 128): the pair (i, i + 64) turned by position * theta^(-i/64)."""
    half = x.shape[-1] // 2
    angle = positions.double()[:, None] * theta ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * cos - hi * sin, lo * sin + hi * cos], dim=-1)


def _softmax_v(q, keys, values, seen):
    """q (..., G, 128), keys and values (..., L, 128), seen broadcast to (..., G, L)."""
    scores = torch.matmul(q, keys.transpose(-1, -2).contiguous()) / math.sqrt(128.0)
    return torch.matmul(scores.masked_fill(~seen, float("-inf")).softmax(dim=-1), values)


def _decode_attention(q, k, v, q_norm, k_norm, positions, k_pool, v_pool):
    b, hkv, length = positions.numel(), k_pool.shape[1], k_pool.shape[2]
    q = _rope(_rms(q.double().view(b, -1, 128), q_norm), positions)
    keys, values, at = k_pool.double(), v_pool.double(), torch.arange(b, device=q.device)
    keys[at, :, positions] = _rope(_rms(k.double().view(b, hkv, 128), k_norm), positions)
    values[at, :, positions] = v.double().view(b, hkv, 128)
    seen = torch.arange(length, device=q.device) <= positions[:, None]
    return _softmax_v(q.view(b, hkv, -1, 128), keys, values, seen[:, None, None]).reshape(b, -1)


def _prompt_attention(q, k, v, layer, positions, heads, kv_heads):
    t = positions.numel()
    q = _rope(_rms(q.view(t, heads, 128), layer["q_norm"]), positions)
    k = _rope(_rms(k.view(t, kv_heads, 128), layer["k_norm"]), positions).transpose(0, 1).contiguous()
    v = v.view(t, kv_heads, 128).transpose(0, 1).contiguous()
    q = q.view(t, kv_heads, -1, 128).permute(1, 2, 0, 3).contiguous()
    seen = positions <= positions[:, None]
    out = _softmax_v(q, k[:, None], v[:, None], seen)
    return out.permute(2, 0, 1, 3).reshape(t, -1), k, v


def _model(weights, tokens, attention):
    """The residual stream after the last layer and its head's logits; attention(i, layer, q, k, v)."""
    def project(x, quant):
        return x @ _dense(quant).T

    ids = torch.tensor(tokens, device=DEVICE)
    h = _dense(tuple(t[ids] for t in weights.embed))
    for i, layer in enumerate(weights.layers):
        x = _rms(h, layer["input_norm"])
        h = h + project(attention(i, layer, *(project(x, layer[n]) for n in ("q", "k", "v"))), layer["o"])
        x = _rms(h, layer["post_norm"])
        h = h + project(torch.nn.functional.silu(project(x, layer["gate"])) * project(x, layer["up"]), layer["down"])
    return h, lambda rows: project(_rms(rows, weights.norm), weights.embed)


def exact(case, seed):
    state, kind = prepare(case, seed), case["kind"]
    if kind == "linear":
        return state.x.double() @ _dense(state.quant).T
    if kind == "moe":
        dense = _dense(state.quant)
        x = state.x.double().expand(case["tokens"], case["top"], 1, case["k"]).reshape(-1, case["k"])
        expert = state.indices.reshape(-1)
        out = torch.empty((expert.numel(), case["n"]), dtype=torch.float64, device=DEVICE)
        for e in range(case["experts"]):
            out[expert == e] = x[expert == e] @ dense[e].T
        return out.view(case["tokens"], case["top"], 1, case["n"])
    if kind == "stream":
        return torch.cat([_dense(q) @ x.double() for weights, x, _ in state.stages for q in weights])
    if kind == "attend":
        out = _decode_attention(state.q, state.k, state.v, state.q_norm, state.k_norm, state.positions,
                                state.k_pool, state.v_pool)
        return {"out": out, "keys": None, "values": None}
    weights = state.weights
    if kind == "decode":
        positions = state.state.positions
        h, head = _model(weights, state.tokens, lambda i, layer, q, k, v: _decode_attention(
            q, k, v, layer["q_norm"], layer["k_norm"], positions, state.keys[i], state.values[i]))
        return {"logits": head(h), "h": h, "keys": None, "values": None}
    positions = torch.arange(case["tokens"], device=DEVICE)
    keys, values = torch.zeros_like(state.keys, dtype=torch.float64), torch.zeros_like(state.values, dtype=torch.float64)

    def attention(i, layer, q, k, v):
        out, keys[i, 0, :, :case["tokens"]], values[i, 0, :, :case["tokens"]] = _prompt_attention(
            q, k, v, layer, positions, case["heads"], case["kv_heads"])
        return out

    h, head = _model(weights, state.tokens, attention)
    return {"logits": head(h[-1:])[0], "keys": keys, "values": values}
