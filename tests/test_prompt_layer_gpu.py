"""GPU parity of the prompt kernels against 64-bit references: one layer at a time with its
rounding points (imq_prompt_layer, imq_prompt_finish), and products, expert batches and grouped
products at sizes whose plan takes each tile height and K-ranges.  Every case names the plan it is
there for and fails if the plan no longer selects it.

Bars of a layer, as the 2-norm of a row's (for keys and values a head's) difference over the row's.
Both sides round to bf16 at the same places and differ where fp32 sums push a value over a rounding
edge: one ulp of that value, and at most as much in a whole row as rounding it once, 2^-8.  So 2^-8
for keys and values and for what the MLP alone adds to the stream (one row in many there has a
flipped value before its last rounding: 2^-11 on average); 2^-7 for what attention alone adds, whose
output's rounding passes o's; and 2^-6 for a whole layer, where these two pass two more in the MLP.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.gpu_util import announce, bf16_bits, to_device

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

SPLITS = 8  # the K-ranges a product may take; q/k/v and gate/up of a layer take one


@pytest.fixture(scope="module")
def env():
    import torch

    from ironmule_amd import _native
    from oracle import oracle as orc
    code, arch, _ = _native.device_check()
    assert code == 0, f"device {arch} is not supported"
    orc.lib()
    return torch, _native, orc


def _plan(n_, sizes, m, k, most=SPLITS):
    """(rows of a tile, K-ranges) of a product."""
    rows, splits = ctypes.c_int32(), ctypes.c_int32()
    cus = n_.device_check()[2]
    assert n_.lib().imq_prompt_plan((ctypes.c_int32 * len(sizes))(*sizes), len(sizes), m, k, most, cus,
                                    ctypes.byref(rows), ctypes.byref(splits)) == 0
    return rows.value, splits.value


def _weight(torch, gen, n, k, gain=1.0):
    """A zero-mean 4-bit weight with a standard deviation of about gain / sqrt(k)."""
    w = torch.randint(-2**31, 2**31, (n, k // 8), dtype=torch.int32, device="cuda", generator=gen)
    s = torch.empty((n, k // 64), device="cuda").uniform_(0.7, 1.3, generator=gen) * (gain / (4.61 * k ** 0.5))
    b = torch.empty((n, k // 64), device="cuda").uniform_(0.95, 1.05, generator=gen) * s * -7.5
    return w, s.to(torch.bfloat16), b.to(torch.bfloat16)


def _dense(torch, n_, quant):
    return n_.dequant(*quant).double()


# ------------------------------------------------------------------ a layer in 64 bits

class _Config:
    head_dim, eps, theta = 128, 1e-6, 1e6

    def __init__(self, heads, kv_heads, hidden, intermediate):
        self.heads, self.kv_heads, self.hidden, self.intermediate = heads, kv_heads, hidden, intermediate
        q, kv = heads * 128, kv_heads * 128
        self.projections = {"q": (q, hidden), "k": (kv, hidden), "v": (kv, hidden), "o": (hidden, q),
                            "gate": (intermediate, hidden), "up": (intermediate, hidden), "down": (hidden, intermediate)}


def _layer(torch, gen, config, sharp=1.0):
    layer = {name: _weight(torch, gen, n, k) for name, (n, k) in config.projections.items()}
    for name, size in (("input_norm", config.hidden), ("post_norm", config.hidden), ("q_norm", 128), ("k_norm", 128)):
        layer[name] = torch.empty(size, device="cuda").uniform_(0.9, 1.1, generator=gen).to(torch.bfloat16)
    layer["q_norm"] *= sharp
    return layer


def _reference(torch, n_, config, layer, h):
    """(what the layer adds to h, keys, values) in float64, rounded to bf16 where the kernels do."""
    def bf(t):
        return t.to(torch.bfloat16).double()

    def rms(t, weight):
        return bf(t * torch.rsqrt(t.square().mean(dim=-1, keepdim=True) + config.eps) * weight.double())

    def project(x, name):
        return bf(x @ _dense(torch, n_, layer[name]).T)

    count = h.shape[0]
    angle = torch.arange(count, device="cuda", dtype=torch.float64)[:, None] * config.theta ** (
        -torch.arange(64, device="cuda", dtype=torch.float64) / 64)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(t):
        lo, hi = t[..., :64], t[..., 64:]
        return bf(torch.cat([lo * cos - hi * sin, lo * sin + hi * cos], dim=-1))

    h = h.double()
    x = rms(h, layer["input_norm"])
    q = rope(rms(project(x, "q").view(count, -1, 128), layer["q_norm"]))
    k = rope(rms(project(x, "k").view(count, -1, 128), layer["k_norm"]))
    v = project(x, "v").view(count, -1, 128)
    seen = torch.ones((count, count), dtype=torch.bool, device="cuda").tril()
    out = torch.empty_like(q)
    for head in range(config.heads):
        kv = head // (config.heads // config.kv_heads)
        scores = (q[:, head] @ k[:, kv].T) * 128 ** -0.5
        out[:, head] = scores.masked_fill(~seen, float("-inf")).softmax(dim=-1) @ v[:, kv]
    first = project(bf(out.flatten(1)), "o")
    x = rms(h + first, layer["post_norm"])
    gate, up = project(x, "gate"), project(x, "up")
    return first + project(bf(gate / (1 + (-gate).exp()) * up), "down"), k, v


def _run(torch, n_, config, layers, h, slots=2, slot=1):
    """The stream after the layers (every row) and the pools, through the C ABI's calls."""
    count, capacity = h.shape[0], h.shape[0] + 3
    pools = [[torch.zeros((slots, config.kv_heads, capacity, 128), dtype=torch.bfloat16, device="cuda")
              for _ in range(2)] for _ in layers]
    run = n_.PromptLayers(config, h.clone(), slots, capacity, slot)
    for layer, (k_pool, v_pool) in zip(layers, pools):
        run.layer(layer, k_pool, v_pool)
    n_._check(n_.lib().imq_prompt_finish(ctypes.byref(run.shape), run.h.data_ptr(), count, run.workspace.data_ptr(),
                                         run.nbytes, n_._stream(None)))
    for pool in (p for pair in pools for p in pair):
        assert not pool[1 - slot].any() and not pool[slot, :, count:].any()
    return run.h, [[p[slot, :, :count].transpose(0, 1).double() for p in pair] for pair in pools]


def _row_errors(got, ref):
    """Every row's relative 2-norm of the difference."""
    return (got.double() - ref).norm(dim=-1) / ref.norm(dim=-1)


# tokens, heads, kv_heads, hidden, intermediate, {launch: (rows of a tile, K-ranges)}
LAYERS = [
    # a long prompt's shape: two norm pieces a thread, gate/up in 64-row tiles, down in three K-ranges
    (512, 32, 8, 2560, 9728, {"gate_up": (64, 1), "o": (64, 1), "down": (128, 3)}),
    # gate/up in 128-row tiles, the last one in part; an odd head count (half a chunk of zeros)
    (4200, 3, 1, 192, 9728, {"gate_up": (128, 1)}),
    (1300, 16, 8, 320, 2048, {"qkv": (64, 1), "gate_up": (64, 1)}),
    (1030, 32, 8, 2560, 512, {"qkv": (128, 1)}),
    # o in K-ranges; four norm pieces a thread and odd heads over an o weight of unaligned scales
    (300, 32, 8, 192, 256, {"o": (32, 2)}),
    (70, 5, 5, 4160, 256, {"qkv": (32, 1)}),
    (1, 1, 1, 64, 64, {}),
    (33, 3, 3, 8192, 64, {}),
]


@pytest.mark.parametrize("tokens,heads,kv_heads,hidden,intermediate,plans", LAYERS)
def test_layers_one_at_a_time_against_64_bits(env, tokens, heads, kv_heads, hidden, intermediate, plans):
    torch, n_, orc = env
    announce("layer", tokens, heads, kv_heads, hidden, intermediate)
    q, kv = heads * 128, kv_heads * 128
    made = {"qkv": _plan(n_, [q, kv, kv], tokens, hidden, 1), "o": _plan(n_, [hidden], tokens, q),
            "gate_up": _plan(n_, [intermediate] * 2, tokens, hidden, 1),
            "down": _plan(n_, [hidden], tokens, intermediate)}
    for name, (rows, splits) in plans.items():
        assert made[name][0] == rows and (made[name][1] > 1) == (splits > 1), (name, made)
    config = _Config(heads, kv_heads, hidden, intermediate)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens)
    layers = [_layer(torch, gen, config), _layer(torch, gen, config, sharp=3.0)]
    h = torch.randn((tokens, hidden), device="cuda", generator=gen)

    def check(name, before, after, layer, pools, bar, mean=1.0):
        added, k, v = _reference(torch, n_, config, layer, before)
        keys, values, stream = (_row_errors(*pair) for pair in ((pools[0], k), (pools[1], v),
                                                                (after.double() - before.double(), added)))
        print("[row errors]", name, *(f"{float(e.max()):.5f}" for e in (keys, values, stream)),
              f"mean {float(stream.mean()):.6f}", flush=True)
        assert float(keys.max()) <= 2.0**-8 and float(values.max()) <= 2.0**-8
        assert float(stream.max()) <= bar and float(stream.mean()) <= mean

    # a layer whose down or whose o adds nothing: attention and MLP each by itself
    silent = {name: (layers[0][name][0], *(torch.zeros_like(t) for t in layers[0][name][1:])) for name in ("o", "down")}
    for name, off, bar, mean in (("attention", "down", 2.0**-7, 1.0), ("mlp", "o", 2.0**-8, 2.0**-11)):
        layer = dict(layers[0], **{off: silent[off]})
        out, pools = _run(torch, n_, config, [layer], h)
        check(name, h, out, layer, pools[0], bar, mean)
    # two layers; the second one's reference starts from the first one's own output
    one, _ = _run(torch, n_, config, layers[:1], h)
    two, pools = _run(torch, n_, config, layers, h)
    check("first layer", h, one, layers[0], pools[0], 2.0**-6)
    check("second layer", one, two, layers[1], pools[1], 2.0**-6)
    assert torch.equal(_run(torch, n_, config, layers, h)[0], two)  # no order of arrival in any sum


def test_layer_rows_of_huge_values_and_nan(env):
    """A row whose normed activations pass 2^96 gives finite gate, up and down values, computed one
    by one; NaN and infinities in the last rows stay in them."""
    torch, n_, orc = env
    announce("layer huge")
    tokens, config = 70, _Config(4, 2, 256, 512)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    layer = _layer(torch, gen, config)
    h = torch.randn((tokens, 256), device="cuda", generator=gen)
    h[:, 77] = 0.0
    for t in layer["o"][1:]:
        t[77] = 0.0  # o adds nothing to column 77,
    w, s, b = layer["up"]  # and up does not read it: 8 s - 8 s
    s.fill_(2.0**-7)
    b.fill_(-8 * 2.0**-7)
    w[:, 77 // 8] = (w[:, 77 // 8] & ~(15 << 4 * (77 % 8))) | (8 << 4 * (77 % 8))
    layer["post_norm"][77] = 2.0**100
    clean, _ = _run(torch, n_, config, [layer], h)
    h[37, 77] = 0.5
    ref, _, _ = _reference(torch, n_, config, layer, h)
    got, _ = _run(torch, n_, config, [layer], h)
    assert torch.equal(got[:37], clean[:37])
    assert float(ref[37].abs().max()) > 2.0**90 and torch.isfinite(got).all()
    assert float(_row_errors(got.double() - h.double(), ref).max()) <= 2.0**-6
    h[68, 3], h[69, 200] = float("inf"), float("nan")
    marked, _ = _run(torch, n_, config, [layer], h)
    assert torch.equal(marked[:64], got[:64]) and torch.isnan(marked[68:]).all()


# ------------------------------------------------------------------ products by tile height

@pytest.mark.parametrize("m,n,k,rows,splits", [
    (65, 33, 2560, 32, 5), (4200, 130, 1600, 64, 1), (2100, 33, 9728, 64, 7), (1700, 15990, 320, 128, 1),
    (97, 8200, 9728, 128, 3), (200, 10000, 9728, 128, 3)])
def test_products_of_each_tile_height(env, m, n, k, rows, splits):
    torch, n_, orc = env
    announce("product plan", m, n, k)
    made = _plan(n_, [n], m, k)
    assert made[0] == rows and (made[1] > 1) == (splits > 1), made
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m)
    quant, x = _weight(torch, gen, n, k), torch.randn((m, k), device="cuda", generator=gen).to(torch.bfloat16)
    x[m // 2, k // 2], x[m - 1, 0] = 1e38, float("nan")
    dense = _dense(torch, n_, quant)
    ref, mag = x.double() @ dense.T, x.double().abs() @ dense.abs().T
    del dense
    y = n_.prompt_matmul(*quant, x, torch.float32)
    assert torch.isnan(y[m - 1]).all()
    bound = 2.0**-20 * mag[:-1] + 2.0**-23 * ref[:-1].abs()
    bound[m // 2] += k * 2.0**-24 * mag[m // 2]  # the row added value by value
    assert ((y[:-1].double() - ref[:-1]).abs() <= bound).all()
    got = n_.prompt_matmul(*quant, x)
    assert ((got[:-1].double() - ref[:-1]).abs() <= bound + 2.0**-8 * ref[:-1].abs()).all()
    assert torch.equal(got[:-1], n_.prompt_matmul(*quant, x)[:-1])


@pytest.mark.parametrize("m,sizes,k,rows", [(65, (130, 66, 31), 9728, 32), (161, (1030, 514, 90), 9728, 64),
                                            (500, (131, 301), 9728, 32)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_grouped_products_in_k_ranges(env, m, sizes, k, rows, dtype):
    """Two and three weights whose planes are added by one launch, N off multiples of four."""
    torch, n_, orc = env
    announce("grouped plan", m, sizes, k, dtype)
    made = _plan(n_, sizes, m, k)
    assert made[0] == rows and made[1] > 1, made
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m)
    quants = [_weight(torch, gen, n, k) for n in sizes]
    x = torch.randn((m, k), device="cuda", generator=gen).to(torch.bfloat16)
    lib, stream, out = n_.lib(), n_._stream(None), getattr(torch, dtype)
    packed = torch.empty(lib.imq_prompt_packed_bytes(m, k), dtype=torch.uint8, device="cuda")
    n_._check(lib.imq_prompt_pack(x.data_ptr(), k, m, k, packed.data_ptr(), stream))
    # rows of y further apart than N, what lies between them kept
    ys = [torch.full((m, n + 5), 7.0, dtype=out, device="cuda") for n in sizes]
    arr = (n_.Problem * len(sizes))(*[n_.Problem(*(t.data_ptr() for t in quant), None, 0, y.data_ptr(), n + 5, n, k)
                                      for quant, y, n in zip(quants, ys, sizes)])
    nbytes = lib.imq_prompt_product_workspace(arr, len(sizes), m)
    assert nbytes == made[1] * m * sum(-(-n // 4) * 4 for n in sizes) * 4
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    n_._check(lib.imq_prompt_product(arr, len(sizes), packed.data_ptr(), m, 64, 4, n_._DTYPE_CODE[out], ws.data_ptr(),
                                     nbytes, stream))
    for quant, y, n in zip(quants, ys, sizes):
        dense = _dense(torch, n_, quant)
        ref, mag = x.double() @ dense.T, x.double().abs() @ dense.abs().T
        bound = 2.0**-20 * mag + (2.0**-8 if dtype == "bfloat16" else 2.0**-23) * ref.abs()
        assert ((y[:, :n].double() - ref).abs() <= bound).all()
        assert (y[:, n:] == 7.0).all()


@pytest.mark.parametrize("experts,tokens,top,n,rows", [
    (8, 28, 8, 12290, 32), (8, 29, 8, 12290, 64), (8, 160, 8, 66, 32), (8, 161, 8, 2200, 64), (1, 700, 1, 66, 32),
    (1, 3000, 1, 1100, 64), (1024, 40, 8, 66, 32)])
def test_expert_batches_of_each_tile_height(env, experts, tokens, top, n, rows):
    """Around the edges of the tile rule, with uneven experts: half of the pairs on the first one."""
    torch, n_, orc = env
    from ironmule_amd.quantized import library_gather_matmul
    announce("experts plan", experts, tokens, top, n)
    made = ctypes.c_int32()
    assert n_.lib().imq_prompt_experts_plan(experts, tokens * top, n, n_.device_check()[2], ctypes.byref(made)) == 0
    assert made.value == rows
    k = 192
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens)
    stack = tuple(t.view(experts, n, -1) for t in _weight(torch, gen, experts * n, k))
    x = torch.randn((tokens, 1, 1, k), device="cuda", generator=gen).to(torch.bfloat16)
    idx = torch.randint(0, experts, (tokens, top), device="cuda", generator=gen)
    idx[:, ::2] = 0
    y = library_gather_matmul(x, *stack, idx)[:, :, 0]
    dense = _dense(torch, n_, tuple(t.flatten(0, 1) for t in stack)).view(experts, n, k)
    for e in idx.unique().tolist():
        token, at = (idx == e).nonzero(as_tuple=True)
        rows_x = x[token, 0, 0].double()
        ref, mag = rows_x @ dense[e].T, rows_x.abs() @ dense[e].abs().T
        assert ((y[token, at].double() - ref).abs() <= 2.0**-8 * ref.abs() + 2.0**-20 * mag).all(), e
