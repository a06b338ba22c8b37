"""GPU parity of the product for more than 32 rows (imq_prompt_matmul, imq_prompt_product)
through the C ABI, against the oracle's float64 product.

Bars (the qmv kernels'): fp32 outputs within 2^-20 sum|w x| + 2^-23 |ref|, bf16 outputs within
one ulp of the rounded reference plus that allowance.  Sizes (32-row tiles; the taller ones, and
layers one at a time, are in test_prompt_layer_gpu.py): one row past a 32-row block, N off the 128
columns of a workgroup, K of one group, groups off the chunks of four (scales of every alignment),
and K-ranges.
"""

from __future__ import annotations

import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.gpu_util import announce, bf16_bits, to_device

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


@pytest.fixture(scope="module")
def env():
    import torch

    from ironmule_amd import _native
    from oracle import oracle as orc
    code, arch, _ = _native.device_check()
    assert code == 0, f"device {arch} is not supported"
    orc.lib()
    return torch, _native, orc


SIZES = [(33, 64, 64), (40, 130, 192), (65, 1, 256), (97, 300, 320), (129, 257, 1600), (77, 512, 9728),
         (200, 2560, 256), (512, 384, 2560), (600, 4100, 768), (2100, 2500, 128)]


@pytest.mark.parametrize("m,n,k", SIZES)
def test_prompt_matmul_against_the_oracle(env, m, n, k):
    torch, n_, orc = env
    announce("prompt", m, n, k)
    pr = orc.synthetic(n, k, m, seed=orc.SEED_BASE + 900 + m)
    w, s, b, x = to_device(pr)
    ref, mag = orc.qmv_f64(pr.w, pr.s, pr.b, pr.x)
    verdict = orc.check_f32(n_.prompt_matmul(w, s, b, x, torch.float32).cpu().numpy(), ref, mag)
    assert verdict.ok, verdict.detail
    got = n_.prompt_matmul(w, s, b, x)
    verdict = orc.check_bf16(bf16_bits(got), ref, mag)
    assert verdict.ok, verdict.detail
    assert torch.equal(got, n_.prompt_matmul(w, s, b, x))  # no order of arrival in any sum


def test_rows_and_scales_of_any_alignment(env):
    """x rows with a stride and rows off a 16-byte boundary, scales off an 8-byte boundary."""
    torch, n_, orc = env
    announce("prompt alignment")
    m, n, k = 70, 200, 512
    pr = orc.synthetic(n, k, m, seed=orc.SEED_BASE + 930)
    w, s, b, x = to_device(pr)
    want = n_.prompt_matmul(w, s, b, x)
    wide = torch.zeros((m, k + 72), dtype=torch.bfloat16, device="cuda")
    for at in (0, 8, 3):
        wide[:, at:at + k] = x
        assert torch.equal(n_.prompt_matmul(w, s, b, wide[:, at:at + k]), want), at
    odd = torch.empty(s.numel() + 1, dtype=torch.bfloat16, device="cuda")[1:].view_as(s)
    odd.copy_(s)
    assert torch.equal(n_.prompt_matmul(w, odd, b, x), want)


def test_infinities_nan_and_large_values_stay_in_their_rows(env):
    """A row whose values could overflow the group sums is computed value by value: infinities
    keep their sign, NaN stays NaN, 1e38 gives the finite result, and other rows keep their bits."""
    torch, n_, orc = env
    announce("prompt non-finite rows")
    m, n, k = 100, 200, 320
    w, s, b, x = to_device(orc.synthetic(n, k, m, seed=orc.SEED_BASE + 940))
    clean = n_.prompt_matmul(w, s, b, x, torch.float32)
    x[5, 7], x[50, 100], x[64, 319], x[99, 0] = float("inf"), float("nan"), -float("inf"), 1e38
    y = n_.prompt_matmul(w, s, b, x, torch.float32).double()
    ref = x.double() @ n_.dequant(w, s, b).double().T
    touched = [5, 50, 64, 99]
    others = [r for r in range(m) if r not in touched]
    assert torch.equal(y[others], clean[others].double())
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert inf.any() and torch.equal(y[inf], ref[inf])
    # the 1e38 row: one term dominates, fp32 rounding of 320 terms
    assert ((y[99] - ref[99]).abs() <= 320 * 2.0**-24 * (x[99].double().abs() @ n_.dequant(w, s, b).double().abs().T)).all()


def test_more_rows_than_a_launch_dimension(env):
    """600,000 rows (150,000 workgroups of eight rows): first, middle and last rows against a
    product of those rows alone."""
    torch, n_, orc = env
    announce("prompt many rows")
    w, s, b, _ = to_device(orc.synthetic(48, 64, 1, seed=orc.SEED_BASE + 945))
    x = torch.randn((600_000, 64), device="cuda").to(torch.bfloat16)
    y = n_.prompt_matmul(w, s, b, x)
    for at in (0, 299_990, 599_960):
        assert torch.equal(y[at:at + 40], n_.prompt_matmul(w, s, b, x[at:at + 40]))


def test_grouped_products_share_one_packing(env):
    """Three weights of one K, N off multiples of four and of 128, over one packing."""
    import ctypes
    torch, n_, orc = env
    announce("prompt grouped")
    m, k, sizes = 161, 1024, (300, 131, 64)
    probs = [orc.synthetic(n, k, m, seed=orc.SEED_BASE + 950 + n) for n in sizes]
    x = to_device(probs[0])[3]
    weights = [to_device(p)[:3] for p in probs]
    lib = n_.lib()
    packed = torch.empty(lib.imq_prompt_packed_bytes(m, k), dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.imq_prompt_pack(x.data_ptr(), k, m, k, packed.data_ptr(), stream) == 0
    outs = [torch.empty((m, n), dtype=torch.float32, device="cuda") for n in sizes]
    arr = (n_.Problem * 3)(*[n_.Problem(w.data_ptr(), s.data_ptr(), b.data_ptr(), None, 0, y.data_ptr(), n, n, k)
                             for (w, s, b), y, n in zip(weights, outs, sizes)])
    ws = torch.empty(lib.imq_prompt_product_workspace(arr, 3, m) + 16, dtype=torch.uint8, device="cuda")
    assert lib.imq_prompt_product(arr, 3, packed.data_ptr(), m, 64, 4, n_.IMQ_F32, ws.data_ptr(), ws.numel(), stream) == 0
    for p, y in zip(probs, outs):
        ref, mag = orc.qmv_f64(p.w, p.s, p.b, probs[0].x)
        verdict = orc.check_f32(y.cpu().numpy(), ref, mag)
        assert verdict.ok, verdict.detail


def test_calls_that_autograd_follows_keep_the_torch_product(env):
    torch, n_, orc = env
    from ironmule_amd import hip_native
    announce("prompt autograd")
    w, s, b, x = to_device(orc.synthetic(64, 128, 40, seed=orc.SEED_BASE + 960))
    x.requires_grad_(True)
    hip_native.matmul(x, w, s, b).float().sum().backward()
    dense = n_.dequant(w, s, b)
    want = dense.sum(dim=0).expand(40, 128)
    assert (x.grad.float() - want).abs().max() <= 2.0**-7 * want.abs().max()  # fp16 weights, bf16 gradient


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("native", [False, True])
def test_a_traced_module_computes_new_inputs(env, native):
    """torch.jit.trace records torch operations: the trace has to hold the product, not its result,
    and the dequantised weight as a constant (device memory is overwritten before the replay)."""
    torch, n_, orc = env
    from ironmule_amd import hip_native
    from ironmule_amd.quantized import QuantizedLinear
    announce("traced module", native)
    m, n, k = 40, 96, 256
    w, s, b, x = to_device(orc.synthetic(n, k, m, seed=orc.SEED_BASE + 965))
    module = (hip_native.NativeQuantizedLinear if native else QuantizedLinear)(w, s, b)
    traced = torch.jit.trace(module, x, check_trace=False)
    junk = [torch.full((n, k), 7.0, device="cuda") for _ in range(8)] + [torch.full((n, k), 7.0, device="cuda").half() for _ in range(8)]
    del junk
    other = torch.randn((m, k), device="cuda").to(torch.bfloat16)
    dense = n_.dequant(w, s, b).double()
    ref, mag = other.double() @ dense.T, other.double().abs() @ dense.abs().T
    # bf16 outputs; weights rounded to fp16 in the native module, fp32 sums in the plain one
    assert ((traced(other).double() - ref).abs() <= 2.0**-8 * ref.abs() + 2.0**(-11 if native else -20) * mag).all()


@pytest.mark.parametrize("e,n,k,tokens,top", [(8, 130, 192, 13, 5), (32, 256, 768, 128, 8), (3, 100, 1600, 200, 2),
                                              (64, 64, 256, 9, 8), (2, 300, 512, 400, 1)])
@pytest.mark.parametrize("shared", [True, False])
def test_expert_batches_against_the_oracle(env, e, n, k, tokens, top, shared):
    """Pairs sorted by expert, experts without pairs (64 experts, 72 pairs on the even ones), a token's
    row shared by its experts or a row per pair."""
    torch, n_, orc = env
    from ironmule_amd.quantized import library_gather_matmul
    announce("experts", e, n, k, tokens, top, shared)
    stack = [orc.synthetic(n, k, 1, seed=orc.SEED_BASE + 970 + i) for i in range(e)]
    w, s, b = (np.stack([getattr(p, f) for p in stack]) for f in "wsb")
    dw = torch.from_numpy(w.view(np.int32)).cuda()
    ds, db = (torch.from_numpy(t).cuda().view(torch.bfloat16) for t in (s, b))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens)
    x = torch.randn((tokens, 1 if shared else top, 1, k), device="cuda", generator=gen).to(torch.bfloat16)
    idx = torch.randint(0, e, (tokens, top), device="cuda", generator=gen)
    if e == 64:
        idx = idx // 2 * 2
    y = library_gather_matmul(x, dw, ds, db, idx)
    assert tuple(y.shape) == (tokens, top, 1, n)
    ref, mag = orc.gather_qmv_f64(w, s, b, bf16_bits(x.reshape(-1, k)), idx.reshape(-1).cpu().numpy(),
                                  top if shared else 1)
    verdict = orc.check_bf16(bf16_bits(y.reshape(-1, n)), ref, mag)
    assert verdict.ok, verdict.detail
    wrapped = torch.where(idx % 3 == 0, idx - e, idx)  # the same experts counted from the last
    assert torch.equal(library_gather_matmul(x, dw, ds, db, wrapped), y)


def test_expert_batch_forms(env):
    """Several rows per pair, a broadcast index and indices outside the stack."""
    torch, n_, orc = env
    from ironmule_amd.quantized import library_gather_matmul
    announce("expert forms")
    e, n, k = 4, 96, 320
    stack = [to_device(orc.synthetic(n, k, 1, seed=orc.SEED_BASE + 990 + i)) for i in range(e)]
    w, s, b = (torch.stack([p[f] for p in stack]) for f in range(3))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    x = torch.randn((6, 1, 3, k), device="cuda", generator=gen).to(torch.bfloat16)
    idx = torch.randint(0, e, (5,), device="cuda", generator=gen)
    y = library_gather_matmul(x, w, s, b, idx)
    assert tuple(y.shape) == (6, 5, 3, n)
    for t in range(6):
        for j in range(5):
            i = int(idx[j])
            want = x[t, 0].double() @ n_.dequant(w[i], s[i], b[i]).double().T
            assert (y[t, j].double() - want).abs().max() <= 2.0**-8 * want.abs().max()
    out = n_.prompt_experts(w, s, b, x[:, 0, 0], torch.tensor([0, 4, -5, 3, 2, 1], device="cuda"))
    assert not out[1].any() and not out[2].any() and out[0].any() and out[3:].any(dim=1).all()


def test_expert_stacks_of_any_stride_and_alignment(env):
    """One half of a fused gate/up stack, every other expert, scales of another order and words off a
    16-byte boundary: the same products as a stack copied whole, through both entry points."""
    torch, n_, orc = env
    from ironmule_amd import hip_native
    from ironmule_amd.quantized import library_gather_matmul
    announce("expert stack strides")
    e, n, k, tokens, top = 8, 128, 256, 20, 4
    stack = [to_device(orc.synthetic(n, k, 1, seed=orc.SEED_BASE + 1000 + i)) for i in range(e)]
    whole = tuple(torch.stack([p[f] for p in stack]) for f in range(3))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    x = torch.randn((tokens, 1, 1, k), device="cuda", generator=gen).to(torch.bfloat16)
    off = torch.empty(whole[0].numel() + 1, dtype=torch.int32, device="cuda")[1:].view_as(whole[0]).copy_(whole[0])
    turned = whole[1].transpose(0, 1).contiguous().transpose(0, 1)
    for w, s, b in (tuple(t[:, n // 2:] for t in whole), tuple(t[::2] for t in whole), (off, *whole[1:]),
                    (whole[0], turned, whole[2])):
        idx = torch.randint(0, w.shape[0], (tokens, top), device="cuda", generator=gen)
        copied = [t.clone(memory_format=torch.contiguous_format) for t in (w, s, b)]
        want = library_gather_matmul(x, *copied, idx).float()
        for call in (library_gather_matmul, hip_native.gather_matmul):
            got = call(x, w, s, b, idx).float()
            # two fp32 sums, each within 2^-20 sum|w x| (at most 16 times the outputs' root mean square
            # at K = 256) and rounded to bf16: one ulp, at most 2^-7 of the value, and that much
            assert ((got - want).abs() <= 2.0**-7 * want.abs() + 2.0**-15 * want.abs().max()).all()


@pytest.mark.parametrize("tokens,heads,kv_heads,hidden,intermediate", [
    (1, 4, 2, 256, 512), (16, 4, 2, 256, 512), (33, 6, 3, 320, 448), (63, 8, 1, 192, 256), (64, 4, 4, 256, 512),
    (65, 4, 2, 256, 512), (130, 8, 2, 576, 1088), (257, 16, 2, 1024, 768)])
def test_prompt_layers_against_the_torch_composition(env, monkeypatch, tokens, heads, kv_heads, hidden, intermediate):
    """A prompt through imq_prompt_layer and through the same steps in torch operations: both
    round to bf16 at the same places, so keys and values differ by a rounding (an ulp is 2^-8 of a
    value, and a layer's differences pass through the next) and nothing outside the prompt's rows
    is written.  Query blocks of 64 in part and in full, grouped heads, K off the chunks."""
    torch, n_, orc = env
    from ironmule_amd import decode
    announce("prompt layers", tokens, heads, kv_heads, hidden, intermediate)
    cfg = decode.DecoderConfig(hidden=hidden, layers=3, heads=heads, kv_heads=kv_heads, head_dim=128,
                               intermediate=intermediate, vocab=512)
    weights = decode.random_weights(cfg, "cuda", seed=tokens)
    for layer in weights.layers:  # zero-mean weights: the layers' outputs do not line up
        for name in cfg.projections:
            layer[name][2].copy_(layer[name][1] * -7.5)
    ids = np.random.default_rng(tokens).integers(0, cfg.vocab, tokens).tolist()
    states = [decode.DecodeState(cfg, batch=1, slots=3, capacity=tokens + 5, max_len=tokens + 5, device="cuda")
              for _ in range(2)]
    got = decode.prefill(weights, states[0], ids, 1)
    monkeypatch.setattr(decode, "_layers_fit", lambda *a: False)
    want = decode.prefill(weights, states[1], ids, 1)
    assert (got - want).abs().max() <= 2.0**-6 * want.abs().max()
    for mine, theirs in zip(states[0].k_pool + states[0].v_pool, states[1].k_pool + states[1].v_pool):
        assert not mine[0].any() and not mine[2].any() and not mine[1, :, tokens:].any()
        assert (mine.float() - theirs.float()).abs().max() <= 2.0**-6 * theirs.float().abs().max()


def test_prompt_layers_replay_in_a_graph(env):
    """A captured prompt (the layers alone: the embedding is set before) gives the eager bits on
    every replay, with eager work between the replays."""
    torch, n_, orc = env
    from ironmule_amd import decode
    announce("prompt layers graph")
    cfg = decode.DecoderConfig(hidden=256, layers=2, heads=4, kv_heads=2, head_dim=128, intermediate=512, vocab=512)
    weights = decode.random_weights(cfg, "cuda", seed=3)
    state = decode.DecodeState(cfg, batch=1, slots=1, capacity=80, max_len=80, device="cuda")
    start = torch.randn((70, 256), device="cuda")
    h, out = torch.empty_like(start), torch.empty((1, 256), device="cuda")

    def go():
        h.copy_(start)
        run = n_.PromptLayers(cfg, h, 1, 80, 0)
        for layer, k, v in zip(weights.layers, state.k_pool, state.v_pool):
            run.layer(layer, k, v)
        out.copy_(run.finish())

    go()
    want = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        go()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        torch.randn(1 << 16, device="cuda").sum().item()


@pytest.mark.parametrize("m,k", [(33, 3840), (4095, 3840), (4096, 3840), (5120, 3072), (8192, 2560)])
def test_native_rows_keep_their_range_at_any_length(env, m, k):
    """Activations past fp16's range (65504) and up to 1e38 give the finite products they give in a
    short prompt, however long the prompt is."""
    torch, n_, orc = env
    from ironmule_amd import hip_native
    announce("native range", m, k)
    x = torch.randn((m, k), device="cuda").to(torch.bfloat16)
    x[7, 5], x[9] = 1e38, x[9] * 1e5
    assert hip_native._route(x, k) == "prompt"
    w, s, b, _ = to_device(orc.synthetic(64, k, 1, seed=orc.SEED_BASE + 980))
    y = hip_native.matmul(x, w, s, b).double()
    dense = n_.dequant(w, s, b).double()
    ref, mag = x.double() @ dense.T, x.double().abs() @ dense.abs().T
    assert torch.isfinite(ref.float()).all()
    # one rounding to bf16, and fp32 sums: 2^-20 sum|w x|, the row of one large value added value by
    # value, k roundings of 2^-24
    bound = 2.0**-8 * ref.abs() + 2.0**-20 * mag
    bound[7] += k * 2.0**-24 * mag[7]
    assert ((y - ref).abs() <= bound).all()
