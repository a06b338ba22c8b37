"""GPU parity of the decode-step kernels (include/ironmule_decode.h) and of a whole
decode step, against the decode oracle, through the C ABI.

Bars: embedding rows and the residual add bit-exact (fp32); RMSNorm, SiLU * up and
attention outputs within one bf16 ulp of the float64 reference plus a small absolute
allowance for cancellation; q/k after norm + rotation within two bf16 ulps of their
pair's length (the rotation mixes two values that each carry one rounding); v and the
KV placement exact.  The whole step (a small decoder: 2 layers, hidden 256, 4/2 heads)
within max|logit - ref| / max|ref| <= 2e-7 (RMSNorm launches) or 5e-4 (RMSNorms folded into
the projections) of the oracle step with the same bf16 rounding points: about twice the
observed values (the reference's own probe tolerance is 1e-2, ironmule/cuda_native.py:253-268).
"""

from __future__ import annotations

import math

import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.gpu_util import announce, bf16_bits

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

RNG = np.random.default_rng(20261207)


@pytest.fixture(scope="module")
def env():
    import torch

    from ironmule_amd import _native
    from oracle import decode_oracle as do
    from oracle import oracle as orc
    code, arch, _ = _native.device_check()
    assert code == 0, f"device {arch} is not supported"
    orc.lib()
    return torch, _native, do, orc


def _bf16(torch, a, device="cuda"):
    """float array -> bf16 device tensor (round to nearest even) and its exact values."""
    t = torch.from_numpy(np.asarray(a, np.float32)).to(torch.bfloat16)
    return t.to(device), t.float().numpy().astype(np.float64)


def _vals(t):
    return t.float().cpu().numpy().astype(np.float64)


def _ulp(v):
    from oracle import oracle as orc
    return orc.bf16_ulp(np.asarray(v, np.float32)).astype(np.float64)


def test_embed_rows_are_bit_exact(env):
    torch, n, do, orc = env
    announce("embed 1000 x 512")
    pr = orc.synthetic(1000, 512, 1, seed=11)
    w = torch.from_numpy(pr.w.view(np.int32)).cuda()
    s = torch.from_numpy(pr.s).view(torch.bfloat16).cuda()
    b = torch.from_numpy(pr.b).view(torch.bfloat16).cuda()
    tokens = torch.tensor([0, 999, 17, 17, 500], dtype=torch.int32, device="cuda")
    h = torch.empty((5, 512), dtype=torch.float32, device="cuda")
    n.embed(w, s, b, tokens, h)
    want = orc.dequant_f32(pr.w, pr.s, pr.b)[[0, 999, 17, 17, 500]]
    assert np.array_equal(h.cpu().numpy().view(np.uint32), want.view(np.uint32))
    bad = torch.tensor([1000, -1], dtype=torch.int32, device="cuda")
    h2 = torch.zeros((2, 512), dtype=torch.float32, device="cuda")
    n.embed(w, s, b, bad, h2)
    assert torch.isnan(h2).all()


@pytest.mark.parametrize("rows,dim,with_delta", [(1, 2560, True), (32, 2560, True), (3, 100, False),
                                                 (2, 8192, True)])
def test_add_rmsnorm(env, rows, dim, with_delta):
    torch, n, do, orc = env
    announce("add_rmsnorm", rows, dim, with_delta)
    h0 = RNG.standard_normal((rows, dim)).astype(np.float32) * 3
    h = torch.from_numpy(h0.copy()).cuda()
    w, wv = _bf16(torch, RNG.uniform(0.5, 1.5, dim))
    delta, dv = _bf16(torch, RNG.standard_normal((rows, dim)))
    out = torch.empty((rows, dim), dtype=torch.bfloat16, device="cuda")
    n.add_rmsnorm(h, w, out, 1e-6, delta=delta if with_delta else None)
    h_new = h0 + (dv.astype(np.float32) if with_delta else 0)
    assert np.array_equal(h.cpu().numpy(), h_new.astype(np.float32))  # the add is exact fp32
    ref = do.rms_norm(h_new.astype(np.float64), wv, 1e-6)
    err = np.abs(_vals(out) - ref)
    assert (err <= _ulp(ref) + 1e-6 * np.abs(ref).max()).all(), err.max()


@pytest.mark.parametrize("B,hq,hkv", [(1, 32, 8), (32, 32, 8), (3, 8, 8)])
def test_qk_norm_rope_and_kv_write(env, B, hq, hkv):
    torch, n, do, orc = env
    announce("qk_norm_rope", B, hq, hkv)
    slots_n, cap, theta, eps = max(B, 4), 700, 1e6, 1e-6
    q, qv = _bf16(torch, RNG.standard_normal((B, hq * 128)))
    k, kv = _bf16(torch, RNG.standard_normal((B, hkv * 128)))
    v, vv = _bf16(torch, RNG.standard_normal((B, hkv * 128)))
    qn, qnv = _bf16(torch, RNG.uniform(0.8, 1.2, 128))
    kn, knv = _bf16(torch, RNG.uniform(0.8, 1.2, 128))
    slots = RNG.permutation(slots_n)[:B].astype(np.int32)
    pos = RNG.integers(0, cap, B).astype(np.int32)
    pos[0] = cap - 1
    kp = torch.zeros((slots_n, hkv, cap, 128), dtype=torch.bfloat16, device="cuda")
    vp = torch.zeros_like(kp)
    q_out = torch.empty((B, hq * 128), dtype=torch.bfloat16, device="cuda")
    n.qk_norm_rope(q, k, v, qn, kn, torch.from_numpy(pos).cuda(), torch.from_numpy(slots).cuda(),
                   q_out, kp, vp, theta, eps)

    def reference(x, nw, heads):
        x = x.reshape(B, heads, 128)
        normed = do.bf16_round(do.rms_norm(x, nw, eps))
        return do.rope(normed, pos, theta), normed

    for got, (ref, normed) in ((_vals(q_out).reshape(B, hq, 128), reference(qv, qnv, hq)),
                               (_vals(kp)[slots, :, pos], reference(kv, knv, hkv))):
        pair = np.sqrt(normed[..., :64] ** 2 + normed[..., 64:] ** 2)
        bound = 2.0 ** -7 * np.concatenate([pair, pair], axis=-1) + 1e-30
        err = np.abs(got - ref)
        assert (err <= bound).all(), (err / bound).max()
    assert np.array_equal(bf16_bits(vp)[slots, :, pos], bf16_bits(v).reshape(B, hkv, 128))
    # nothing else was written
    mask = np.zeros((slots_n, cap), bool)
    mask[slots, pos] = True
    assert not bf16_bits(kp).transpose(0, 2, 1, 3)[~mask].any()
    assert not bf16_bits(vp).transpose(0, 2, 1, 3)[~mask].any()


def test_qk_norm_rope_refuses_out_of_range_requests(env):
    torch, n, do, orc = env
    announce("qk_norm_rope refusals")
    q = torch.ones((2, 8 * 128), dtype=torch.bfloat16, device="cuda")
    k = torch.ones((2, 2 * 128), dtype=torch.bfloat16, device="cuda")
    kp = torch.zeros((2, 2, 16, 128), dtype=torch.bfloat16, device="cuda")
    vp = torch.zeros_like(kp)
    q_out = torch.zeros_like(q)
    norm = torch.ones(128, dtype=torch.bfloat16, device="cuda")
    n.qk_norm_rope(q, k, k, norm, norm, torch.tensor([16, 3], dtype=torch.int32, device="cuda"),
                   torch.tensor([0, 2], dtype=torch.int32, device="cuda"), q_out, kp, vp, 1e6, 1e-6)
    assert not kp.any() and not vp.any() and not q_out.any()


def _fused_pair(torch, n, B, positions, slots, slots_n, hq=32, hkv=8, cap=700, max_len=700,
                seed=0):
    """The same inputs through imq_attention_fused and through imq_qk_norm_rope followed
    by imq_attention_decode (lengths positions + 1, or 0 for an invalid request, the fused
    entry's contract); returns both (out, k_pool, v_pool), the fused call's arguments and
    its split counters."""
    g = np.random.default_rng(seed)
    q, _ = _bf16(torch, g.standard_normal((B, hq * 128)))
    k, _ = _bf16(torch, g.standard_normal((B, hkv * 128)))
    v, _ = _bf16(torch, g.standard_normal((B, hkv * 128)))
    qn, _ = _bf16(torch, g.uniform(0.8, 1.2, 128))
    kn, _ = _bf16(torch, g.uniform(0.8, 1.2, 128))
    kp, _ = _bf16(torch, g.standard_normal((slots_n, hkv, cap, 128)))
    vp, _ = _bf16(torch, g.standard_normal((slots_n, hkv, cap, 128)))
    pos = torch.tensor(positions, dtype=torch.int32, device="cuda")
    sl = torch.tensor(slots, dtype=torch.int32, device="cuda")
    theta, eps = 1e6, 1e-6
    kp_a, vp_a = kp.clone(), vp.clone()
    q_rot = torch.empty_like(q)
    out_a = torch.full((B, hq, 128), 7.0, dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(n.attention_workspace(B, hq, max_len), dtype=torch.float32, device="cuda")
    n.qk_norm_rope(q, k, v, qn, kn, pos, sl, q_rot, kp_a, vp_a, theta, eps)
    valid = (pos >= 0) & (pos < cap) & (sl >= 0) & (sl < slots_n)
    lengths = torch.where(valid, pos + 1, torch.zeros_like(pos))  # the fused entry's contract
    n.attention_decode(q_rot, kp_a, vp_a, lengths, sl, out_a, max_len, 128 ** -0.5, ws)
    kp_b, vp_b = kp.clone(), vp.clone()
    out_b = torch.full((B, hq, 128), -7.0, dtype=torch.bfloat16, device="cuda")
    ws_b = torch.empty_like(ws)
    counters = torch.zeros(B * hkv, dtype=torch.int32, device="cuda")
    fused = (q, k, v, qn, kn, pos, sl, kp_b, vp_b, out_b, max_len, theta, eps, ws_b, counters)
    n.attention_fused(*fused)
    torch.cuda.synchronize()
    return (out_a, kp_a, vp_a), (out_b, kp_b, vp_b), fused, counters


def _fused_against_oracle(a, b, positions, slots, slots_n, cap, hq=32, hkv=8):
    """The fused call's KV pools equal the three-launch form's bit for bit, and its output
    is within the attention bar of the oracle over the three-launch form's rotated q and
    pools (zeros for an invalid request)."""
    out_a, kp_a, vp_a = a
    out_b, kp_b, vp_b = b
    assert np.array_equal(bf16_bits(kp_a), bf16_bits(kp_b))
    assert np.array_equal(bf16_bits(vp_a), bf16_bits(vp_b))
    return _vals(out_b)


# 8, 16 and 32 requests over 8 KV heads take the wide plan (12 wavefronts per workgroup; for
# these 700-row pools four splits of 192 keys per (request, KV head) at 8, two at 16, one at
# 32): positions at the 16-key unit, 64-key chunk and split boundaries and at the last row
# of the pools
WIDE_8 = [699, 191, 192, 0, 383, 384, 575, 576]
WIDE_16 = [699, 0, 255, 256, 64, 383, 384, 511, 512, 17, 640, 641, 320, 321, 5, 698]
WIDE_32 = [0, 1, 15, 16, 63, 64, 65, 127, 128, 191, 192, 255, 256, 257, 300, 383, 384, 447,
           448, 511, 512, 513, 575, 576, 600, 639, 640, 650, 690, 698, 699, 100]


@pytest.mark.parametrize("B,positions", [(1, [63]), (1, [64]), (1, [511]), (1, [699]),
                                         (3, [0, 127, 128]), (3, [64, 650, 5]),
                                         (8, WIDE_8), (16, WIDE_16), (32, WIDE_32)])
def test_attention_fused_matches_the_oracle_and_writes_the_same_pools(env, B, positions):
    """imq_attention_fused against imq_qk_norm_rope + imq_attention_decode: both KV pools
    bit for bit, and the attention output within the attention bar of the oracle's
    attention over the rotated q and the pools, with positions on both sides of the 64-key
    chunk (split) boundaries, at the last row of the pools, for three requests, and for 8,
    16 and 32 requests (the wide plan); a second call (its split counters back at zero)
    repeats its bits."""
    torch, n, do, orc = env
    announce("attention fused vs oracle", B, positions)
    slots = list(RNG.permutation(B + 2)[:B].astype(int))
    cap = 700
    a, b, fused, counters = _fused_pair(torch, n, B, positions, slots, B + 2, seed=B * 1000 + positions[0])
    got = _fused_against_oracle(a, b, positions, slots, B + 2, cap)
    q_rot = _vals(fused_q_rot(torch, n, fused))
    kp, vp = _vals(a[1]), _vals(a[2])
    for r in range(B):
        L = positions[r] + 1
        ref = do.attention(q_rot[r].reshape(32, 128), kp[slots[r], :, :L], vp[slots[r], :, :L], 128 ** -0.5)
        err = np.abs(got[r].reshape(32, 128) - ref)
        bound = _ulp(ref) + 1e-5 * np.abs(vp[slots[r], :, :L]).max()
        assert (err <= bound).all(), (r, (err - bound).max())
    assert not counters.any()
    first = bf16_bits(b[0]).copy()
    n.attention_fused(*fused)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits(b[0]), first)


@pytest.mark.parametrize("B,positions,cap", [(1, [1023], 1024), (1, [1024], 1025), (1, [2099], 2100),
                                             (4, [0, 1087, 640, 1500], 1600), (6, [5, 1279, 64, 1200, 1, 900], 1280),
                                             (14, [37 * r for r in range(14)], 520),
                                             (20, [26 * r for r in range(20)], 520)])
def test_attention_fused_long_contexts_and_split_counts(env, B, positions, cap):
    """The wide plan below 64 (request, KV head) pairs, from 17 chunks of 64 keys (16 keep the
    narrow one), and request counts whose pairs do not divide 256: as the test above."""
    torch, n, do, orc = env
    announce("attention fused long", B, cap)
    slots = list(RNG.permutation(B + 1)[:B].astype(int))
    a, b, fused, counters = _fused_pair(torch, n, B, positions, slots, B + 1, cap=cap, max_len=cap, seed=B + cap)
    got = _fused_against_oracle(a, b, positions, slots, B + 1, cap)
    q_rot = _vals(fused_q_rot(torch, n, fused))
    kp, vp = _vals(a[1]), _vals(a[2])
    for r in range(B):
        L = positions[r] + 1
        ref = do.attention(q_rot[r].reshape(32, 128), kp[slots[r], :, :L], vp[slots[r], :, :L], 128 ** -0.5)
        err = np.abs(got[r].reshape(32, 128) - ref)
        assert (err <= _ulp(ref) + 1e-5 * np.abs(vp[slots[r], :, :L]).max()).all(), (r, err.max())
    assert not counters.any()
    first = bf16_bits(b[0]).copy()
    n.attention_fused(*fused)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits(b[0]), first)


@pytest.mark.parametrize("B,positions,cap", [
    # a cache of 17 to 32 chunks, narrow with shared chunks: 16 chunks, 17 (two a split), nearly all
    (1, [1023], 1100), (1, [1024], 2048), (1, [2040], 2048), (1, [3], 2048),
    # 8 wavefronts: two chunks a split and less, more splits than a merge loads, the last one in part
    (1, [2047], 4096), (1, [2048], 4096), (1, [4090], 4096), (2, [129, 4000], 4096), (3, [0, 700, 2040], 2048),
    # 12 wavefronts: short requests beside full ones, 128 chunks and 129
    (4, [8191, 64, 1000, 8192], 8200), (5, [31, 4095, 900, 2000, 6], 4096), (2, [16383, 9000], 16384),
    (8, [500 * r + 63 for r in range(8)], 4096), (14, [147 * r for r in range(14)], 2048)])
def test_attention_fused_short_requests_in_roomy_caches(env, B, positions, cap):
    """Each request's chunks shared over its own splits, at lengths around the shares' edges: the
    oracle's attention and the composition's pools, counters back at zero, the same bits again."""
    test_attention_fused_long_contexts_and_split_counts(env, B, positions, cap)


def fused_q_rot(torch, n, fused):
    """The rotated q of the fused call's inputs, by imq_qk_norm_rope on fresh pools."""
    q, k, v, qn, kn, pos, sl, kp, vp, out, max_len, theta, eps, ws, counters = fused
    q_rot = torch.empty_like(q)
    n.qk_norm_rope(q, k, v, qn, kn, pos, sl, q_rot, kp.clone(), vp.clone(), theta, eps)
    torch.cuda.synchronize()
    return q_rot


def test_attention_fused_bad_requests(env):
    """A request with a slot outside the pools or a position at the capacity gets a zero
    output and writes nothing, in both forms, and the valid request beside them meets the
    oracle's attention bar."""
    torch, n, do, orc = env
    announce("attention fused bad requests")
    cap = 96
    a, b, fused, _ = _fused_pair(torch, n, 3, [40, 10, cap], [1, 7, 0], 3, cap=cap, max_len=cap, seed=5)
    out = _fused_against_oracle(a, b, [40, 10, cap], [1, 7, 0], 3, cap)
    assert np.isfinite(out[0]).all() and out[0].any()
    assert not out[1].any() and not out[2].any()
    q_rot = _vals(fused_q_rot(torch, n, fused))
    kp, vp = _vals(a[1]), _vals(a[2])
    ref = do.attention(q_rot[0].reshape(32, 128), kp[1, :, :41], vp[1, :, :41], 128 ** -0.5)
    err = np.abs(out[0].reshape(32, 128) - ref)
    assert (err <= _ulp(ref) + 1e-5 * np.abs(vp[1, :, :41]).max()).all(), err.max()


def test_attention_fused_bad_requests_wide_plan(env):
    """The same at 8 requests (the 12-wavefront plan, splits of 192 keys): a slot outside
    the pools and a position at the capacity give zeros and write nothing, a request at
    position 0 attends to its new key alone, and the valid requests meet the oracle's
    bar."""
    torch, n, do, orc = env
    announce("attention fused bad requests, wide plan")
    cap = 700
    positions = [40, 10, cap, 0, 699, 191, 384, 5]
    slots = [1, 9, 0, 2, 3, 4, 5, 6]  # 9: past the 8 slots
    a, b, fused, counters = _fused_pair(torch, n, 8, positions, slots, 8, seed=8)
    out = _fused_against_oracle(a, b, positions, slots, 8, cap)
    assert not out[1].any() and not out[2].any()
    q_rot = _vals(fused_q_rot(torch, n, fused))
    kp, vp = _vals(a[1]), _vals(a[2])
    for r in (0, 3, 4, 5, 6, 7):
        L = positions[r] + 1
        ref = do.attention(q_rot[r].reshape(32, 128), kp[slots[r], :, :L], vp[slots[r], :, :L], 128 ** -0.5)
        err = np.abs(out[r].reshape(32, 128) - ref)
        assert (err <= _ulp(ref) + 1e-5 * np.abs(vp[slots[r], :, :L]).max()).all(), (r, err.max())
    assert not counters.any()


def _attention_case(torch, n, do, B, hq, hkv, lengths, cap=600, slots_n=None, max_len=None):
    slots_n = slots_n or B + 1
    kp, kpv = _bf16(torch, RNG.standard_normal((slots_n, hkv, cap, 128)))
    vp, vpv = _bf16(torch, RNG.standard_normal((slots_n, hkv, cap, 128)))
    q, qv = _bf16(torch, RNG.standard_normal((B, hq, 128)))
    slots = RNG.permutation(slots_n)[:B].astype(np.int32)
    lengths = np.asarray(lengths, np.int32)
    max_len = max_len or max(1, int(lengths.max()))
    out = torch.empty((B, hq, 128), dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(n.attention_workspace(B, hq, max_len), dtype=torch.float32, device="cuda")
    args = (q, kp, vp, torch.from_numpy(lengths).cuda(), torch.from_numpy(slots).cuda(), out,
            max_len, 128 ** -0.5, ws)
    n.attention_decode(*args)
    return args, out, (qv, kpv, vpv, slots, lengths)


@pytest.mark.parametrize("B,hq,hkv,lengths", [
    (1, 32, 8, [513]), (5, 32, 8, [1, 63, 64, 65, 513]), (32, 32, 8, None),
    (3, 8, 8, [7, 128, 300]), (2, 16, 2, [200, 129]), (2, 8, 1, [64, 1])])
def test_attention_matches_oracle(env, B, hq, hkv, lengths):
    torch, n, do, orc = env
    lengths = lengths if lengths is not None else [513] * B
    announce("attention", B, hq, hkv, lengths[:4])
    args, out, (qv, kpv, vpv, slots, lens) = _attention_case(torch, n, do, B, hq, hkv, lengths)
    got = _vals(out)
    for b in range(B):
        L = int(lens[b])
        ref = do.attention(qv[b], kpv[slots[b], :, :L], vpv[slots[b], :, :L], 128 ** -0.5)
        err = np.abs(got[b] - ref)
        bound = _ulp(ref) + 1e-5 * np.abs(vpv[slots[b], :, :L]).max()
        assert (err <= bound).all(), (b, (err - bound).max())
    first = bf16_bits(out).copy()
    n.attention_decode(*args)  # deterministic: the same bits again
    assert np.array_equal(bf16_bits(out), first)


def test_attention_edge_requests_get_zeros(env):
    torch, n, do, orc = env
    announce("attention edges")
    args, out, _ = _attention_case(torch, n, do, 3, 8, 2, [0, 5, -3], slots_n=4, max_len=16)
    got = _vals(out)
    assert not got[0].any() and not got[2].any() and np.isfinite(got[1]).all()
    q, kp, vp, lengths, slots, out, max_len, scale, ws = args
    bad_slots = torch.tensor([9, 0, 1], dtype=torch.int32, device="cuda")
    n.attention_decode(q, kp, vp, torch.tensor([5, 5, 5], dtype=torch.int32, device="cuda"),
                       bad_slots, out, max_len, scale, ws)
    assert not _vals(out)[0].any()


@pytest.mark.parametrize("count", [8, 311296, 13])
def test_silu_mul(env, count):
    torch, n, do, orc = env
    announce("silu_mul", count)
    g, gv = _bf16(torch, RNG.standard_normal(count) * 4)
    u, uv = _bf16(torch, RNG.standard_normal(count))
    out = torch.empty(count, dtype=torch.bfloat16, device="cuda")
    n.silu_mul(g, u, out)
    ref = do.silu_mul(gv, uv)
    err = np.abs(_vals(out) - ref)
    assert (err <= _ulp(ref) + 1e-30).all(), err.max()


def _tiny():
    from ironmule_amd.decode import DecoderConfig
    return DecoderConfig(hidden=256, layers=2, heads=4, kv_heads=2, head_dim=128,
                         intermediate=512, vocab=512, eps=1e-6, theta=1e6)


def _oracle_model(torch, do, orc, weights):
    def deq(q):
        w, s, b = (t.cpu() for t in q)
        return orc.dequant_f32(w.numpy().view(np.uint32), s.view(torch.int16).numpy().view(np.uint16),
                               b.view(torch.int16).numpy().view(np.uint16)).astype(np.float64)
    c = weights.config
    layers = [do.Layer(wq=deq(L["q"]), wk=deq(L["k"]), wv=deq(L["v"]), wo=deq(L["o"]),
                       wg=deq(L["gate"]), wu=deq(L["up"]), wd=deq(L["down"]),
                       input_norm=_vals(L["input_norm"]), post_norm=_vals(L["post_norm"]),
                       q_norm=_vals(L["q_norm"]), k_norm=_vals(L["k_norm"]))
              for L in weights.layers]
    return do.Model(layers=layers, embed=deq(weights.embed), norm=_vals(weights.norm),
                    heads=c.heads, kv_heads=c.kv_heads, eps=c.eps, theta=c.theta)


@pytest.mark.parametrize("batch", [2, 3, 6])
def test_decode_step_matches_oracle(env, batch):
    """B = 2 runs the per-kernel step with RMSNorm launches; B = 3 and 6 the step with the
    RMSNorms folded into the projections (decode.FUSED_NORM_ROWS)."""
    torch, n, do, orc = env
    from ironmule_amd.decode import FUSED_NORM_ROWS, DecodeState, decode_step, random_weights
    assert (batch >= FUSED_NORM_ROWS) == (batch >= 3)
    announce("decode step, small decoder", batch)
    cfg = _tiny()
    weights = random_weights(cfg, "cuda", seed=5)
    state = DecodeState(cfg, batch=batch, slots=max(4, batch), capacity=80, max_len=80, device="cuda")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000 + batch)
    for kp, vp in zip(state.k_pool, state.v_pool):  # a synthetic context in every slot
        kp.copy_(torch.randn(kp.shape, device="cuda", generator=gen).to(torch.bfloat16))
        vp.copy_(torch.randn(vp.shape, device="cuda", generator=gen).to(torch.bfloat16))
    keys = [_vals(kp) for kp in state.k_pool]
    values = [_vals(vp) for vp in state.v_pool]
    model = _oracle_model(torch, do, orc, weights)
    tokens, slots, positions = [5, 511, 200][:batch], [3, 0, 1][:batch], [64, 0, 79][:batch]
    if batch == 6:
        tokens, slots, positions = tokens + [7, 300, 42], slots + [2, 5, 4], positions + [1, 33, 63]
    for step in range(2):  # a second step reads the keys the first one wrote
        state.set_requests(tokens, slots, positions)
        logits = decode_step(weights, state)
        torch.cuda.synchronize()
        # the folded step's rounding points: every layer norm folded, the final one not
        folded = batch >= FUSED_NORM_ROWS
        ref = do.decode_step(model, keys, values, tokens, slots, positions, round_bf16=True,
                             fold_norms=folded, fold_first=True, fold_final=False)
        got = logits.cpu().numpy().astype(np.float64)
        rel = np.abs(got - ref).max() / np.abs(ref).max()
        print(f"[observed] small decoder batch {batch} step {step}: max|dlogit|/max|logit| = {rel:.3e}", flush=True)
        # against the oracle with the step's own rounding points the first step is at the
        # fp32 level (observed 7.1e-8 to 9.1e-8 at 2, 3 and 6 requests); the second reads the
        # keys and values the first one wrote, where a bf16 element the GPU rounded to the
        # other side of a tie moves the logits by a few 1e-5 (observed 2.7e-5 and 3.9e-5
        # folded, 7.1e-8 with RMSNorm launches)
        assert rel <= (2e-7 if step == 0 else 1e-4), (step, rel)
        for i in range(cfg.layers):
            for r in range(batch):
                kg = _vals(state.k_pool[i])[slots[r], :, positions[r]]
                kr = keys[i][slots[r], :, positions[r]]
                assert np.abs(kg - kr).max() <= 0.05 * np.abs(kr).max(), (step, i, r)
        tokens = [int(t) for t in np.argmax(got, axis=1)]
        positions = [p + 1 if p + 1 < 80 else p for p in positions]


@pytest.mark.parametrize("layers,batches", [(2, (32, 1)), (36, (32,))])
def test_decode_step_at_qwen3_4b_shapes_is_deterministic(env, layers, batches):
    """Real Qwen3-4B shapes (2 layers, and the full 36), full vocabulary head, a 512-token
    context, B = 32 (and 1): the step runs, its logits are finite, and a second call on
    the same state gives the same bits."""
    torch, n, do, orc = env
    from ironmule_amd.decode import DecodeState, DecoderConfig, decode_step, random_weights
    cfg = DecoderConfig(layers=layers)
    weights = random_weights(cfg, "cuda", seed=9)
    for batch in batches:
        announce("decode step qwen3-4b shapes", batch)
        state = DecodeState(cfg, batch=batch, slots=batch, capacity=520, max_len=520, device="cuda")
        for kp in state.k_pool + state.v_pool:
            kp.copy_(torch.randn(kp.shape, device="cuda").to(torch.bfloat16))
        state.set_requests(list(range(batch)), list(range(batch)), [512] * batch)
        first = decode_step(weights, state).clone()
        torch.cuda.synchronize()
        assert torch.isfinite(first).all()
        again = decode_step(weights, state)
        torch.cuda.synchronize()
        assert torch.equal(first, again)
        assert math.isfinite(float(first.abs().max()))
