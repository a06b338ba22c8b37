"""Host-side rules of the calls through `_native`, above all those for more than 32 rows: what
they refuse before a kernel is launched.  No GPU: meta tensors stand for the device's, and a
launch fails the test."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from ironmule_amd import _native

N, K = 64, 128


@pytest.fixture
def no_launch(monkeypatch):
    def refuse(*args):
        raise AssertionError("a kernel would be launched")

    monkeypatch.setattr(_native, "lib", lambda: SimpleNamespace(
        imq_prompt_matmul_workspace=lambda *a: 256, imq_prompt_experts_workspace=lambda *a: 256,
        imq_prompt_layer_workspace=lambda *a: 256, imq_prompt_matmul=refuse, imq_prompt_experts=refuse,
        imq_prompt_layer=refuse, imq_qmv=refuse, imq_qmv_ws=refuse, imq_qmv_workspace=lambda *a: 0,
        imq_gather_qmv=refuse))
    monkeypatch.setattr(_native, "_lib", None)
    # the check that weights are on a GPU; meta tensors stand for those
    monkeypatch.setattr(_native, "check_weights", lambda w, s, b: (int(w.shape[0]), int(w.shape[1]) * 8))
    monkeypatch.setattr(_native, "_check_stack", lambda w, s, b: (int(w.shape[0]), int(w.shape[1]), int(w.shape[2]) * 8))
    monkeypatch.setattr(_native, "_stream", lambda stream: 0)


class _OnGpu1(torch.Tensor):
    """A tensor that says it lies on GPU 1."""

    def get_device(self):
        return 1


def _on(device, t):
    return t.as_subclass(_OnGpu1) if device == "meta" else t


def _quant(device, lead=()):
    return tuple(_on(device, t) for t in _made(device, lead))


def _made(device, lead):
    return (torch.empty((*lead, N, K // 8), dtype=torch.int32, device=device),
            torch.empty((*lead, N, K // 64), dtype=torch.bfloat16, device=device),
            torch.empty((*lead, N, K // 64), dtype=torch.bfloat16, device=device))


def _move(tensors, which):
    return [torch.zeros(t.shape, dtype=t.dtype) if i == which else _on("meta", t) for i, t in enumerate(tensors)]


@pytest.mark.parametrize("which", [1, 2, 3])
def test_products_refuse_operands_of_another_device(no_launch, which):
    w, s, b, x = _move([*_quant("meta"), torch.empty((40, K), dtype=torch.bfloat16, device="meta")], which)
    with pytest.raises(ValueError, match="on cpu"):
        _native.prompt_matmul(w, s, b, x)


@pytest.mark.parametrize("which", [1, 2, 3, 4])
def test_expert_batches_refuse_operands_of_another_device(no_launch, which):
    w, s, b, x, idx = _move([*_quant("meta", (4,)), torch.empty((40, K), dtype=torch.bfloat16, device="meta"),
                             torch.empty(40, dtype=torch.int32, device="meta")], which)
    with pytest.raises(ValueError, match="on cpu"):
        _native.prompt_experts(w, s, b, x, idx)


@pytest.mark.parametrize("where", ["up", "post_norm", "k_pool", "v_pool", "h"])
def test_prompt_layers_refuse_operands_of_another_device(no_launch, where):
    projections = {name: (N, K) for name in ("q", "k", "v", "o", "gate", "up", "down")}
    config = SimpleNamespace(hidden=K, heads=1, kv_heads=1, head_dim=128, intermediate=N, eps=1e-6, theta=1e6,
                             projections=projections)
    h = _on("cpu" if where == "h" else "meta", torch.empty((40, K), device="cpu" if where == "h" else "meta"))
    if where == "h":
        with pytest.raises(ValueError, match="GPU"):
            _native.PromptLayers(config, h, 1, 64, 0)
        return
    run = object.__new__(_native.PromptLayers)
    run.config, run.h, run.first, run.pool_shape, run.nbytes = config, h, 1, (1, 1, 64, 128), 256
    run.shape, run.workspace = _native.PromptShape(), torch.empty(256, dtype=torch.uint8, device="meta")

    def made(name, *shape):
        device = "cpu" if name == where else "meta"
        return _on(device, torch.empty(shape, dtype=torch.bfloat16, device=device))

    layer = {name: _quant("cpu" if name == where else "meta") for name in projections}
    layer.update(input_norm=made("input_norm", K), post_norm=made("post_norm", K), q_norm=made("q_norm", 128),
                 k_norm=made("k_norm", 128))
    with pytest.raises(ValueError, match="on cpu"):
        run.layer(layer, made("k_pool", 1, 1, 64, 128), made("v_pool", 1, 1, 64, 128))


@pytest.mark.parametrize("rows", [1, 3])
def test_up_to_32_rows_refuse_x_of_another_device(no_launch, rows):
    w, s, b = _quant("meta")
    with pytest.raises(ValueError, match="x is on cpu"):
        _native.qmv(w, s, b, torch.zeros((rows, K), dtype=torch.bfloat16))


def test_gathered_rows_refuse_x_of_another_device(no_launch):
    w, s, b = _quant("meta", (4,))
    with pytest.raises(ValueError, match="x is on cpu"):
        _native.gather_qmv(w, s, b, torch.zeros((3, K), dtype=torch.bfloat16),
                           torch.empty(3, dtype=torch.int32, device="meta"))


def test_rows_are_taken_as_their_values_whatever_the_view():
    x = torch.randn((40, K + 8)).to(torch.bfloat16)
    for view in (x[:, :K], x[:, 3:3 + K], x[::2, :K], x[:1, :K].expand(40, K), torch._neg_view(x[:, :K].contiguous()),
                 x[:, :K].t().contiguous().t(), x[:32, :K].reshape(4, 8, K).transpose(0, 1)):
        rows, ld = _native._aligned_rows(view, K)
        assert not rows.is_neg() and rows.stride(1) == 1 and rows.data_ptr() % 16 == 0 and ld % 8 == 0 and ld >= K
        assert rows.shape[0] == 1 or rows.stride(0) == ld
        assert torch.equal(rows, view.reshape(-1, K))


def test_only_whole_aligned_expert_stacks_are_read_in_place():
    from ironmule_amd.quantized import _stack_as_stored

    def stack(e, n):
        return (torch.zeros((e, n, K // 8), dtype=torch.int32), torch.zeros((e, n, K // 64), dtype=torch.bfloat16),
                torch.zeros((e, n, K // 64), dtype=torch.bfloat16))

    assert _stack_as_stored(*stack(4, N))
    assert _stack_as_stored(*(t[1:3] for t in stack(4, N)))
    assert not _stack_as_stored(*(t[:, :N // 2] for t in stack(4, N)))
    assert not _stack_as_stored(*(t[::2] for t in stack(4, N)))
    w, s, b = stack(4, N)
    assert not _stack_as_stored(w, s.transpose(0, 1).contiguous().transpose(0, 1), b)
    off = torch.zeros(w.numel() + 1, dtype=torch.int32)[1:].view_as(w)
    assert not _stack_as_stored(off, s, b)


def test_malformed_expert_stacks_are_refused():
    w, s, b = (torch.zeros((4, N, d), dtype=t) for d, t in ((K // 8, torch.int32), (K // 64, torch.bfloat16),
                                                           (K // 64, torch.bfloat16)))
    for bad in ((w, s, b), (w[0], s, b), (w, s[:, :-1], b), (w.float(), s, b), (w, s.float(), b), (w[:, :, :-1], s, b)):
        with pytest.raises(ValueError):  # the first: not on a GPU
            _native._check_stack(*bad)
