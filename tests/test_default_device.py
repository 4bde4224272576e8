"""A default device is no reason to leave the row kernels: it is a torch
function mode that changes no op; any other mode is."""

from __future__ import annotations

import pytest
import torch
from torch.overrides import TorchFunctionMode

from leanstack_amd import dispatch, kernels
from leanstack_amd.geometry import QWEN3_4B as G
from leanstack_amd.layout import PackedWeight
from tests.helpers import activations, seeded_normal, weight


class _Recorder(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(func)
        return func(*args, **(kwargs or {}))


def test_modes():
    assert not dispatch._follows_ops()
    with torch.device("cpu"):
        assert not dispatch._follows_ops()
        with torch.device("meta"):
            assert not dispatch._follows_ops()
            with _Recorder():
                assert dispatch._follows_ops()
    torch.set_default_device("cpu")
    try:
        assert not dispatch._follows_ops()
    finally:
        torch.set_default_device(None)


@pytest.fixture
def taken(monkeypatch):
    names = []
    for name in ("_rmsnorm_rows", "_qk_norm_rope", "_gqa_attention"):
        monkeypatch.setattr(kernels, name, lambda *a, f=getattr(kernels, name), n=name: names.append(n) or f(*a))
    return names


@pytest.mark.gpu
@pytest.mark.parametrize("default", [None, "cuda", "cpu"])
def test_kernels_taken_under_a_default_device(gpu, taken, default):
    dev = torch.device("cuda:0")
    x = activations(3, G.hidden_size, seed=1).view(1, 3, -1).to(dev)
    nw = (seeded_normal((G.hidden_size,), 0.2, 2) + 1).to(dev)
    hw = (seeded_normal((128,), 0.2, 3) + 1).to(dev)
    w = PackedWeight.from_rowmajor(weight(G.qkv_dim, G.hidden_size, seed=4).to(dev))
    cos, sin = (f(torch.arange(3 * 64).view(1, 3, 64) / 64).to(torch.bfloat16).to(dev) for f in (torch.cos, torch.sin))
    kv = activations(8 * 200, 128, seed=5).view(1, 8, 200, 128).to(dev)

    def call():
        h = dispatch.qwen_rmsnorm(x, nw, G.rms_norm_eps)
        q, k, v = dispatch._semantic_attention_qkv(h, w, G.q_dim, G.kv_dim, 32, 8, 128, hw, hw, cos, sin,
                                                   G.rms_norm_eps)
        attn = dispatch._attend_row(q[:, :, :1].contiguous(), kv, kv, 128 ** -0.5, 4)
        return h, q, k, v, attn

    expect = call()
    taken.clear()
    torch.set_default_device(default)
    try:
        got = call()
    finally:
        torch.set_default_device(None)
    assert taken == ["_rmsnorm_rows", "_qk_norm_rope", "_gqa_attention"]
    assert all(torch.equal(a, b) and a.device == dev for a, b in zip(got, expect))


@pytest.mark.gpu
def test_another_mode_sees_the_ops(gpu, taken):
    x = activations(3, 2560, seed=1).to("cuda:0")
    w = torch.ones(2560, dtype=torch.bfloat16, device="cuda:0")
    with _Recorder() as mode:
        dispatch.qwen_rmsnorm(x, w, 1e-6)
    assert not taken and torch.nn.functional.rms_norm in mode.seen
