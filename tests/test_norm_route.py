"""The RMSNorm in front of gate_up: which of the two forms (inside the
projection kernel, or a norm of its own) a call takes, with the kernels
replaced by recorders."""

from __future__ import annotations

import pytest
import torch

from leanstack_amd import _lib, dispatch, kernels
from leanstack_amd.layout import PackedWeight


@pytest.fixture
def calls(monkeypatch):
    seen = []
    monkeypatch.setattr(kernels, "rmsnorm_linear", lambda *a, **k: seen.append("fused"))
    monkeypatch.setattr(kernels, "linear", lambda *a, **k: seen.append("linear"))
    return seen


def _gate_up(n: int, k: int) -> PackedWeight:
    return PackedWeight(torch.empty(n * k, dtype=torch.bfloat16, device="meta"), n, k, _lib.LAYOUT_MFMA16X32_GATEUP)


@pytest.mark.parametrize("rows", [1, 8, 9, 12, 16])
@pytest.mark.parametrize("shape", [(2560,), (1, 2560)])
def test_rows_without_the_norm_kernel_stay_fused(calls, rows, shape):
    """Up to 16 rows a call that the row kernel does not serve (here: CPU
    tensors) goes to rmsnorm_linear, which flattens the norm weight."""
    hidden = torch.ones(1, rows, 2560, dtype=torch.bfloat16)
    dispatch._norm_gate_up(hidden, torch.ones(shape, dtype=torch.bfloat16), 1e-6, _gate_up(19456, 2560))
    assert calls == ["fused"]


def test_more_rows_take_a_norm_of_their_own(calls):
    hidden = torch.ones(1, 17, 2560, dtype=torch.bfloat16)
    dispatch._norm_gate_up(hidden, torch.ones(2560, dtype=torch.bfloat16), 1e-6, _gate_up(19456, 2560))
    assert calls == ["linear"]


@pytest.mark.parametrize("rows,n,k,route", [
    (8, 19456, 2560, ["fused"]), (9, 2432, 2560, ["fused"]), (16, 8192, 2560, ["fused"]),
    (9, 8224, 2560, ["norm", "linear"]), (16, 19456, 2560, ["norm", "linear"]), (12, 2048, 512, ["fused"]),
    (12, 2048, 1024, ["norm", "linear"]), (8, 2048, 1024, ["fused"]), (17, 2432, 2560, ["norm", "linear"]),
])
def test_route_by_width(calls, monkeypatch, rows, n, k, route):
    """9..16 rows that the row kernel serves: fused where the fused kernel was
    measured faster."""
    monkeypatch.setattr(dispatch, "_plain_eager", lambda *tensors: True)
    monkeypatch.setattr(kernels, "_rmsnorm_rows", lambda *a: calls.append("norm"))
    hidden = torch.ones(rows, k, dtype=torch.bfloat16)
    dispatch._norm_gate_up(hidden, torch.ones(k, dtype=torch.bfloat16), 1e-6, _gate_up(n, k))
    assert calls == route
