"""The 17..128-row kernel at the sizes where its steps and units can go wrong:
K of one k-tile, odd k-tile counts (a half last step), fewer steps than waves
and than ring slots, single and odd row-block counts, SiLU*up units in a
part-full last workgroup; against the oracle's F.linear."""

from __future__ import annotations

import pytest
import torch

import oracle.projections as ref
from leanstack_amd import _lib, kernels
from leanstack_amd.layout import PackedWeight
from tests.helpers import activations, assert_parity, weight

pytestmark = pytest.mark.gpu

CASES = [  # (N, K, epilogue); the last four take five units per workgroup
    (16, 32, 0), (48, 64, 0), (2560, 96, 2), (16, 2560, 2), (80, 544, 0), (4096, 1056, 0), (32, 32, 1), (96, 160, 1),
    (2592, 608, 1), (16416, 96, 1), (19456, 288, 1), (20512, 64, 1),
    (16416, 800, 1),
]


@pytest.mark.parametrize("m,n,k,epi", [(m, *c) for c in CASES for m in (17, 33, 64, 81, 128)]
                         + [(m, n, k, 1) for m in (9, 16) for n, k in ((16384, 96), (16416, 64), (19456, 2560))])
def test_skinny_edges(gpu, m, n, k, epi):
    layout = _lib.LAYOUT_MFMA16X32_GATEUP if epi == _lib.EPI_SILU_MUL else _lib.LAYOUT_MFMA16X32
    dev = torch.device("cuda:0")
    w, x = weight(n, k, seed=n + k), activations(m, k, seed=m)
    r = activations(m, n, seed=3) if epi == _lib.EPI_RESIDUAL_ADD else None
    pw = PackedWeight.from_rowmajor(w.to(dev), layout)
    args = dict(epilogue=epi, residual=None if r is None else r.to(dev))
    auto = kernels.linear(x.to(dev), pw, **args)
    plain = kernels.linear(x.to(dev), pw, workspace=None, **args)
    assert torch.equal(auto, kernels.linear(x.to(dev), pw, **args))
    y = ref.linear(x, w)
    expect = ref.silu_mul(y, n // 2) if epi == _lib.EPI_SILU_MUL else (r + y if r is not None else y)
    assert_parity(auto.cpu(), expect, f"M={m} N={n} K={k}")
    assert_parity(plain.cpu(), expect, f"M={m} N={n} K={k} no workspace")
