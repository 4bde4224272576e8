"""SiLU*up projections of 9..128 rows around the widths where the units per
workgroup change (one round of fives, three rounds of twos, fours and fives
beyond) and on both sides of the routes' limits in N and K; against the
oracle's F.linear."""

from __future__ import annotations

import pytest
import torch

import oracle.projections as ref
from leanstack_amd import _lib, kernels
from leanstack_amd.layout import PackedWeight
from tests.helpers import activations, assert_parity, weight

pytestmark = pytest.mark.gpu

CASES = [(m, n, k) for m in (9, 16) for n, k in ((16384, 992), (16384, 1024), (16416, 1056), (20512, 1024))]
CASES += [(m, n, k) for m in (17, 33, 64, 65, 128) for n, k in (
    (20480, 96), (20512, 32), (20512, 160), (24576, 64), (24608, 96), (32800, 64), (36896, 160), (41024, 64))]
CASES += [(m, n, k) for m in (65, 97) for n, k in (
    (8192, 256), (9728, 448), (12288, 512), (20480, 768), (24576, 2048), (24704, 2048), (40960, 1984), (41088, 64))]


@pytest.mark.parametrize("m,n,k", CASES)
def test_skinny_rounds(gpu, m, n, k):
    dev = torch.device("cuda:0")
    w, x = weight(n, k, seed=n + k), activations(m, k, seed=m)
    pw = PackedWeight.from_rowmajor(w.to(dev), _lib.LAYOUT_MFMA16X32_GATEUP)
    got = kernels.linear(x.to(dev), pw, epilogue=_lib.EPI_SILU_MUL)
    assert torch.equal(got, kernels.linear(x.to(dev), pw, epilogue=_lib.EPI_SILU_MUL))
    # fp32 products of the same bf16 values on the device; the oracle's chain of roundings after them
    y = torch.nn.functional.linear(x.to(dev).float(), w.to(dev).float()).to(torch.bfloat16).cpu()
    assert_parity(got.cpu(), ref.silu_mul(y, n // 2), f"M={m} N={n} K={k}")
