"""The block GEMM at every token tile count (129..256 tokens per block in
32-token tiles, part-full last blocks) and every remainder of its stage
rotation, 128- and 256-row blocks, with a workspace (only K >= 1152 splits, 128-row
blocks in two chunks; other splits: test_gpu_gemm_split_tiles.py) and without;
against the oracle's F.linear."""

from __future__ import annotations

import pytest
import torch

import oracle.projections as ref
from leanstack_amd import _lib, kernels
from leanstack_amd.layout import PackedWeight
from tests.helpers import activations, assert_parity, weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,epi", [
    (256, 128, 0), (384, 256, 2), (512, 384, 1), (640, 512, 0), (256, 640, 2), (1024, 768, 1), (128, 1152, 0),
    (512, 1408, 2),
])
@pytest.mark.parametrize("m", [129, 160, 161, 192, 193, 224, 225, 256, 257, 321, 385, 513])
def test_block_gemm_tokens(gpu, m, n, k, epi):
    layout = _lib.LAYOUT_MFMA16X32_GATEUP if epi == _lib.EPI_SILU_MUL else _lib.LAYOUT_MFMA16X32
    dev = torch.device("cuda:0")
    w, x = weight(n, k, seed=n + k), activations(m, k, seed=m)
    r = activations(m, n, seed=3) if epi == _lib.EPI_RESIDUAL_ADD else None
    pw = PackedWeight.from_rowmajor(w.to(dev), layout)
    args = dict(epilogue=epi, residual=None if r is None else r.to(dev))
    y = ref.linear(x, w)
    expect = ref.silu_mul(y, n // 2) if epi == _lib.EPI_SILU_MUL else (r + y if r is not None else y)
    split = kernels.linear(x.to(dev), pw, **args)
    assert torch.equal(split, kernels.linear(x.to(dev), pw, **args))
    assert_parity(split.cpu(), expect, f"M={m} N={n} K={k}")
    whole = kernels.linear(x.to(dev), pw, workspace=None, **args)
    assert_parity(whole.cpu(), expect, f"M={m} N={n} K={k} no workspace")
