"""The K split of the block GEMM on blocks of fewer than eight token tiles: the
chunks share 5, 6, 7 (128-row blocks) or 10, 12, 14 (256-row) accumulator tiles
unevenly, some none, also beside blocks that run whole.  The plan is asserted, so
that a case cannot become unsplit unseen; against F.linear in fp32 of the same
bf16 values."""

from __future__ import annotations

import ctypes

import pytest
import torch

import oracle.projections as ref
from leanstack_amd import _lib, kernels
from leanstack_amd.layout import PackedWeight
from tests.helpers import activations, assert_parity, weight

pytestmark = pytest.mark.gpu

# (M, N, K, epilogue) and the plan on 256 CUs: block rows, blocks, split blocks, chunks
CASES = {
    "128x5_s8": (150, 2560, 4096, _lib.EPI_RESIDUAL_ADD, [128, 20, 20, 8]),
    "128x5_s16": (150, 1024, 8192, _lib.EPI_NONE, [128, 8, 8, 16]),
    "128x5_s4": (301, 2560, 9728, _lib.EPI_RESIDUAL_ADD, [128, 40, 40, 4]),
    "128x6_s8": (180, 2560, 4096, _lib.EPI_NONE, [128, 20, 20, 8]),
    "128x6_s2": (560, 4096, 4096, _lib.EPI_SILU_MUL, [128, 96, 96, 2]),
    "128x7_s2": (1300, 2560, 9728, _lib.EPI_RESIDUAL_ADD, [128, 120, 120, 2]),
    "256x5_s4": (300, 34304, 2048, _lib.EPI_SILU_MUL, [256, 268, 12, 4]),
    "256x6_s4": (560, 22528, 2560, _lib.EPI_NONE, [256, 264, 8, 4]),
    "256x7_s4": (800, 19456, 2560, _lib.EPI_SILU_MUL, [256, 304, 48, 4]),
    "256x7_s2": (1100, 19456, 2560, _lib.EPI_SILU_MUL, [256, 380, 124, 2]),
    "256x7_s3": (1550, 2560, 4096, _lib.EPI_RESIDUAL_ADD, [256, 70, 70, 3]),
    "256x7_s3_deep": (1550, 2560, 9728, _lib.EPI_RESIDUAL_ADD, [256, 70, 70, 3]),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_uneven_split(gpu, case):
    m, n, k, epi, expected = CASES[case]
    lib, dev = _lib.load(), torch.device("cuda:0")
    plan = (ctypes.c_int * 4)()
    assert lib.lsk_linear_plan(m, n, k, lib.lsk_workspace_bytes(_lib.OP_LINEAR, m, n, k), plan) == _lib.OK
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert list(plan) == expected
    layout = _lib.LAYOUT_MFMA16X32_GATEUP if epi == _lib.EPI_SILU_MUL else _lib.LAYOUT_MFMA16X32
    w, x = weight(n, k, seed=n + k).to(dev), activations(m, k, seed=m).to(dev)
    r = activations(m, n, seed=3).to(dev) if epi == _lib.EPI_RESIDUAL_ADD else None
    pw = PackedWeight.from_rowmajor(w, layout)
    ws = kernels.prefill_workspace(dev, m, n, k)
    y = kernels.linear(x, pw, epilogue=epi, residual=r, workspace=ws)
    assert torch.equal(y, kernels.linear(x, pw, epilogue=epi, residual=r, workspace=ws))
    assert kernels.linear_error(ws) == 0
    assert int(ws.view(torch.int32)[64:2048].abs().sum()) == 0  # arrival and departure words zero again
    yl = torch.nn.functional.linear(x.float(), w.float()).to(torch.bfloat16).cpu()
    expect = ref.silu_mul(yl, n // 2) if epi == _lib.EPI_SILU_MUL else (r.cpu() + yl if r is not None else yl)
    assert_parity(y.cpu(), expect, case)
    whole = kernels.linear(x, pw, epilogue=epi, residual=r, workspace=None)
    assert_parity(whole.cpu(), expect, f"{case} no workspace")
