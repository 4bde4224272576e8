"""The MLP names at 9..16 rows: every norm weight form and surrounding that up
to 8 rows take, against the oracle."""

from __future__ import annotations

import pytest
import torch

import oracle.projections as ref
from leanstack_amd import _lib, dispatch
from leanstack_amd.geometry import QWEN3_4B as G
from leanstack_amd.layout import PackedWeight
from tests.helpers import activations, assert_parity, seeded_normal, weight

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
EPS = G.rms_norm_eps
K = G.hidden_size


def _mlp(rows: int, inter: int):
    """A gate_up / down pair over `rows` rows, and the oracle's result."""
    wgu, wd = weight(2 * inter, K, seed=inter), weight(K, inter, seed=inter + 1)
    h, nw = activations(rows, K, seed=rows), seeded_normal((K,), 0.2, 3) + 1
    expect = h + ref.linear(ref.silu_mul(ref.linear(ref.rmsnorm(h, nw, EPS), wgu), inter), wd)
    gu = PackedWeight.from_rowmajor(wgu.to(DEV), _lib.LAYOUT_MFMA16X32_GATEUP)
    down = PackedWeight.from_rowmajor(wd.to(DEV))
    return h.to(DEV).view(1, rows, K), nw.to(DEV), gu, down, expect


@pytest.mark.parametrize("rows", [8, 9, 12, 16])
def test_norm_weight_forms(gpu, rows):
    """A [1, K] norm weight, a strided one, and autocast around the call."""
    h, nw, gu, down, expect = _mlp(rows, 320)
    plain = dispatch._semantic_mlp_epilogue(h, nw, gu, 320, down, EPS)
    assert_parity(plain[0].cpu(), expect, f"rows={rows}")
    assert_parity(dispatch._semantic_mlp_epilogue(h, nw.view(1, K), gu, 320, down, EPS)[0].cpu(), expect, "[1, K]")
    strided = torch.stack((nw, nw), 1)[:, 0]
    assert_parity(dispatch._semantic_mlp_epilogue(h, strided, gu, 320, down, EPS)[0].cpu(), expect, "strided")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert_parity(dispatch._semantic_mlp_epilogue(h, nw, gu, 320, down, EPS)[0].cpu(), expect, "autocast")
    with pytest.raises(ValueError, match="norm_weight"):
        dispatch._semantic_mlp_epilogue(h, nw.float(), gu, 320, down, EPS)


@pytest.mark.parametrize("rows", [9, 12, 16])
@pytest.mark.parametrize("inter", [1216, 4096, 4128, G.intermediate_size])
def test_mlp_names(gpu, rows, inter):
    """Both routes on either side of the width where they meet, through both
    MLP names (o_proj in front: an identity o_proj adds the attention rows)."""
    h, nw, gu, down, expect = _mlp(rows, inter)
    assert_parity(dispatch._semantic_mlp_epilogue(h, nw, gu, inter, down, EPS)[0].cpu(), expect, f"{rows} x {inter}")
    eye = PackedWeight.from_rowmajor(torch.eye(K, dtype=torch.bfloat16, device=DEV))
    out = dispatch._semantic_post_attention_mlp(h, torch.zeros_like(h), eye, nw, gu, inter, down, EPS)
    assert_parity(out[0].cpu(), expect, f"post attention {rows} x {inter}")
