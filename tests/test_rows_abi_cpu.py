"""The row kernels' C entry points (lsk_rmsnorm_bf16, lsk_qk_norm_rope_bf16,
lsk_gqa_attention_bf16) refuse what their kernels do not take before anything
touches the device."""

from __future__ import annotations

import pytest

from leanstack_amd import _lib

FAKE = 0x10000  # aligned, never dereferenced
INVALID, WORKSPACE = -1, -4


@pytest.mark.parametrize("bad", [
    dict(m=0), dict(k=0), dict(k=256), dict(k=2576), dict(k=4608), dict(ldx=2552), dict(ldx=2564), dict(x=0),
    dict(x=FAKE + 8), dict(w=0), dict(w=FAKE + 2), dict(y=0), dict(y=FAKE + 8), dict(eps=-1.0),
    dict(eps=float("nan")), dict(eps=float("inf")),
])
def test_rmsnorm_rejects_before_launch(bad):
    a = dict(x=FAKE, m=4, k=2560, ldx=2560, w=FAKE, eps=1e-6, y=FAKE) | bad
    assert _lib.load().lsk_rmsnorm_bf16(a["x"], a["m"], a["k"], a["ldx"], a["w"], a["eps"], a["y"], None) == INVALID
    assert _lib.load().lsk_last_error()


@pytest.mark.parametrize("bad", [
    dict(b=0), dict(t=0), dict(b=1 << 16, t=1 << 16), dict(d=64), dict(n_q=0), dict(n_kv=0), dict(n_q=4097),
    dict(ld=5112), dict(ld=5124), dict(rb=-8), dict(rr=4), dict(qkv=0), dict(qkv=FAKE + 8), dict(qw=0),
    dict(kw=FAKE + 2), dict(cos=0), dict(sin=FAKE + 4), dict(q=0), dict(k=FAKE + 8), dict(eps=-1.0),
])
def test_qk_norm_rope_rejects_before_launch(bad):
    a = dict(qkv=FAKE, b=1, t=4, ld=6144, n_q=32, n_kv=8, d=128, qw=FAKE, kw=FAKE, eps=1e-6, cos=FAKE, sin=FAKE,
             rb=0, rr=64, q=FAKE, k=FAKE) | bad
    status = _lib.load().lsk_qk_norm_rope_bf16(a["qkv"], a["b"], a["t"], a["ld"], a["n_q"], a["n_kv"], a["d"], a["qw"],
                                               a["kw"], a["eps"], a["cos"], a["sin"], a["rb"], a["rr"], a["q"],
                                               a["k"], None)
    assert status == INVALID
    assert _lib.load().lsk_last_error()


@pytest.mark.parametrize("bad,code", [
    (dict(d=64), INVALID), (dict(n_q=24), INVALID), (dict(n_kv=65, n_q=65), INVALID), (dict(rows=0), INVALID),
    (dict(rows=16385), INVALID), (dict(stride=700 * 128 - 8), INVALID), (dict(stride=700 * 128 + 4), INVALID),
    (dict(q=0), INVALID), (dict(k=FAKE + 8), INVALID), (dict(v=0), INVALID), (dict(out=0), INVALID),
    (dict(scale=float("nan")), INVALID), (dict(ws=None), WORKSPACE), (dict(ws_bytes=1024), WORKSPACE),
    (dict(ws=FAKE + 64), WORKSPACE),
])
def test_gqa_attention_rejects_before_launch(bad, code):
    lib = _lib.load()
    a = dict(q=FAKE, n_q=32, n_kv=8, d=128, k=FAKE, v=FAKE, stride=700 * 128, rows=700, scale=0.088, out=FAKE, ws=FAKE,
             ws_bytes=lib.lsk_attention_workspace_bytes(32, 8, 128, 700)) | bad
    status = lib.lsk_gqa_attention_bf16(a["q"], a["n_q"], a["n_kv"], a["d"], a["k"], a["v"], a["stride"], a["rows"],
                                        a["scale"], a["out"], a["ws"], a["ws_bytes"], None)
    assert status == code
    assert lib.lsk_last_error()
