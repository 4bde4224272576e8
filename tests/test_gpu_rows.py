"""The row kernels between the projections (RMSNorm rows, q / k heads) against
the oracle's torch ops on the CPU, and the calls they stand in for against the
general torch path of the same dispatch names."""

from __future__ import annotations

import pytest
import torch

from leanstack_amd import dispatch, kernels
from leanstack_amd.geometry import QWEN3_4B as G
from leanstack_amd.layout import PackedWeight
from oracle import attention as ref_attention
from oracle import projections as ref
from tests.helpers import activations, seeded_normal, weight

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
EPS = G.rms_norm_eps


@pytest.mark.parametrize("k", [512, 2560, 4096])
@pytest.mark.parametrize("m", [1, 3, 4, 5, 129])
def test_rmsnorm_rows(gpu, m, k):
    """At most one bf16 step from the oracle (its fp32 sum of squares is added
    in another order, so r may differ in the last bits), and only where the
    value lies next to a rounding boundary."""
    x = activations(m, k, seed=m + k) * torch.tensor([0.05, 1.0, 400.0])[torch.arange(m) % 3].view(m, 1)
    x = x.to(torch.bfloat16)
    x[m // 2] = 0
    w = seeded_normal((k,), 0.2, 3) + 1
    got = dispatch.qwen_rmsnorm(x.to(DEV), w.to(DEV), EPS).cpu().float()
    expect = ref.rmsnorm(x, w, EPS).float()
    assert bool(((got - expect).abs() <= expect.abs() * 2.0 ** -7).all())
    assert float((got != expect).float().mean()) <= 0.02


@pytest.mark.parametrize("b,t,n_q,n_kv,rope", [
    (1, 1, 32, 8, "rows"), (1, 3, 32, 8, "rows"), (1, 4, 4, 1, "rows"), (1, 33, 32, 8, "rows"), (2, 5, 6, 3, "rows"),
    (2, 5, 8, 8, "batch"), (3, 1, 2, 1, "one"), (1, 6, 1, 1, "wide"),
])
def test_qk_norm_rope(gpu, b, t, n_q, n_kv, rope):
    """A head's norm may differ by one bf16 step next to a rounding boundary;
    each rotation product then moves by at most 2^-7 of its factor and each
    output by less than 2^-6 (|n0| + |n1|)."""
    d = 128
    qkv = activations(b * t, (n_q + 2 * n_kv) * d, seed=t).view(b, t, -1)
    qw, kw = seeded_normal((d,), 0.2, 5) + 1, seeded_normal((d,), 0.2, 6) + 1
    angle = torch.rand((b if rope == "batch" else 1, 1 if rope == "one" else t, d), generator=torch.Generator().manual_seed(7)) * 6
    cos, sin = angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16)
    if rope != "wide":  # "wide": rows of a wider table
        cos, sin = cos[..., : d // 2].contiguous(), sin[..., : d // 2].contiguous()
    dc, ds = cos.to(DEV)[..., : d // 2], sin.to(DEV)[..., : d // 2]
    cos, sin = cos[..., : d // 2], sin[..., : d // 2]
    q, k = kernels.qk_norm_rope(qkv.to(DEV), qw.to(DEV), kw.to(DEV), EPS, dc, ds, num_attention_heads=n_q,
                                num_key_value_heads=n_kv)
    qs, ks, _ = torch.split(qkv, (n_q * d, n_kv * d, n_kv * d), dim=-1)
    eq = ref.rmsnorm(qs.reshape(b, t, n_q, d), qw, EPS).transpose(1, 2)
    ek = ref.rmsnorm(ks.reshape(b, t, n_kv, d), kw, EPS).transpose(1, 2)
    for got, n, expect in zip((q, k), (eq, ek), ref_attention.rope(eq, ek, cos, sin)):
        a0, a1 = n.float().abs().chunk(2, dim=-1)
        bound = torch.cat((a0 + a1, a0 + a1), dim=-1) * 2.0 ** -6
        diff = (got.cpu().float() - expect.float()).abs()
        assert got.shape == expect.shape and bool((diff <= bound).all())
        assert float((diff > 0).float().mean()) <= 0.03


@pytest.mark.parametrize("t", [1, 5, 40])
def test_qkv_routes_agree(gpu, t):
    """The head kernel's route and the torch route (taken when a norm weight
    wants a gradient) give the same shapes, strides and, within the bound
    above, values; v is bit for bit the same view."""
    w = PackedWeight.from_rowmajor(weight(G.qkv_dim, G.hidden_size, seed=1).to(DEV))
    h = activations(t, G.hidden_size, seed=2).view(1, t, -1).to(DEV)
    qn, kn = (seeded_normal((128,), 0.2, s).to(DEV) + 1 for s in (3, 4))
    angle = torch.outer(torch.arange(t).float(), torch.linspace(1, 0.01, 64))
    cos, sin = angle.cos().to(torch.bfloat16)[None].to(DEV), angle.sin().to(torch.bfloat16)[None].to(DEV)
    args = (w, G.q_dim, G.kv_dim, 32, 8, 128)
    fast = dispatch._semantic_attention_qkv(h, *args, qn, kn, cos, sin, EPS)
    slow = dispatch._semantic_attention_qkv(h, *args, qn.clone().requires_grad_(), kn, cos, sin, EPS)
    assert slow[0].requires_grad and not fast[0].requires_grad
    for a, b in zip(fast, slow):
        assert a.shape == b.shape and a.stride() == b.stride()
        assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -5 * float(b.float().abs().max())
        assert float((a != b).float().mean()) <= 0.03
    assert torch.equal(fast[2], slow[2])


def test_rows_keep_the_general_path(gpu):
    """Calls outside the kernels' reach run the torch ops as before."""
    w = (seeded_normal((2560,), 0.2, 3) + 1).to(DEV)
    x = activations(4, 2560, seed=1).to(DEV)
    expect = ref.rmsnorm(x.cpu(), w.cpu(), EPS).float()
    for h, nw in ((x.float(), w.float()), (x.repeat(1, 2)[:, :2560], w), (x.t().contiguous().t(), w),
                  (x.clone().requires_grad_(), w)):
        got = dispatch.qwen_rmsnorm(h, nw, EPS)
        assert got.dtype == h.dtype and got.requires_grad == h.requires_grad
        assert float((got.detach().float().cpu() - expect).abs().max()) <= 2.0 ** -7 * float(expect.abs().max())
    assert dispatch.qwen_rmsnorm(x[:0], w, EPS).shape == (0, 2560)
    dual = torch.func.jvp(lambda v: dispatch.qwen_rmsnorm(v, w, EPS), (x,), (torch.ones_like(x),))[1]
    assert dual.shape == x.shape and bool(dual.isfinite().all())


@pytest.mark.parametrize("rows", [1, 16, 127, 128, 129, 512, 513, 700, 4096, 4097, 16384])
@pytest.mark.parametrize("n_q,n_kv", [(32, 8), (4, 4), (8, 1), (4, 2)])
def test_gqa_attention(gpu, rows, n_q, n_kv):
    """Every chunk-rule regime on the written part of a longer cache (rows past
    it hold NaN).  fp32 softmax weights sum to 1 and the output is rounded
    once: within one bf16 step of the oracle plus 2^-14 of the largest |v|
    (expf and the fp32 sums of up to 16384 weights)."""
    if rows > 4097 and n_q != 32:
        pytest.skip("one geometry at the longest cache")
    q = activations(n_q, 128, seed=rows).view(1, n_q, 1, 128)
    k = torch.full((1, n_kv, rows + 16, 128), float("nan"), dtype=torch.bfloat16)
    v = k.clone()
    k[:, :, :rows] = activations(n_kv * rows, 128, seed=2).view(1, n_kv, rows, 128)
    v[:, :, :rows] = activations(n_kv * rows, 128, seed=3).view(1, n_kv, rows, 128)
    dk, dv = k.to(DEV)[:, :, :rows], v.to(DEV)[:, :, :rows]
    scale = 128 ** -0.5
    got = dispatch._attend_row(q.to(DEV), dk, dv, scale, n_q // n_kv)
    assert got is not None and torch.equal(got, dispatch._attend_row(q.to(DEV), dk, dv, scale, n_q // n_kv))
    expect = ref_attention.sdpa_gqa(q, k[:, :, :rows], v[:, :, :rows], scale, n_q // n_kv).float().view(-1)
    diff = (got.cpu().float() - expect).abs()
    assert bool((diff <= expect.abs() * 2.0 ** -7 + 2.0 ** -14 * float(v[:, :, :rows].abs().max())).all())


def test_gqa_attention_extremes_and_routes(gpu):
    """Scores of -inf in a whole chunk and NaN rows behave as the torch ops;
    shapes the kernel does not serve take them; a captured call replays."""
    scale, rows = 128 ** -0.5, 700
    q = activations(32, 128, seed=1).abs().view(1, 32, 1, 128).to(DEV)
    k = activations(8 * rows, 128, seed=2).view(1, 8, rows, 128).to(DEV)
    v = activations(8 * rows, 128, seed=3).view(1, 8, rows, 128).to(DEV)
    k[:, 1, 128:256] = float("-inf")  # q > 0: the whole second chunk scores -inf
    k[:, 2, 300, 5] = float("nan")
    k[:, 3, 17] = float("inf")
    got = dispatch._attend_row(q, k, v, scale, 4).float()
    expect = dispatch._sdpa(q, k, v, scale, 4).view(-1).float()
    assert torch.equal(got.isnan(), expect.isnan()) and bool(got.isnan().any()) and not bool(got.isnan().all())
    assert float((got - expect).nan_to_num().abs().max()) <= 2.0 ** -6
    for bad in ((q.expand(2, -1, -1, -1), k.expand(2, -1, -1, -1), v.expand(2, -1, -1, -1), scale, 4),
                (q.expand(-1, -1, 3, -1), k, v, scale, 4), (q, k, v.clone()[..., ::2].repeat(1, 1, 1, 2)[:, :, ::1, :], scale, 2),
                (q, k.transpose(1, 2).contiguous().transpose(1, 2), v, scale, 4), (q.float(), k, v, scale, 4),
                (q.clone().requires_grad_(), k, v, scale, 4), (q, k[:, :, :0], v[:, :, :0], scale, 4)):
        assert dispatch._attend_row(*bad) is None
    k[:, 1:4] = 0.5
    expect = dispatch._attend_row(q, k, v, scale, 4)
    side = torch.cuda.Stream()  # no warm-up on it: the graph brings its own workspace
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = dispatch._attend_row(q, k, v, scale, 4)
    for _ in range(3):
        out.zero_()
        graph.replay()
        eager = dispatch._attend_row(q, k, v, scale, 4)
        torch.cuda.synchronize()
        assert torch.equal(out, expect) and torch.equal(eager, expect)
