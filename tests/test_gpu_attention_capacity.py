"""Short contexts in large caches with the position on the device: the code for
the context's own chunk size runs, one of up to four in the launch.  Outputs and
caches are bit for bit those of the host-position entry point, whose code the
host picks."""

from __future__ import annotations

import pytest
import torch

from leanstack_amd import _lib, kernels

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
D = 128
# the first and last row counts of each chunk size: one chunk, 64-row chunks, 128, 256, 384 and 512 rows
POSITIONS = (0, 15, 16, 127, 128, 511, 512, 1087, 4095, 4096, 8191, 8192, 12287, 12288, 16383)


@pytest.mark.parametrize("n_q,n_kv", [(4, 4), (4, 2), (8, 2), (16, 2)])
@pytest.mark.parametrize("s_max", [4096, 8192, 12288, 16384])
def test_device_position_in_a_large_cache(gpu, s_max, n_q, n_kv):
    gen = torch.Generator(device=DEV).manual_seed(s_max + n_q)

    def normal(*shape, mean=0.0, std=1.0):
        return torch.empty(shape, device=DEV, dtype=torch.bfloat16).normal_(mean, std, generator=gen)

    qkv, qn, kn = normal((n_q + 2 * n_kv) * D), normal(D, mean=1.0, std=0.2), normal(D, mean=1.0, std=0.2)
    cos, sin = normal(s_max, D // 2), normal(s_max, D // 2)
    caches = [normal(n_kv, s_max, D), normal(n_kv, s_max, D)]
    host, device = [c.clone() for c in caches], [c.clone() for c in caches]
    at = torch.zeros(1, dtype=torch.int32, device=DEV)
    nbytes = _lib.load().lsk_attention_workspace_bytes(n_q, n_kv, D, s_max)
    ws = [torch.zeros(nbytes, dtype=torch.uint8, device=DEV) for _ in range(2)]
    heads = dict(num_attention_heads=n_q, num_key_value_heads=n_kv)
    for pos in (p for p in POSITIONS if p < s_max):
        at.fill_(pos)
        a = kernels.decode_attention(qkv, qn, kn, 1e-6, cos[pos], sin[pos], *host, pos, D ** -0.5, workspace=ws[0],
                                     **heads)
        b = kernels.decode_attention(qkv, qn, kn, 1e-6, cos, sin, *device, at, D ** -0.5, workspace=ws[1], **heads)
        assert bool(a.isfinite().all()) and torch.equal(a, b), f"{pos} of {s_max}"
        assert all(torch.equal(x, y) for x, y in zip(host, device)), f"caches at {pos} of {s_max}"
    assert not any(bool(w[:256].any()) for w in ws)
