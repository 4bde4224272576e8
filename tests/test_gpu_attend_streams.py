"""The single-row attention over cached rows from two streams at once: each
stream has its own workspace, so overlapping calls do not count arrivals in each
other's words."""

from __future__ import annotations

import pytest
import torch

from leanstack_amd import dispatch, kernels
from tests.helpers import activations

pytestmark = pytest.mark.gpu


def test_two_streams(gpu):
    dev, rows, scale = torch.device("cuda:0"), 3000, 128 ** -0.5
    q = [activations(32, 128, seed=s).view(1, 32, 1, 128).to(dev) for s in (1, 2)]
    k, v = (activations(8 * rows, 128, seed=s).view(1, 8, rows, 128).to(dev) for s in (3, 4))
    expect = [dispatch._attend_row(x, k, v, scale, 4) for x in q]
    streams = [torch.cuda.Stream() for _ in q]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(40):
        for i, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                got[i].append(dispatch._attend_row(q[i], k, v, scale, 4))
    torch.cuda.synchronize()
    for outs, want in zip(got, expect):
        assert all(torch.equal(o, want) for o in outs)
    used = [w for (_, stream, _), w in kernels._gqa_workspaces.items() if stream in {s.cuda_stream for s in streams}]
    assert len({w.data_ptr() for w in used}) == 2
    assert not any(bool(w[:kernels.ATTENTION_COUNTER_BYTES].any()) for w in used)
