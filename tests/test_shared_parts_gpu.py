"""The two ways in which the parts of a shared block of queries are added up: by the workgroup that comes last and by a kernel
behind it."""
import math

import pytest
import torch

import plain_ops
from test_kernels_gpu import DEV, close, ops, prefill_case  # noqa: F401 (`ops` is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nk,hd,window", [(4, 2, 16, 0), (14, 2, 64, 0), (5, 5, 80, 300), (16, 2, 128, 0), (4, 2, 256, 0)])
@pytest.mark.parametrize("new,start", [([300], [0]), ([700, 3, 90], [200, 0, 2500])])
@pytest.mark.parametrize("meet", [True, False])
def test_parts_of_shared_blocks(ops, monkeypatch, nh, nk, hd, window, new, start, meet):  # noqa: F811
    """Two shares and up to eight; against 64 bits, and the same bits run after run (the counters are found as they were)."""
    asked = []
    monkeypatch.setattr(ops, "prefill_parts_meet", lambda *a: (asked.append(a), meet)[1])
    q, kc, vc, table, ctx_on = prefill_case(nh, nk, hd, new, start, 31)
    scale = 1.0 / math.sqrt(hd)
    ref = torch.empty(q.shape, dtype=torch.float64)
    plain_ops.attn_prefill(q, kc, vc, table, ctx_on("cpu"), ref, nh, nk, hd, scale, window)
    args = [t.to(DEV) for t in (q, kc, vc, table)]
    outs = []
    for _ in range(3):
        outs.append(torch.empty(q.shape, dtype=torch.bfloat16, device=DEV))
        ops.attn_prefill(*args, ctx_on(DEV), outs[-1], nh, nk, hd, scale, window)
    assert len(asked) == 3 and asked[0][1] >= 2
    close(outs[0], ref, 1.5e-2, 1.5e-2)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
