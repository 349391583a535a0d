"""Products that copy their weights straight into LDS, from the matrix and from its tiled copy: the same sums in the same order, so the
same bits (where the plan is the same: one kernel reads the tiled copy alone, and its sums are those of test_tile_stream_gpu.py), whatever is left over past whole tiles of 16 weight rows, past a block's tile and past a part of K."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _operands(m, n, k):
    g = torch.Generator(device=DEV)
    g.manual_seed(m * 7 + n * 3 + k)
    x = torch.randn((m, k), generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn((n, k), generator=g, device=DEV).mul_(k ** -0.5).to(torch.bfloat16)
    return x, w, torch.randn(n, generator=g, device=DEV)


def _same_plan(*shape, **kw):
    from minfer_amd.kernels import ops
    plans = [ops.plan_linear(*shape, tiled=t, **kw) for t in (False, True)]
    assert plans[0] == plans[1] or plans[1]["kernel"].startswith("tile_stream_kernel")
    return plans[0] == plans[1]


# one tile row and several; the last weight row in the first, a middle and the last place of a tile of 16; one k tile of 64 and odd numbers of them
@pytest.mark.parametrize("m,n,k", [(65, 16, 64), (65, 2049, 192), (129, 4608, 896), (203, 3600, 960), (257, 24577, 64), (300, 9744, 448),
                                   (604, 2560, 2048), (700, 8224, 1088), (1030, 4093, 512), (2048, 8200, 320)])
def test_products(m, n, k):
    from minfer_amd.kernels import ops
    x, w, bias = _operands(m, n, k)
    tiled = ops.tile_weight(w)
    for out_type, accumulate in ((torch.float32, False), (torch.float32, True), (torch.bfloat16, False)):
        got = [torch.ones((m, n), device=DEV, dtype=out_type) for _ in range(2)]
        for out, t in zip(got, (None, tiled)):
            ops.linear(x, w, bias, out, accumulate=accumulate, tiled=t)
        if _same_plan(m, n, k, accumulate=accumulate, out_bf16=out_type is torch.bfloat16):
            assert torch.equal(*got)
    want = x.float() @ w.float().t() + bias
    assert float((got[1].float() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max()) + 1e-4      # (rounded to bfloat16 once)


@pytest.mark.parametrize("m,n,k", [(17, 1152, 512), (40, 22016, 2048), (64, 22016, 2048), (64, 37888, 128), (100, 37888, 192), (203, 9728, 896),
                                   (604, 17920, 320)])
def test_swiglu(m, n, k):
    from minfer_amd.kernels import ops
    x, w, _ = _operands(m, n, k)
    tiled = ops.tile_weight(w)
    plans = [ops.plan_linear(m, n, k, swiglu=True, tiled=t) for t in (False, True)]
    got = [torch.empty((m, n // 2), device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    for out, t in zip(got, (None, tiled)):
        ops.linear_swiglu(x, w, out, tiled=t)
    if plans[0] == plans[1]:
        assert torch.equal(*got)
    gate, up = (x.float() @ w.float().t()).view(m, -1, 2, 32).unbind(2)
    want = (torch.nn.functional.silu(gate) * up).reshape(m, n // 2)
    for out in got:
        assert float((out.float() - want).abs().max()) <= 2.0 ** -7 * float(want.abs().max())


@pytest.mark.parametrize("m,n,k", [(65, 896, 4864), (203, 3584, 4672), (604, 2048, 11008), (1100, 1536, 8960)])
def test_parts_of_k(m, n, k):
    from minfer_amd.kernels import ops
    x, w, bias = _operands(m, n, k)
    tiled, gain = ops.tile_weight(w), torch.rand(n, device=DEV) + 0.5
    parts = [ops.linear_parts(x, w, tiled=t) for t in (None, tiled)]
    if parts[0] is not None and _same_plan(m, n, k, behind=1):
        first = parts[0].clone()                 # (both are in the scratch that the next one takes)
        assert torch.equal(first, ops.linear_parts(x, w, tiled=tiled))
        assert torch.equal(first, ops.linear_parts(x, w))
    got = [torch.ones((m, n), device=DEV) for _ in range(2)]
    normed = [ops.linear_norm_out(x, w, bias, out, True, gain, 1e-6, tiled=t) for out, t in zip(got, (None, tiled))]
    if _same_plan(m, n, k, behind=2, accumulate=True):
        assert normed[0] is not None and torch.equal(*got) and torch.equal(*normed)
