"""Products that copy their weights straight into LDS, from the matrix and from its tiled copy, against 64 bits, whatever is left over past
whole tiles of 16 weight rows, past a block's tile and past a part of K; and the same sums in the same order, so the same bits, where the
plan is the same (one kernel reads the tiled copy alone)."""
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


def _bound(x, w):
    # 32-bit sums of k products in some order: k ulps of the sum of their sizes at the very most, of which random signs leave a few
    return 2.0 ** -24 * 16 * float((x.double().abs() @ w.double().abs().t()).max())


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
    tiled, bound = ops.tile_weight(w), _bound(x, w)
    want = x.double() @ w.double().t() + bias.double()
    for out_type, accumulate in ((torch.float32, False), (torch.float32, True), (torch.bfloat16, False)):
        got = [torch.ones((m, n), device=DEV, dtype=out_type) for _ in range(2)]
        for out, t in zip(got, (None, tiled)):
            ops.linear(x, w, bias, out, accumulate=accumulate, tiled=t)
        if _same_plan(m, n, k, accumulate=accumulate, out_bf16=out_type is torch.bfloat16):
            assert torch.equal(*got)
        new = want + 1 if accumulate else want
        rounded = 2.0 ** -8 * float(want.abs().max()) if out_type is torch.bfloat16 else 0.
        for out in got:
            assert float((out.double() - new).abs().max()) <= rounded + 2 * bound


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


# each kind of tile in parts of K, the last of them shorter, rows and weight rows past whole tiles; 64 x 64 tiles more than the CUs (fewer read
# the matrix); where the plan is not the same with the copy, "" says so
@pytest.mark.parametrize("m,n,k,kernel", [(65, 896, 4864, "tile_step_kernel<64,64>"), (203, 3584, 4672, ""), (604, 2048, 11008, ""), (1100, 1536, 8960, ""),
                                          (100, 2052, 4672, "tile_step_kernel<64,64>"), (65, 2568, 4672, "tile_step_kernel<128,128>"),
                                          (604, 5132, 4864, "tile_dma_kernel<128,256>"), (203, 3588, 8960, "tile_dma_kernel<128>"),
                                          (1101, 3588, 4672, "tile_dma_kernel<256>")])
def test_parts_of_k(m, n, k, kernel):
    from minfer_amd.kernels import ops
    x, w, bias = _operands(m, n, k)
    tiled, bound = ops.tile_weight(w), _bound(x, w)
    want, gain = x.double() @ w.double().t(), torch.rand(n, device=DEV) + 0.5
    first = []
    for t in (None, tiled):
        plan = ops.plan_linear(m, n, k, tiled=t is not None, behind=1)
        parts = ops.linear_parts(x, w, tiled=t)
        assert (parts is None) == (plan["splits"] == 1)
        if kernel:
            assert plan["kernel"] == kernel + "(split K)"
        if parts is not None:
            assert parts.shape[0] == plan["splits"]
            assert float((parts.double().sum(0) - want).abs().max()) <= bound
            first.append(parts.clone())          # (both are in the scratch that the next one takes)
    if len(first) == 2 and _same_plan(m, n, k, behind=1):
        assert torch.equal(*first)
    new = want + bias.double() + 1
    scaled = new / (new.square().mean(-1, keepdim=True) + 1e-6).sqrt() * gain.double()
    got = [torch.ones((m, n), device=DEV) for _ in range(2)]
    normed = [ops.linear_norm_out(x, w, bias, out, True, gain, 1e-6, tiled=t) for out, t in zip(got, (None, tiled))]
    for out, rows in zip(got, normed):
        assert float((out.double() - new).abs().max()) <= 2 * bound
        assert float((rows.double() - scaled).abs().max()) <= 2.0 ** -8 * float(scaled.abs().max()) + bound
    if _same_plan(m, n, k, behind=2, accumulate=True):
        assert torch.equal(*got) and torch.equal(*normed)
