"""`tile_stream_kernel`: products of more than 64 rows whose weights go from the tiled copy straight into MFMA operands, against 64 bits."""
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


# tiles of 96 and of 128 rows; one k tile and every number past whole rounds of four; weight rows past tiles of 16 and of 128, not in fours, below 16
@pytest.mark.parametrize("variant", [26, 28])
@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (65, 9, 128), (96, 128, 192), (97, 129, 256), (128, 1150, 320), (129, 2052, 448), (203, 257, 1088),
                                   (300, 1001, 2048)])
def test_whole(variant, m, n, k):
    from minfer_amd.kernels import ops
    x, w, bias = _operands(m, n, k)
    tiled, bound = ops.tile_weight(w), _bound(x, w)
    want = x.double() @ w.double().t() + bias.double()
    out = torch.full((m, n), 0.5, device=DEV)
    ops.linear(x, w, bias, out, variant=variant, tiled=tiled)
    assert float((out.double() - want).abs().max()) <= bound
    ops.linear(x, w, bias, out, accumulate=True, variant=variant, tiled=tiled)
    assert float((out.double() - 2 * want).abs().max()) <= 3 * bound
    half = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
    ops.linear(x, w, bias, half, variant=variant, tiled=tiled)
    assert float((half.double() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max()) + bound
    ops.linear(x, w, bias, half, variant=variant, tiled=tiled, relu2=True)
    assert float((half.double() - want.clamp_min(0).square()).abs().max()) <= 2.0 ** -7 * float(want.square().max())
    both = torch.cat([bias, torch.tensor([0.8, 0.5], device=DEV)])
    ops.linear(x, w, both, half, variant=variant, tiled=tiled, xielu=True)
    act = torch.where(want > 0, 0.8 * want.square() + 0.5 * want, 0.5 * (torch.expm1(want) - want) + 0.5 * want)
    assert float((half.double() - act).abs().max()) <= 2.0 ** -7 * float(act.abs().max())


def test_refused():
    from minfer_amd.kernels import ops
    x, w, _ = _operands(100, 128, 128)
    out = torch.empty((100, 128), device=DEV)
    for kw in (dict(variant=26), dict(variant=27, tiled=ops.tile_weight(w))):      # no tiled copy; no such tile
        with pytest.raises(ops.KernelError):
            ops.linear(x, w, None, out, **kw)
    with pytest.raises(ops.KernelError):                                           # k not in 64s
        ops.linear(x[:, :96].contiguous(), w[:, :96].contiguous(), None, out, variant=26, tiled=ops.tile_weight(w[:, :96].contiguous()))


# the plan's own choice: parts of K in front of the rotation and of the norm, and whole; a last part that is shorter, rows past whole tiles
@pytest.mark.parametrize("m,n,k,behind", [(470, 2560, 2048, 1), (300, 4608, 3584, 1), (150, 4608, 3584, 1), (257, 1536, 8960, 2), (203, 3584, 3584, 2),
                                          (150, 2048, 11008, 2), (1000, 1024, 4096, 2), (300, 8192, 4096, 0), (520, 6144, 3584, 0), (2651, 768, 3072, 2),
                                          (2994, 1024, 4096, 0)])
def test_planned(m, n, k, behind):
    from minfer_amd.kernels import ops
    x, w, bias = _operands(m, n, k)
    tiled, bound = ops.tile_weight(w), _bound(x, w)
    want = x.double() @ w.double().t()
    plan = ops.plan_linear(m, n, k, tiled=True, behind=behind, accumulate=behind == 2)
    assert plan["kernel"].startswith("tile_stream_kernel"), plan
    if behind == 1:
        parts = ops.linear_parts(x, w, tiled=tiled)
        assert parts.shape[0] == plan["splits"] > 1
        assert float((parts.double().sum(0) - want).abs().max()) <= bound
        return
    out = torch.ones((m, n), device=DEV)
    if behind == 2:
        gain = torch.rand(n, device=DEV) + 0.5
        normed = ops.linear_norm_out(x, w, bias, out, True, gain, 1e-6, tiled=tiled)
        new = want + bias.double() + 1
        scaled = new / (new.square().mean(-1, keepdim=True) + 1e-6).sqrt() * gain.double()
        assert float((normed.double() - scaled).abs().max()) <= 2.0 ** -8 * float(scaled.abs().max()) + bound
    else:
        ops.linear(x, w, bias, out, accumulate=True, tiled=tiled)
        new = want + bias.double() + 1
    assert float((out.double() - new).abs().max()) <= 2 * bound
