"""Products of 17 to 64 rows over the whole of K in one kernel, a norm folded in on either side, against products in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one and two tiles of rows and of weight rows a block; K of fewer steps than waves, a last wave without one, of one load of the
# ring, of a round and a rest, of whole rounds; weight rows that fill no block
@pytest.mark.parametrize("m,n,k", [(17, 1152, 896), (32, 896, 896), (33, 2048, 1536), (64, 2048, 2048), (64, 2560, 2048), (48, 2576, 2048),
                                   (64, 912, 896), (20, 896, 4864), (61, 1008, 4864), (17, 512, 64), (40, 1008, 96), (31, 528, 320),
                                   (64, 8000, 288)])
def test_both_sides(m, n, k):
    from minfer_amd.kernels import ops
    parts = ops.norm_sum_parts(n, m, k)
    assert parts > ops.norm_sum_parts(n, m), "one kernel takes these"
    for kw in (dict(norm_out=True), dict(scale_in=True), dict(scale_in=True, norm_out=True)):
        assert ops.plan_linear(m, n, k, accumulate=True, **kw)["kernel"] == "whole_kernel"
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV)
    w = (torch.randn((n, k), generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV)
    b, g, base = (torch.randn(s, generator=gen).to(DEV) for s in ((n,), (n,), (m, n)))
    tiled = ops.tile_weight(w)
    product = x.double() @ w.double().t()
    tol = 4 * 2.0 ** -20 * k ** 0.5                                      # 32-bit sums of exact products of size one and below

    def fused(out, tiled=tiled, **kw):
        assert ops.linear_fused(x, w, out=out, tiled=tiled, **kw)
        return out
    left = []
    for copy in (tiled, tiled, None):                                    # twice, and without the tiled copy: the same bits
        xg = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        sums = torch.full((m, parts), float("nan"), device=DEV)
        out = fused(base.clone(), tiled=copy, bias=b, accumulate=True, norm_out=(g, xg, sums))
        left.append((out, xg, sums))
    assert all(torch.equal(p[0], q) for p in zip(*left) for q in p[1:])
    assert (out - (product + b.double() + base.double())).abs().max() <= tol
    assert torch.equal(xg, (out * g).to(torch.bfloat16))
    squares = (out.double() ** 2).sum(-1)
    assert ((sums.double().sum(-1) - squares).abs() <= 1e-5 * squares).all()
    for n_parts in (1, 7, 100, 300):                                     # the rows' sums of squares in few parts and in many
        s = torch.rand((m, n_parts), generator=gen).to(DEV)
        scale = 1.0 / (s.double().sum(-1, keepdim=True) / k + 1e-6).sqrt()
        out = fused(torch.full((m, n), float("nan"), device=DEV), bias=b, scale_in=(s, 1e-6))
        want = product * scale + b.double()
        assert ((out - want).abs() <= tol * scale + 1e-6 * want.abs()).all()
        xg, sums = torch.empty((m, n), dtype=torch.bfloat16, device=DEV), torch.empty((m, parts), device=DEV)
        out = fused(base.clone(), bias=None, accumulate=True, scale_in=(s, 1e-6), norm_out=(g, xg, sums))
        assert ((out - (product * scale + base.double())).abs() <= tol * scale + 1e-6 * want.abs() + 1e-6).all()


# the products that read such rows next: 64 x 64 tiles, the panel kernels, the K-split kernels, each with parts for one pass of
# its lanes, for several, and for a rest
@pytest.mark.parametrize("m,nf,k", [(33, 4864, 896), (64, 11008, 2048), (40, 18944, 512), (20, 18944, 256), (18, 512, 2048)])
@pytest.mark.parametrize("parts", [3, 5, 64, 83, 130, 256, 261])
def test_readers_of_many_parts(m, nf, k, parts):
    from minfer_amd.kernels import ops
    gen = torch.Generator().manual_seed(m + nf + parts)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV)
    wg, wu = ((torch.randn((nf, k), generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV) for _ in range(2))
    s = torch.rand((m, parts), generator=gen).to(DEV)
    scale = 1.0 / (s.double().sum(-1, keepdim=True) / k + 1e-6).sqrt()
    gate, up = x.double() @ wg.double().t() * scale, x.double() @ wu.double().t() * scale
    out = torch.empty((m, nf), dtype=torch.bfloat16, device=DEV)
    w = ops.interleave_gate_up(wg, wu)
    assert ops.linear_fused(x, w, None, out, swiglu=True, scale_in=(s, 1e-6), tiled=ops.tile_weight(w) if k == 2048 else None)
    want = gate / (1 + torch.exp(-gate)) * up
    assert ((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + 1e-4 * scale ** 2).all()


# places for the sums over runs of 256 columns alone, at shapes that the one kernel takes otherwise: the kernels that cut K, whose stream
# is that of the plain product bit for bit
@pytest.mark.parametrize("m,n,k", [(20, 896, 4864), (33, 2048, 1536), (64, 912, 896), (17, 512, 512)])
def test_sums_over_runs(m, n, k):
    from minfer_amd.kernels import ops
    runs = ops.norm_sum_parts(n, m)
    assert runs == (n + 255) // 256 < ops.norm_sum_parts(n, m, k)
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV)
    w = (torch.randn((n, k), generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV)
    b, g, base = (torch.randn(s, generator=gen).to(DEV) for s in ((n,), (n,), (m, n)))
    want, out = base.clone(), base.clone()
    ops.linear(x, w, b, want, accumulate=True)
    xg, sums = torch.empty((m, n), dtype=torch.bfloat16, device=DEV), torch.full((m, runs), float("nan"), device=DEV)
    assert ops.linear_fused(x, w, b, out, accumulate=True, norm_out=(g, xg, sums))
    if ops.plan_linear(m, n, k)["kernel"].startswith("skinny"):
        assert torch.equal(out, want)
    tol = 4 * 2.0 ** -20 * k ** 0.5                                      # 32-bit sums of exact products of size one and below
    assert (out - (x.double() @ w.double().t() + b.double() + base.double())).abs().max() <= tol
    assert torch.equal(xg, (out * g).to(torch.bfloat16))
    squares = torch.nn.functional.pad(out.double() ** 2, (0, -n % 256)).view(m, runs, 256).sum(-1)
    assert ((sums.double() - squares).abs() <= 1e-5 * squares + 1e-9).all()
    with pytest.raises(ops.KernelError):
        ops.linear_fused(x, w, b, out, accumulate=True, norm_out=(g, xg, torch.empty((m, runs + 1), device=DEV)))
