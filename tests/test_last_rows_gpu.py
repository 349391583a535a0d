"""Products whose last few weight rows are a launch of their own, against the product in 32 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m,n,k", [(65, 257, 64), (300, 512 + 16, 128), (257, 768 + 33, 192), (1030, 1024 + 64, 256), (2048, 8224, 64)])
def test_last_weight_rows_apart(m, n, k):
    from minfer_amd.kernels import ops
    gen = torch.Generator().manual_seed(m + n)
    x, w = (torch.randn(s, generator=gen).to(torch.bfloat16) for s in ((m, k), (n, k)))
    b, base = torch.randn(n, generator=gen), torch.randn((m, n), generator=gen)
    want = (x.double() @ w.double().t()).float()
    bound = 2.0 ** -20 * float(want.abs().max()) * k ** 0.5            # 32-bit sums of exact products
    xd, wd, bd = x.to(DEV), w.to(DEV), b.to(DEV)
    out = torch.full((m, n), float("nan"), device=DEV)
    ops.linear(xd, wd, bd, out, variant=16)
    assert (out.cpu() - (want + b)).abs().max() <= bound
    acc = base.to(DEV)
    ops.linear(xd, wd, None, acc, accumulate=True, variant=16)
    assert (acc.cpu() - (want + base)).abs().max() <= bound
    half = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    ops.linear(xd, wd, bd, half, variant=16)
    assert ((half.cpu().float() - (want + b)).abs() <= bound + (want + b).abs() * 2.0 ** -8).all()


def test_which_products_take_it():
    """2,048 rows against 8,224 of 2,048 do on 256 CUs; whole tiles, longer rests, SwiGLU and the general kernels' shapes never."""
    from minfer_amd.kernels import ops
    named = "tile kernels (the last weight rows apart)"
    assert ops.plan_linear(2048, 8224, 2048, n_cu=256)["kernel"] == named
    for n, k, kw in ((8192, 2048, {}), (8320, 2048, {}), (8256, 2048, dict(swiglu=True)), (8224, 2056, {})):
        assert ops.plan_linear(2048, n, k, n_cu=256, **kw)["kernel"] != named
    with pytest.raises(ops.KernelError):
        x = torch.zeros((128, 64), dtype=torch.bfloat16, device=DEV)
        ops.linear(x, torch.zeros((512, 64), dtype=torch.bfloat16, device=DEV), None, torch.empty((128, 512), device=DEV), variant=16)


# as above, rests of up to 64 rows behind one tile and several
@pytest.mark.parametrize("m,n,k", [(65, 257, 64), (257, 768 + 33, 192), (1030, 1024 + 64, 256), (2048, 8200, 4096)])
def test_square_of_relu_of_the_last_rows(m, n, k):
    """max(z, 0)^2 in the epilogues of both launches: the bits of the product in 32 bits, cut the same way, and the activation's kernel."""
    from minfer_amd.kernels import ops
    gen = torch.Generator().manual_seed(m + n)
    x, w = (torch.randn(s, generator=gen).to(torch.bfloat16).to(DEV) for s in ((m, k), (n, k)))
    b, sums = torch.randn(n, generator=gen).to(DEV), torch.empty((m, n), device=DEV)
    ops.linear(x, w, b, sums, variant=16)
    want, out = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.relu2(sums, want)
    ops.linear(x, w, b, out, variant=16, relu2=True)
    assert torch.equal(out, want)
    if m == 2048:
        assert ops.tile_plan(m, n, k, ops.EPI_RELU2, n_cu=256)[0] == 16
        ops.linear(x, w, b, out.fill_(0), relu2=True)
        assert torch.equal(out, want)
