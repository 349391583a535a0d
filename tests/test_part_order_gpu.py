"""Products cut along K on either side of two tiles a CU, where the order of the parts' tiles changes, against 32 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m,n,k", [(1030, 896, 4864), (2600, 3584, 18944), (5754, 3584, 18944)])
def test_every_tile_of_every_part(m, n, k):
    from minfer_amd.kernels import ops
    assert ops.plan_linear(m, n, k, n_cu=256)["splits"] > 1
    gen = torch.Generator(device=DEV).manual_seed(m)
    x, w = (torch.randn(s, generator=gen, device=DEV).to(torch.bfloat16) for s in ((m, k), (n, k)))
    base = torch.randn((m, n), generator=gen, device=DEV)
    want = base + x.float() @ w.float().t()
    out = base.clone()
    ops.linear(x, w, None, out, accumulate=True)
    # two 32-bit sums of k exact products, each some sqrt(k) roundings of at most half a unit of the largest sum
    assert (out - want).abs().max() <= 2.0 ** -22 * float(want.abs().max()) * k ** 0.5


@pytest.mark.parametrize("m,n,k", [(604, 896, 4864), (680, 896, 4864), (300, 1024, 8192), (300, 2048, 8192), (300, 2112, 8192)])
def test_either_side_of_the_activations_that_change_the_order(m, n, k):
    """Between one and one and a half times an XCD's L2, and more; few weight rows of a long K and others."""
    test_every_tile_of_every_part(m, n, k)
