"""The whole-K products of 17 to 128 rows with copies straight into LDS, against products in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def operands(m, n, k, seed):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV),
            (torch.randn((n, k), generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV), torch.randn(n, generator=gen).to(DEV))


@pytest.fixture()
def wide():
    """Weight rows that give every CU more than 128 and at most 160: (the least, one that ends inside a unit, the most)."""
    from minfer_amd.kernels import ops
    cu = ops.cu_count()
    return 128 * cu + 1, 144 * cu + 17, 160 * cu


@pytest.mark.parametrize("m", [17, 33, 64, 65, 104, 128])
@pytest.mark.parametrize("which,k", [(0, 64), (1, 192), (2, 512)])
def test_products(wide, m, which, k):
    """One k tile, fewer than the stages hold, more; the first and the last row count; rows and columns that fill no block."""
    from minfer_amd.kernels import ops
    n = wide[which]
    x, w, b = operands(m, n, k, m + n + k)
    want = x.double() @ w.double().t() + b.double()
    tol = 2.0 ** -20 * k ** 0.5                                          # 32-bit sums of exact products of size one and below
    out = torch.full((m, n), float("nan"), device=DEV)
    ops.linear(x, w, b, out, variant=17)
    assert (out - want).abs().max() <= tol * 4
    acc = torch.ones((m, n), device=DEV)
    ops.linear(x, w, None, acc, accumulate=True, variant=17)
    assert (acc - (want - b.double() + 1.0)).abs().max() <= tol * 4
    half = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    ops.linear(x, w, b, half, variant=17)
    assert ((half.double() - want).abs() <= tol * 4 + want.abs() * 2.0 ** -8).all()


@pytest.mark.parametrize("m,nf,k", [(17, 18944, 256), (64, 18944, 512), (100, 18944, 64), (128, 20470, 192), (51, 11008, 1536), (64, 8960, 320),
                                    (53, 12288, 64)])
@pytest.mark.parametrize("clamped", [False, True])
def test_swiglu(m, nf, k, clamped):
    """Gates and ups that different waves hold; outputs that end inside a unit; both activations; the scaled form's rows (at most 64)
    come with their sums of squares in parts, more than are asked for early among them."""
    from minfer_amd.kernels import ops
    if ops.cu_count() != 256:
        pytest.skip("sizes for 256 CUs")
    gen = torch.Generator().manual_seed(m + nf)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV)
    wg, wu = ((torch.randn((nf, k), generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV) for _ in range(2))
    w = ops.interleave_gate_up(wg, wu)
    g, u = x.double() @ wg.double().t(), x.double() @ wu.double().t()
    limit = torch.tensor([1.5], device=DEV) if clamped else None

    def act(g, u):
        if not clamped:
            return g * torch.sigmoid(g) * u
        g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
        return g * torch.sigmoid(1.702 * g) * (u + 1.0)
    out = torch.empty((m, nf), dtype=torch.bfloat16, device=DEV)
    ops.linear_swiglu(x, w, out, variant=17, limit=limit)
    want = act(g, u)
    assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()
    if m > 64 or clamped:
        return
    for parts in (1, 14, 19):
        sums = torch.rand((m, parts), generator=gen).to(DEV) + 0.1
        f = 1.0 / (sums.double().sum(1, keepdim=True) / k + 1e-6).sqrt()
        assert ops.linear_fused(x, w, None, out, swiglu=True, scale_in=(sums, 1e-6))
        want = act(g * f, u * f)
        assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * f * f).all()


def test_which_products_take_it():
    from minfer_amd.kernels import ops
    name = lambda m, n, k, **kw: ops.plan_linear(m, n, k, n_cu=256, **kw)["kernel"]
    for m, n, k in ((65, 37888, 3584), (128, 40960, 512), (100, 32800, 2048), (51, 22016, 2048), (64, 17920, 1536)):
        assert name(m, n, k, swiglu=True) == "panel_dma_kernel"
    for m, n, k in ((129, 37888, 3584), (100, 32768, 2048), (100, 41024, 2048), (50, 22016, 2048), (64, 16384, 1536), (64, 9728, 896)):
        assert name(m, n, k, swiglu=True) != "panel_dma_kernel"
    assert name(64, 22016, 2048) != "panel_dma_kernel" and name(100, 37888, 3584, aligned=False) != "panel_dma_kernel"


@pytest.mark.parametrize("m", [17, 65, 128])
@pytest.mark.parametrize("which,at", [(0, 0), (1, 0), (2, 0), (2, 1), (2, 4)])
def test_bf16_results_are_the_32_bit_ones_rounded(wide, m, which, at):
    """Rows of results that four values do and do not divide, from an address that 8 bytes do and do not; plain and through xIELU."""
    from minfer_amd.kernels import ops
    n, k = wide[which], 192
    x, w, b = operands(m, n, k, m + n)
    out = torch.empty((m, n), device=DEV)
    ops.linear(x, w, b, out, variant=17)
    flat = torch.empty(m * n + at, dtype=torch.bfloat16, device=DEV)
    half = flat[at:].view(m, n)
    ops.linear(x, w, b, half, variant=17)
    assert torch.equal(half, out.to(torch.bfloat16))
    a_pos, a_neg = 0.8, 0.3
    ops.linear(x, w, torch.cat([b, torch.tensor([a_pos, a_neg], device=DEV)]), half, xielu=True, variant=17)
    want = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    ops.xielu(out, want, a_pos, a_neg)
    assert torch.equal(half, want)
