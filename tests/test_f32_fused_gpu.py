"""32-bit products that leave their parts, the norm of the new rows or SwiGLU's values: the same bits as one kernel after the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def operands(m, n, k, seed):
    gen = torch.Generator().manual_seed(seed)
    return tuple(t.to(DEV) for t in (torch.randn((m, k), generator=gen), torch.randn((n, k), generator=gen) * k ** -0.5,
                                     torch.randn(n, generator=gen), torch.randn(n, generator=gen), torch.randn((m, n), generator=gen)))


# rows of one, two, four, eight and sixteen runs of 1,024 values, whole and not; two parts to more than eight
@pytest.mark.parametrize("m,n,k", [(65, 896, 4864), (100, 1028, 2048), (9, 2048, 4096), (70, 3584, 3584), (33, 8192, 2048), (20, 9000, 4096),
                                   (300, 260, 8960)])
def test_norm_and_parts(m, n, k):
    from minfer_amd.kernels import ops
    x, w, b, g, base = operands(m, n, k, m + n)
    parts = ops.linear_parts(x, w)
    assert parts is not None and parts.shape[0] > 1
    for accumulate, bias in ((True, None), (False, b), (True, b)):
        want, got = base.clone(), base.clone()
        ops.linear(x, w, bias, want, accumulate=accumulate)
        want_n = torch.empty_like(want)
        ops.rmsnorm(want, g, 1e-6, want_n)
        normed = ops.linear_norm_out(x, w, bias, got, accumulate, g, 1e-6)
        assert torch.equal(got, want) and torch.equal(normed, want_n)
        total = torch.zeros_like(want)
        for p in parts:
            total = total + p
        total = total if bias is None else total + bias
        assert torch.equal(base + total if accumulate else total, want)
    assert ops.linear_norm_out(x, w[:, :k - 4].contiguous(), None, base.clone(), True, g, 1e-6) is None
    odd = w[:n - 1]
    assert ops.linear_norm_out(x, odd, None, base[:, :n - 1].contiguous(), True, g[:n - 1], 1e-6) is None    # rows not in fours


@pytest.mark.parametrize("m,f,k", [(64, 8192, 32), (611, 4864, 160), (130, 8193, 64), (65, 8222, 96), (1000, 1001, 64)])
@pytest.mark.parametrize("limit", [0.0, 0.8])
def test_swiglu(m, f, k, limit):
    from minfer_amd.kernels import ops
    x, w, _, _, _ = operands(m, 2 * f, k, m + f)
    sums, want, got = torch.empty((m, 2 * f), device=DEV), torch.empty((m, f), device=DEV), torch.full((m, f), float("nan"), device=DEV)
    ops.linear(x, w, None, sums)
    ops.swiglu(sums, want, limit=limit)
    assert ops.linear_swiglu_f32(x, w, got, limit=limit)
    assert torch.equal(got, want)
    assert not ops.linear_swiglu_f32(x[:8], w, got[:8], limit=limit)
