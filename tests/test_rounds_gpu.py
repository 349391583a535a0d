"""Products of few rows whose waves walk their slice of K in rounds of held steps: slices shorter than a round, of whole rounds, with few
and many steps past the last whole one, and waves with a shorter slice than the others or none."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _operands(m, n, k):
    gen = torch.Generator().manual_seed(m + n + k)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16).to(DEV)
    w = (torch.randn((n, k), generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV)
    return x, w, torch.randn(n, generator=gen).to(DEV), torch.randn((m, n), generator=gen).to(DEV)


# steps of 32 a wave (eight waves): 1, 2, 4, 5, 8, 9, 12, 13, 16, 17 .. 31, also with waves that have fewer of them
@pytest.mark.parametrize("k", [32, 96, 416, 1024, 1056, 2048, 2080, 3072, 3104, 3936, 4128, 4352, 4384, 4640, 4864, 5376, 5632, 5920, 6400, 6688, 7424, 7904, 7936])
@pytest.mark.parametrize("m,n", [(1, 80), (16, 896)])
def test_rolling(m, n, k):
    from minfer_amd.kernels import ops
    x, w, b, base = _operands(m, n, k)
    tiled = ops.tile_weight(w)
    assert ops.plan_linear(m, n, k, accumulate=True, tiled=True)["kernel"] == "rolling16_kernel"
    got = [base.clone() for _ in range(2)]
    for out, t in zip(got, (tiled, None)):
        ops.linear(x, w, b, out, accumulate=True, tiled=t)
    assert torch.equal(*got)
    want = x.double() @ w.double().t() + b.double() + base.double()
    assert (got[0] - want).abs().max() <= 4 * 2.0 ** -20 * k ** 0.5 + 2.0 ** -22      # 32-bit sums of exact products of size one and below


# eleven to nineteen steps a wave: two rounds of six, eight and ten
@pytest.mark.parametrize("m,n,k", [(17, 512, 2816), (20, 528, 3040), (33, 512, 3072), (17, 640, 3104), (48, 512, 3840), (17, 896, 4096),
                                   (30, 896, 4128), (40, 512, 4480)])
def test_whole(m, n, k):
    from minfer_amd.kernels import ops
    x, w, b, base = _operands(m, n, k)
    assert ops.plan_linear(m, n, k, accumulate=True, norm_out=True)["kernel"] == "whole_kernel"
    left = []
    for tiled in (ops.tile_weight(w), None):
        out, xg = base.clone(), torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
        sums = torch.empty((m, ops.norm_sum_parts(n, m, k)), device=DEV)
        assert ops.linear_fused(x, w, b, out, accumulate=True, tiled=tiled, norm_out=(b, xg, sums))
        left.append((out, xg, sums))
    assert all(torch.equal(p, q) for p, q in zip(*left))
    want = x.double() @ w.double().t() + b.double() + base.double()
    assert (left[0][0] - want).abs().max() <= 4 * 2.0 ** -20 * k ** 0.5


# the register-resident kernel with one item a block and with several, old values and biases an item ahead
@pytest.mark.parametrize("m,n,k", [(1, 2064, 1024), (16, 4608, 3584), (8, 20000, 896), (16, 9000, 2048), (3, 16400, 4096)])
def test_stationary(m, n, k):
    from minfer_amd.kernels import ops
    x, w, b, base = _operands(m, n, k)
    assert ops.plan_linear(m, n, k, accumulate=True)["kernel"] == "stationary16_kernel"
    want = x.double() @ w.double().t() + b.double()
    for tiled in (ops.tile_weight(w), None):
        out = base.clone()
        ops.linear(x, w, b, out, accumulate=True, tiled=tiled)
        assert (out - (want + base.double())).abs().max() <= 4 * 2.0 ** -20 * k ** 0.5 + 2.0 ** -22


# the same with the norm folded in and with SwiGLU, at the lengths whose weights go through a shorter ring than a slice
@pytest.mark.parametrize("m,n,k", [(8, 9024, 6144), (16, 4416, 7168), (3, 16384, 5120), (5, 2112, 8192)])
def test_stationary_of_long_rows(m, n, k):
    from minfer_amd.kernels import ops
    x, w, b, _ = _operands(m, n, k)
    h, gain = x.float(), torch.rand(k, device=DEV) + 0.5
    h *= 1.0 + 2.0 ** -9                                    # (not the bfloat16 values themselves)
    xg = (h * gain).to(torch.bfloat16).double()
    z = xg @ w.double().t() / (h.double().square().mean(-1, keepdim=True) + 1e-6).sqrt()
    left = []
    for tiled in (ops.tile_weight(w), None):
        out, half = torch.empty((m, n), device=DEV), torch.empty((m, n // 2), device=DEV, dtype=torch.bfloat16)
        assert ops.linear_normed(h, gain, 1e-6, None, w, b, out, tiled=tiled)
        assert ops.linear_normed(h, gain, 1e-6, None, w, None, half, tiled=tiled, swiglu=True)
        left.append((out, half))
    assert all(torch.equal(p, q) for p, q in zip(*left))
    assert (left[0][0] - (z + b.double())).abs().max() <= 4 * 2.0 ** -20 * k ** 0.5 + 2.0 ** -22
    gate, up = z.view(m, -1, 2, 32).unbind(2)
    want = (torch.nn.functional.silu(gate) * up).reshape(m, n // 2)
    assert (left[0][1].double() - want).abs().max() <= 2.0 ** -8 * want.abs().max() + 2.0 ** -12
