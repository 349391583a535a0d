"""bfloat16 products that are cut over K only because the kernel behind them, the rotation or the norm, adds their parts: a K of up to
3,072, where `linear` runs them whole.  Against products in 64 bits."""
import pytest
import torch

from test_kernels_gpu import make_cache, stored_v

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def operands(m, n, k, seed):
    gen = torch.Generator().manual_seed(seed)
    return tuple(t.to(DEV) for t in (torch.randn((m, k), generator=gen).to(torch.bfloat16),
                                     (torch.randn((n, k), generator=gen) * k ** -0.5).to(torch.bfloat16), torch.randn(n, generator=gen),
                                     torch.randn(n, generator=gen), torch.randn((m, n), generator=gen)))


def cut(ops, m, n, k, epi, behind):
    if ops.cu_count() == 256:
        assert ops._tile_plan(m, n, k, epi, True, 256, 0)[1] == 1
        assert ops._tile_plan(m, n, k, epi, True, 256, behind)[1] > 1
    return ops._tile_plan(m, n, k, epi, True, ops.cu_count(), behind)


# the first and last rows at 1,152 and others; parts of one length and with a shorter last one
@pytest.mark.parametrize("m,n,k", [(65, 1152, 896), (100, 1152, 896), (445, 1152, 896), (200, 2048, 2048), (604, 2048, 2048), (300, 1536, 1536)])
def test_parts_for_the_rotation(m, n, k):
    from minfer_amd.kernels import ops
    _, splits, per = cut(ops, m, n, k, ops.EPI_F32, 1)
    x, w, b, _, _ = operands(m, n, k, m + n)
    parts = ops.linear_parts(x, w)
    assert parts.shape == (splits, m, n)
    tol = 4 * 2.0 ** -20 * per ** 0.5                                    # 32-bit sums of exact products of size one and below
    for p in range(splits):
        s = slice(p * per, min((p + 1) * per, k))
        assert (parts[p].double() - x[:, s].double() @ w[:, s].double().t()).abs().max() <= tol
    # the rotation and the cache from the parts, and from their sum made beforehand in the same order
    hd, nk = 64, 2
    nh = n // hd - 2 * nk
    pos, seq = torch.arange(m, dtype=torch.int32, device=DEV), torch.zeros(m, dtype=torch.int32, device=DEV)
    pages = (m + 63) // 64
    table = torch.arange(pages, dtype=torch.int32, device=DEV).flip(0).view(1, -1).contiguous()
    cs, sn = ops.rope_table(pages * 64, hd // 2, 1e4, 1.0, DEV)
    total = parts[0].clone()
    for p in range(1, splits):
        total += parts[p]
    got = []
    for rows, bias in ((parts, b), (total + b, None)):
        kc, vc = make_cache(pages, nk, hd, torch.bfloat16, 7)
        kd, vd = kc.to(DEV), stored_v(vc).to(DEV)
        q = torch.empty(m, nh * hd, dtype=torch.bfloat16, device=DEV)
        ops.rope_kvwrite(rows, cs, sn, pos, seq, table, q, kd, vd, nh, nk, hd, bias=bias)
        got.append((q, kd, vd))
    for a, c in zip(*got):
        assert torch.equal(a, c)


@pytest.mark.parametrize("m,n,k", [(65, 896, 896), (300, 896, 896), (2455, 896, 896), (604, 2048, 2048), (300, 1536, 1536)])
def test_rows_and_their_norm(m, n, k):
    from minfer_amd.kernels import ops
    x, w, b, g, base = operands(m, n, k, m + n)
    product = x.double() @ w.double().t()
    tol = 4 * 2.0 ** -20 * k ** 0.5
    for accumulate, bias in ((True, None), (False, b), (True, b)):
        if accumulate:
            cut(ops, m, n, k, ops.EPI_ACC_F32, 2)
        got = base.clone()
        normed = ops.linear_norm_out(x, w, bias, got, accumulate, g, 1e-6)
        if normed is None:                                               # stored rows cost less: fewer of them are cut
            assert not accumulate and ops._tile_plan(m, n, k, ops.EPI_F32, True, ops.cu_count(), 2)[1] == 1 and torch.equal(got, base)
            continue
        want = product + (0 if bias is None else bias.double()) + (base.double() if accumulate else 0)
        assert (got.double() - want).abs().max() <= tol
        rows = got.double()
        want_n = rows / (rows.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * g.double()
        assert ((normed.double() - want_n).abs() <= want_n.abs() * (2.0 ** -8 + 1e-5)).all()
