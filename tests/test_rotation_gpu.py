"""The rotation's arithmetic, to the bit: one part and several, few tokens and many, both run types."""
import numpy as np
import pytest
import torch

from test_kernels_gpu import DEV, make_cache, ops, rnd, stored_v  # noqa: F401 (`ops` is a fixture)

pytestmark = pytest.mark.gpu


def fused(a, b, c):
    """a b + c with one rounding: the product of two 32-bit numbers is exact in 64 bits.  (The sum is rounded to 53 bits first, which
    shows once in some 2^29 values.)"""
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(np.float32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("parts", [1, 2, 9])
@pytest.mark.parametrize("t,nh,nk,hd", [(67, 3, 1, 24), (67, 28, 4, 128), (300, 40, 8, 128), (67, 2, 2, 256), (256, 9, 3, 48),
                                        (257, 9, 3, 48), (1300, 9, 3, 48)])
def test_rotation_is_fused_the_same_way_in_every_form(ops, dtype, parts, t, nh, nk, hd):  # noqa: F811
    """A token a CU (256) and more; in parts as many as are on the chip at once (here 256 x 20 / waves of a block) and more."""
    width, half = (nh + 2 * nk) * hd, hd // 2
    rows, bias = rnd((parts, t, width), seed=5), rnd((width,), seed=6)
    pos = torch.arange(3, 3 + t, dtype=torch.int32)
    seq, table = torch.zeros(t, dtype=torch.int32), torch.randperm(22, generator=torch.Generator().manual_seed(1)).int().view(1, -1)
    cs, sn = ops.rope_table(1408, half, 1e4, 1.0, DEV)
    kc, vc = make_cache(22, nk, hd, dtype, 7)
    kd, vd, q = kc.to(DEV), stored_v(vc).to(DEV), torch.empty(t, nh * hd, dtype=dtype, device=DEV)
    ops.rope_kvwrite((rows if parts > 1 else rows[0]).to(DEV), cs, sn, pos.to(DEV), seq.to(DEV), table.to(DEV), q, kd, vd, nh, nk, hd,
                     bias=bias.to(DEV) if parts > 1 else None)
    x = rows[0].clone() if parts == 1 else torch.zeros(t, width)
    if parts > 1:
        for p in rows:
            x = x + p
        x = x + bias
    x = x.view(t, nh + 2 * nk, hd).numpy()
    c, s = (v.cpu().numpy()[pos.numpy()][:, None] for v in (cs, sn))
    x0, x1 = x[:, :nh + nk, :half], x[:, :nh + nk, half:]
    low, high = fused(x0, c + 0 * x0, -(x1 * s)), fused(x1, c + 0 * x1, x0 * s)
    want = torch.from_numpy(np.concatenate([low, high], axis=2)).to(dtype)
    assert torch.equal(q.cpu().view(t, nh, hd), want[:, :nh])
    v = torch.from_numpy(x[:, nh + nk:]).to(dtype)
    k_want, v_want = kc.clone(), vc.clone()
    for i, p in enumerate(pos.tolist()):
        page = table[0, p // 64]
        k_want[page, :, p % 64], v_want[page, :, p % 64] = want[i, nh:], v[i]
    assert torch.equal(kd.cpu(), k_want) and torch.equal(vd.cpu(), stored_v(v_want))
