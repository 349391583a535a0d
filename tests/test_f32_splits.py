"""How the 32-bit product's K is cut (host side only), and a K of nothing."""
import pytest
import torch

from minfer_amd.kernels import ops


@pytest.mark.parametrize("m,n,k,n_cu", [(9, 64, 0, 256), (100, 4096, 0, 256), (9, 64, 32, 0), (100, 4096, 4096, 0), (9, 64, 16, 256),
                                        (9, 64, -32, 256), (8, 64, 4096, 256)])
def test_nothing_to_cut(m, n, k, n_cu):
    assert ops._f32_splits(m, n, k, True, n_cu) == 1


@pytest.mark.parametrize("n_cu", [1, 8, 256])
def test_parts_are_whole_and_not_too_many(n_cu):
    for m in (9, 64, 65, 400, 611, 4000):
        for n in (1, 64, 600, 4096):
            for k in (32, 64, 224, 448, 896, 4864, 18944):
                parts = ops._f32_splits(m, n, k, True, n_cu)
                per = -(-(k // 32) // parts) * 32
                assert 1 <= parts <= 16 and (parts - 1) * per < k <= parts * per and (parts == 1 or per >= 7 * 32)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 9, 100])
def test_a_product_over_nothing_is_refused(m):
    x, w = torch.empty(m, 0, device="cuda"), torch.empty(64, 0, device="cuda")
    with pytest.raises(ops.KernelError):
        ops.linear(x, w, None, torch.empty(m, 64, device="cuda"))
