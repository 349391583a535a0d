"""Rows that a split product adds up and norms at once (`reduce_norm_kernel`): both sizes of its blocks."""
import pytest
import torch

from test_kernels_gpu import DEV, ops, test_split_product_with_norm as split_product_with_norm  # noqa: F401 (`ops` is a fixture)

pytestmark = pytest.mark.gpu


# More rows than CUs (256 threads a row): a thread's one, two, four, eight and sixteen fours, whole and not.  Up to a row a CU:
# 1,024 threads from 1,028 values on; at 16,368 the row and the sums fill 64 KB of LDS, at 16,384 256 threads take it.
@pytest.mark.parametrize("m,n,k,name", [(300, 1024, 4096, "tile_step_kernel<128,128>"), (300, 1028, 4096, "tile_step_kernel<128,128>"),
                                        (300, 1536, 8960, "tile_dma_kernel<128,256>"), (257, 3584, 3584, "tile_dma_kernel<128,256>"),
                                        (300, 8192, 4096, "tile_dma_kernel<128,256>"), (300, 9000, 4096, "tile_dma_kernel<128,256>"),
                                        (256, 1024, 4096, "tile_step_kernel<64,64>"), (256, 3584, 3584, "tile_dma_kernel<128>"),
                                        (256, 9000, 4096, "tile_dma_kernel<128>"), (66, 16368, 4096, "tile_dma_kernel<128,256>"),
                                        (100, 16384, 4096, "tile_dma_kernel<128,256>")])
def test_split_product_with_norm_of_many_rows_and_wide_ones(ops, m, n, k, name):  # noqa: F811
    split_product_with_norm(ops, m, n, k, name)
