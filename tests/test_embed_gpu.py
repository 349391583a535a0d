"""Rows of the embedding table, several values a load where the rows allow it: the very values, whatever the width and the alignment."""
import pytest
import torch

from minfer_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
# a part of a block's threads; all of them once, twice, and once more; fours without eights; single values
@pytest.mark.parametrize("d", [8, 896, 2048, 4096, 4104, 12, 1004, 7, 513])
@pytest.mark.parametrize("offset", [0, 1])
def test_embed(dtype, d, offset):
    vocab = 11
    table = torch.randn(vocab * d + 8, device="cuda").to(dtype)[offset:offset + vocab * d].view(vocab, d)
    ids = torch.tensor([3, 0, 10, 3], dtype=torch.int32, device="cuda")
    out = torch.empty(4, d, dtype=torch.float32, device="cuda")
    ops.embed(table, ids, out)
    assert torch.equal(out, table[ids.long()].float())
