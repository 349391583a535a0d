"""The 32-bit prompt attention alone against the plain one."""
import math

import numpy as np
import pytest
import torch

import plain_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from minfer_amd.kernels import ops as o
    return o


def close(a, b, tol):
    a, b = a.detach().cpu().double(), b.detach().cpu().double()
    err = (a - b).abs()
    assert bool((err <= tol + tol * b.abs()).all()), f"max err {err.max().item():.3e}"


def prompt_case(nh, nk, hd, new, start, seed):
    """Sequences that hold start[b] tokens and bring new[b] more, in shuffled pages whose unwritten rows are NaN."""
    from minfer_amd.engine.batch import StepContext
    gen = torch.Generator().manual_seed(seed)
    lengths = [s + n for s, n in zip(start, new)]
    pages = torch.randperm(sum((l + 63) // 64 for l in lengths), generator=gen).int()
    table = -torch.ones((len(new), (max(lengths) + 63) // 64), dtype=torch.int32)
    kc, vc = (torch.randn((len(pages), nk, 64, hd), generator=gen) for _ in range(2))
    at = 0
    for b, l in enumerate(lengths):
        n = (l + 63) // 64
        table[b, :n] = pages[at:at + n]
        at += n
        if l % 64:
            for cache in (kc, vc):
                cache[table[b, n - 1], :, l % 64:] = float("nan")
    n_tok = sum(new)
    q = torch.randn((n_tok, nh * hd), generator=gen)
    pos = torch.cat([torch.arange(s, s + n) for s, n in zip(start, new)]).int()
    seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new)).int()
    cu = torch.tensor([0] + list(np.cumsum(new)), dtype=torch.int32)

    def ctx_on(dev):
        return StepContext(cache=None, n_tokens=n_tok, n_seqs=len(new), token_ids=torch.zeros(n_tok, dtype=torch.int32, device=dev),
                           positions=pos.to(dev), seq_of_tok=seq.to(dev), cu_seqlens=cu.to(dev),
                           start_pos=torch.tensor(start, dtype=torch.int32, device=dev),
                           slot_ids=torch.zeros(len(new), dtype=torch.int32, device=dev), logit_rows=None,
                           page_tables={}, max_len=max(lengths), max_new=max(new), all_decode=False,
                           host_new=list(new), host_start=list(start))
    return q, kc, vc, table, ctx_on


@pytest.mark.parametrize("nh,nk,hd,window", [(14, 2, 64, 0), (12, 2, 128, 0), (4, 1, 16, 0), (9, 3, 48, 33), (5, 5, 80, 0),
                                             (40, 2, 32, 0), (6, 2, 112, 100), (7, 1, 96, 1)])
def test_attn_prompt_f32(ops, nh, nk, hd, window):
    """32-bit prompts: runs of 16 (token, head of the group) rows that end in the middle of a token's heads, of a sequence and of
    the keys' runs of 16; few tokens on a long context, whose keys are cut over blocks; unwritten rows of the pages are NaN."""
    new = [1, 2, 15, 16, 17, 33, 64, 65, 130, 3]
    start = [0, 5, 0, 63, 64, 0, 700, 0, 0, 1100]
    for cut in (slice(0, 10), slice(9, 10)):                      # the last sequence alone: keys in splits
        q, kc, vc, table, ctx_on = prompt_case(nh, nk, hd, new[cut], start[cut], 29)
        scale = 1.0 / math.sqrt(hd)
        ref = torch.empty(q.shape, dtype=torch.float64)
        plain_ops.attn_prefill(q, kc, vc, table, ctx_on("cpu"), ref, nh, nk, hd, scale, window)
        ctx = ctx_on(DEV)
        tiles = ctx.row_tiles(nh // nk, ops.prompt_f32_rows(hd))[0].numel()
        splits = ops.prompt_f32_splits(tiles * nk, 128, ctx.max_len, ops.cu_count())
        assert cut.start == 0 or splits[0] > 1, splits
        outs = [torch.full(q.shape, float("nan"), device=DEV) for _ in range(2)]
        for out in outs:
            ops.attn_prompt_f32(q.to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), ctx, out, nh, nk, hd, scale, window)
        close(outs[0], ref, 3e-6)                           # (the bound of `test_attn_tokens`)
        assert torch.equal(outs[0], outs[1]), "two runs differ"


def test_attn_prompt_f32_keeps_values_that_are_no_numbers_apart(ops):
    """An infinite value reaches the tokens that see its key and no earlier token of the same block."""
    nh, nk, hd, bad = 4, 2, 64, 41
    q, kc, vc, table, ctx_on = prompt_case(nh, nk, hd, [50], [0], 31)
    clean = torch.empty(q.shape, device=DEV)
    args = (table.to(DEV), ctx_on(DEV))
    ops.attn_prompt_f32(q.to(DEV), kc.to(DEV), vc.to(DEV), *args, clean, nh, nk, hd, 0.125, 0)
    vc[table[0, 0], :, bad, 7] = float("inf")
    out = torch.empty(q.shape, device=DEV)
    ops.attn_prompt_f32(q.to(DEV), kc.to(DEV), vc.to(DEV), *args, out, nh, nk, hd, 0.125, 0)
    same = torch.ones(50, nh, hd, dtype=torch.bool)
    same[bad:, :, 7] = False
    out, clean = out.cpu().view(50, nh, hd), clean.cpu().view(50, nh, hd)
    assert torch.isinf(out[~same]).all()
    # (a run with such a value is added up key by key: other roundings in the other columns)
    close(out[same].double(), clean[same].double(), 1e-6)


@pytest.mark.parametrize("m,n,k", [(65, 130, 896),          # whole, few tiles
                                   (611, 1152, 896),        # in parts of which the last is shorter
                                   (611, 9728, 896),        # whole, an eighth of the tiles an XCD
                                   (300, 200, 4128),        # in parts, 4.9 MB of activations: part by part
                                   (1000, 4100, 1088),      # whole, 4.4 MB of activations: tile by tile
                                   (9, 64, 32)])            # one tile of one k tile
def test_products_of_many_rows(ops, m, n, k):
    """The 32-bit product's parts and tile orders.  Bound: a sum of k terms in chains of 128 whose sums are added in turn errs by at
    most (128 + k / 128 + parts + 2) half units in the last place of the sum of the terms' sizes; a quarter of that is far above
    what roundings of either sign come to."""
    gen = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=gen), torch.randn((n, k), generator=gen)
    b, base = torch.randn(n, generator=gen), torch.randn((m, n), generator=gen)
    want = x.double() @ w.double().t() + b.double()
    size = x.abs().double() @ w.abs().double().t()
    bound = 0.25 * (128 + k / 128 + 18) * 2.0 ** -24 * size + 1e-6
    for accumulate in (False, True):
        out = base.to(DEV)
        ops.linear(x.to(DEV), w.to(DEV), b.to(DEV), out, accumulate=accumulate)
        err = (out.cpu().double() - want - (base.double() if accumulate else 0.0)).abs()
        assert bool((err <= bound).all()), (err / bound).max().item()
