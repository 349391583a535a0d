"""How blocks of queries of the prompt attention are shared out (host side only)."""
import heapq

import pytest
import torch

from minfer_amd.engine.batch import StepContext


def step(new, start):
    one = torch.zeros(1, dtype=torch.int32)
    return StepContext(cache=None, n_tokens=sum(new), n_seqs=len(new), token_ids=one, positions=one, seq_of_tok=one, cu_seqlens=one,
                       start_pos=one, slot_ids=one, logit_rows=None, page_tables={}, max_len=max(a + b for a, b in zip(new, start)),
                       max_new=max(new), all_decode=False, host_new=list(new), host_start=list(start))


@pytest.mark.parametrize("new,start,block,heads,per_cu,window", [
    ([180, 101, 168, 155], [5000, 4997, 4994, 4991], 16, 2, 2, 0),     # 560 workgroups by the even share alone
    ([60, 30], [4000, 3997], 18, 4, 2, 0),
    ([1500], [0], 18, 2, 2, 0),
    ([700, 20], [3000, 100], 16, 2, 2, 1000),
    ([300, 300, 300, 300], [5000] * 4, 10, 8, 1, 0),                   # more blocks than places: not all at once
])
def test_shares_fit_the_chip_and_cover_every_page_once(new, start, block, heads, per_cu, window):
    places = 256 * per_cu
    got = step(new, start).shared_query_tiles(block, 64, window, heads, 256, per_cu, 4, 8, at_once=True)
    blocks = [(b, q) for b, n in enumerate(new) for q in range(0, n, block)]
    if got is None:
        assert len(blocks) * heads > places
        return
    seqs, starts, words, n_slots, most = (x.tolist() if isinstance(x, torch.Tensor) else x for x in got)
    assert len(blocks) * heads > places or len(words) * heads <= places
    listed = {}
    for b, q, w in zip(seqs, starts, words):
        listed.setdefault((b, q), []).append((w & 255, max(1, (w >> 8) & 255)))
    assert sorted(listed) == sorted(blocks)
    for shares in listed.values():
        assert sorted(s for s, _ in shares) == list(range(shares[0][1])) and shares[0][1] <= most <= 8
    assert n_slots == len({w >> 16 for w in words if w})


def last_end(new, start, block, heads, places, at_once):
    """When the last workgroup of a step's plan ends, in pages: each takes the place that is free first, the longest first; four
    pages' time to start and leave."""
    got = step(new, start).shared_query_tiles(block, 64, 0, heads, 256, places // 256, 4, 8, at_once=at_once)
    if got is None:
        entries = [(b, q, 0) for b, n in enumerate(new) for q in range(0, n, block)]
    else:
        entries = list(zip(*(x.tolist() for x in got[:3])))
    walks = []
    for b, q, w in entries:
        pages, shares = (start[b] + min(q + block, new[b]) - 1) // 64 + 1, max(1, (w >> 8) & 255)
        walks += [(pages - (w & 255) + shares - 1) // shares + 4] * heads
    free = [0] * places
    for w in sorted(walks, reverse=True):
        heapq.heapreplace(free, free[0] + w)
    return max(free)


@pytest.mark.parametrize("shorts", [0, 60, 100, 119, 120, 121, 124, 125, 126, 127, 128, 140])
@pytest.mark.parametrize("heads,long_new,long_start", [(4, 36, 30000), (4, 36, 9000), (2, 36, 30000), (3, 36, 120000), (4, 611, 8000), (4, 300, 3000)])
def test_fitting_shares_to_the_chip_costs_no_time(shorts, heads, long_new, long_start):
    """However many prompts of one block there are beside a turn on a long context, the last workgroup ends no later than by the even
    share (a tenth for the rounding of walks)."""
    new, start = [18] * shorts + [long_new], [0] * shorts + [long_start]
    even, fitted = (last_end(new, start, 18, heads, 512, at_once) for at_once in (False, True))
    assert fitted <= 1.1 * even


def test_fitting_shares_to_the_chip_gains_where_a_few_workgroups_would_wait():
    new, start = [180, 101, 168, 155], [5000, 4997, 4994, 4991]
    assert last_end(new, start, 16, 2, 512, True) < 0.75 * last_end(new, start, 16, 2, 512, False)
    assert last_end([611], [8000], 18, 4, 512, True) < 0.8 * last_end([611], [8000], 18, 4, 512, False)

def test_how_parts_are_added_up():
    """The last workgroup of a block adds its parts where they are few and every workgroup has a CU; heads beyond 128 never."""
    from minfer_amd.kernels.ops import prefill_parts_meet as meet
    assert meet(64, 2, 6, 40, 256) and meet(128, 2, 126, 252, 256) and not meet(128, 2, 168, 360, 256)
    assert meet(128, 4, 72, 198, 256) and not meet(128, 3, 8, 24, 256) and not meet(128, 4, 48, 192, 256)
    assert not meet(128, 8, 32, 200, 256) and not meet(144, 2, 6, 40, 256) and not meet(256, 2, 6, 12, 256)
