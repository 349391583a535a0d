"""How blocks of queries of the prompt attention are shared out (host side only)."""
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


@pytest.mark.parametrize("shorts", [0, 60, 100, 119, 120, 121, 124, 125, 126, 127, 128, 140])
@pytest.mark.parametrize("heads,long_start", [(4, 30000), (4, 9000), (2, 30000), (3, 120000)])
def test_the_longest_walk_stays_short_beside_many_short_prompts(shorts, heads, long_start):
    """A step's time is its longest walk: fitting the workgroups to the chip lengthens it by a quarter at most, however many prompts
    of one block there are beside a turn on a long context."""
    new, start = [18] * shorts + [36], [0] * shorts + [long_start]
    blocks = shorts + 2
    pages = (long_start + 36 - 1) // 64 + 1

    def longest(got):
        if got is None:
            return pages
        seqs, starts, words, _, _ = (x.tolist() if isinstance(x, torch.Tensor) else x for x in got)
        return max(-(-((s + min(q + 18, n) - 1) // 64 + 1) // max(1, (w >> 8) & 255))
                   for b, q, w in zip(seqs, starts, words) for n, s in [(new[b], start[b])])
    even = longest(step(new, start).shared_query_tiles(18, 64, 0, heads, 256, 2, 4, 8))
    fitted = longest(step(new, start).shared_query_tiles(18, 64, 0, heads, 256, 2, 4, 8, at_once=True))
    assert fitted <= 1.25 * even and even <= -(-pages // 8) + 1, (blocks, even, fitted, pages)
