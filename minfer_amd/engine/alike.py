"""A step's layers that differ in their tensors alone.

What a layer of a short prompt costs the host (some 85 us of Python and checks for eight launches) is more than what it costs
the device.  Within a step the launches of one layer are recorded as they are made, and for the layers behind it that are
alike (the same parts with the same constants, tensors of the same types and shapes: `Block.alike`) they are made again from
native code with the layer's own tensors in their places (35 us).  Nothing outlives the step, and a layer that is not alike, or
a step whose launches are timed one by one, takes the general path.

What a recorded layer launched with stays allocated together until its record is dropped (the 7B shape: some 85 KB a token, where
52 are live at once in the general path).  So only steps of up to MOST_VALUES values in the stream are recorded (585 tokens of the
7B shape, 50 MB; 2,340 of the 0.5B one), beyond which the device takes longer for a layer than the host does without a record, and
the record is dropped before the last block and the head.
"""
from __future__ import annotations

from ..kernels import ops
from ..parts.base import NormAhead

MOST_VALUES = 1 << 21


def _pair(ahead):
    return (None, None) if ahead is None else (ahead.xg, ahead.sums)


class AlikeLayers:
    """One step's run over its schedule.  Scratch of the recorded layer serves those behind it (they run one after the other on
    one stream); what a layer prepares for the next one's norm (`NormAhead`) goes to the one of two places that it does not
    read."""

    def __init__(self):
        self.record = self.key = None
        self.pairs = ()

    def forward(self, block, h, ctx, entry: int, writes_cache: bool):
        """`block.forward` over all of h's rows, which stay in place."""
        after = ctx.norm_after_block
        mine, behind = block.alike(ctx, entry, writes_cache), None if after is None else after.alike()
        if mine is None or behind is None:
            self.record = None
            return block.forward(h, ctx, entry, writes_cache)
        key, tensors = (mine[0], behind[0], h.shape), mine[1] + behind[1]
        ahead = ctx.norm_ahead
        if ahead is not None and (ahead.norm is not block.first_norm() or ahead.h is not h):
            ahead = None
        if self.record is not None and self.key == key and self._again(block, after, h, ctx, tensors, ahead):
            return h
        self.record = record = ops.record_launches()
        if record is None:
            return block.forward(h, ctx, entry, writes_cache)
        with record:
            out = block.forward(h, ctx, entry, writes_cache)
        left = ctx.norm_ahead
        self.key, self.pairs = key, (_pair(ahead), _pair(left))
        like = [[None if t is None else (t.dtype, t.shape) for t in p] for p in self.pairs]
        if out is not h or like[0] != like[1] or (left is not None and (left.norm is not after or left.h is not h)) or \
                not record.bind(tensors + self.pairs[0] + self.pairs[1]):
            self.record = None
        return out

    def _again(self, block, after, h, ctx, tensors, ahead) -> bool:
        taken = _pair(ahead)
        if taken[0] is self.pairs[0][0]:
            left = self.pairs[1]
        elif taken[0] is self.pairs[1][0]:
            left = self.pairs[0]
        else:
            return False
        rc = self.record.run(tensors + taken + left)
        if rc is None:
            return False
        ops.check_recorded(rc)
        ctx.norm_ahead = None if left[0] is None else NormAhead(after, h, *left)
        return True
