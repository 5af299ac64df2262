"""In which order a weighted sum of deltas is added to the residual stream: term after term, whoever adds it."""
import weakref
from types import SimpleNamespace

import pytest
import torch

from kipp_amd.parts.block import ParallelBlock
from kipp_amd.parts.norm import LayerNorm, RMSNorm
from kipp_amd.runtime import Runtime, WeightedDelta


class PlainRuntime:
    """The runtime's handling of deltas over plain torch operations."""
    act_dtype = torch.float32
    settle, settle_onto, add = Runtime.settle, Runtime.settle_onto, Runtime.add

    def __init__(self):
        self.ops = SimpleNamespace(residual_add=lambda x, d: x.add_(d), residual_add_terms=self.terms, fill_zero=lambda t: t.zero_(),
                                   layer_norm=lambda x, w, b, eps, out, scale=1.0: out.copy_(x), rmsnorm=lambda x, w, eps, out, delta=None: out.copy_(x))

    def empty(self, shape, dtype):
        return torch.empty(shape, dtype=dtype)

    def rows_of(self, h):
        return h

    def terms(self, x, terms):
        for delta, scale, _ in terms:
            x.add_(scale * delta)
        return x


def _terms(rt, count):
    """Deltas whose sum in float32 depends on the order."""
    return WeightedDelta(rt, [(torch.full((2, 4), v), 1.0, None) for v in (2.0 ** 24, -2.0 ** 24, 0.3)[:count]])


def _in_turn(x, *sums):
    for s in sums:
        for delta, scale, _ in s.terms:
            x = x + scale * delta
    return x


@pytest.mark.parametrize("norm", [LayerNorm, RMSNorm])
def test_a_norm_adds_term_after_term(norm):
    rt = PlainRuntime()
    part = norm(SimpleNamespace(eps=1e-5), rt)
    x, s = torch.full((2, 4), 0.7), _terms(rt, 3)
    want = _in_turn(x, s)
    assert not torch.equal(want, x + s.run())
    assert torch.equal(part.add_forward(x, s, torch.float32), want) and torch.equal(x, want)


@pytest.mark.parametrize("norm", [LayerNorm, RMSNorm])
def test_mixer_and_feed_forward_keep_their_order(norm):
    """A parallel block's two results, added by the next block's norm: the mixer's terms, then the feed-forward's."""
    rt = PlainRuntime()
    block = ParallelBlock.__new__(ParallelBlock)
    mixed, fed = _terms(rt, 2), _terms(rt, 3)
    block.rt, block.mixer = rt, SimpleNamespace(forward=lambda h, batch, cache, state: mixed)
    block.parts = {"mixer_norm": norm(SimpleNamespace(eps=1e-5), rt), "ffn": SimpleNamespace(forward=lambda h, batch: fed)}
    start = torch.full((2, 4), 0.7)
    x, pending = block.forward(start.clone(), None, None, None, None)
    block.parts["mixer_norm"].add_forward(x, pending, torch.float32)
    assert torch.equal(x, _in_turn(start, mixed, fed))


@pytest.mark.parametrize("fed_is_a_sum", [True, False])
@pytest.mark.parametrize("rows_are_few", [True, False])
def test_many_rows_are_added_ahead_of_the_feed_forward(rows_are_few, fed_is_a_sum):
    """With more numbers than `TOGETHER` the mixer's result is in x, and nobody holds it, when the feed-forward runs; the sum is the same."""
    rt = PlainRuntime()
    block = ParallelBlock.__new__(ParallelBlock)
    mixed, fed = _terms(rt, 2), _terms(rt, 3)
    start = torch.full((2, 4), 0.7)
    held = weakref.ref(mixed.terms[0][0])
    want = _in_turn(_in_turn(start, mixed), fed) if fed_is_a_sum else _in_turn(start, mixed) + 0.3
    seen = []

    def feed(h, batch):
        seen.append((held() is None, x.clone()))
        return fed if fed_is_a_sum else torch.full((2, 4), 0.3)
    box = [mixed]
    block.rt, block.mixer, block.TOGETHER = rt, SimpleNamespace(forward=lambda h, batch, cache, state: box.pop()), 8 if rows_are_few else 7
    block.parts = {"mixer_norm": RMSNorm(SimpleNamespace(eps=1e-5), rt), "ffn": SimpleNamespace(forward=feed)}
    added = _in_turn(start, mixed)
    del mixed
    x = start.clone()
    _, pending = block.forward(x, None, None, None, None)
    assert len(seen) == 1 and seen[0][0] == (not rows_are_few) and torch.equal(seen[0][1], start if rows_are_few else added)
    rt.add(x, pending)
    assert torch.equal(x, want)
