"""In which order a weighted sum of deltas is added to the residual stream: term after term, whoever adds it."""
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
