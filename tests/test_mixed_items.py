"""What layers with mixed heads make of a step: which form takes which tokens, and the space that is made for it."""
import random
import time
from types import SimpleNamespace

import torch

from kipp_amd.csrc import ops
from kipp_amd.engine.batch import StepBatch
from kipp_amd.parts.mixed_attention import MixedHeadAttention


def batch_of(q_len, ctx_len):
    starts = [sum(q_len[:i]) for i in range(len(q_len))]
    single = [c for n, c in zip(q_len, ctx_len) if n == 1]
    return StepBatch(sum(q_len), len(q_len), 0, torch.zeros(sum(q_len), dtype=torch.int32), *[None] * 7, {}, n_decode=len(single),
                     n_portions=len(q_len) - len(single), max_decode_ctx=max(single, default=0), max_q_len=max(q_len),
                     host={"q_start": starts, "q_len": q_len, "ctx_len": ctx_len})


def layer_of(heads, kv_heads, window=None):
    layer = MixedHeadAttention.__new__(MixedHeadAttention)
    layer.spec = SimpleNamespace(num_heads=heads, num_kv_heads=kv_heads, v_head_dim=32, window=window, keep_first=0)
    layer.rt = SimpleNamespace(ops=ops, device=torch.device("cpu"))
    return layer


def test_layers_of_other_groups_in_one_step():
    """Query heads a key/value head decide whether single tokens take their own form: a layer's answer is not another's."""
    for first, then in ((8, 1), (1, 8)):
        batch = batch_of([1, 1, 1], [40, 300, 7])
        for kv_heads in (first, then):
            single, tiles = layer_of(32, kv_heads)._items(batch)
            assert (single is not None) == (kv_heads == 8) and (tiles is not None) == (kv_heads == 1)


def test_space_for_scores_is_bounded():
    """Many requests behind long contexts, as a recorded step of theirs keeps it: no more than the bound, or one token's scores."""
    for requests, context in ((256, 8192), (512, 4096), (64, 100_000), (1, 1_000_000)):
        (scores, stats, partial), _ = layer_of(32, 8)._items(batch_of([1] * requests, [context] * requests))
        one = -(-context // ops.MIXED_SINGLE_KEYS) * ops.MIXED_SINGLE_KEYS * 32 * 4
        assert scores.numel() * 4 <= max(64 << 20, one) and scores.numel() * 4 >= one
        # four workgroups a compute unit at a time, or one for each token of a share
        assert stats.shape[0] == partial.shape[1] == scores.shape[0] and partial.shape[0] * partial.shape[1] < 1024 + partial.shape[1]


def test_single_tokens_beside_a_portion():
    """They ride along in the portion's tiles until they are work enough for launches of their own; alone they always have those."""
    layer = layer_of(32, 8)
    for tokens, context, rows, own in ((1, 60, 40, False), (236, 60, 40, False), (237, 60, 40, True), (99, 1000, 40, False), (100, 1000, 40, True),
                                       (1, 6336, 40, False), (1, 6337, 40, True), (236, 60, 1000, False), (237, 60, 1000, True)):
        single, tiles = layer._items(batch_of([1] * tokens + [rows], [context] * tokens + [rows]))
        assert (single is not None) == own and tiles is not None
        entries = tiles[0][0].tolist()
        assert set(entries) == ({tokens} if own else set(range(tokens + 1)))
        single, tiles = layer._items(batch_of([1] * tokens, [context] * tokens))
        assert single is not None and tiles is None


def test_work_of_single_tokens_is_their_own_contexts():
    """One long context among short ones is not what all of them see: 90 tokens behind 300 to 1,200 keys are less work than 90 behind 1,200."""
    layer = layer_of(32, 8)
    for contexts, own in (([1200] * 90, True), ([300] * 89 + [1200], False)):
        single, tiles = layer._items(batch_of([1] * 90 + [40], contexts + [40]))
        assert (single is not None) == own


def test_runs_of_tiles():
    """Every tile's keys go into 1 to 16 runs none of which is empty, the longest runs come first and a tile's lie together; a
    prompt fills whole rounds of the chip rather than a round and a part."""
    for q_len, ctx_len in (([1500], [1500]), ([16], [16]), ([17, 40], [3000, 40]), ([700] * 3, [700, 1400, 9000]), ([2], [2])):
        layer = layer_of(32, 8)
        layer.spec.v_head_dim = 128
        _, (lists, n, row_splits, most, _) = layer._items(batch_of(q_len, ctx_len))
        entry, row0, split, runs = (x.tolist() for x in lists)
        at, before, seen = 0, None, {}
        while at < n:
            r = runs[at]
            assert 1 <= r <= 16 and split[at:at + r] == list(range(r)) and {(e, t) for e, t in zip(entry[at:at + r], row0[at:at + r])} == {(entry[at], row0[at])}
            e = entry[at]
            rows = min(16, q_len[e] - row0[at])
            keys = -(-(ctx_len[e] - q_len[e] + row0[at] + rows) // 32)
            length = -(-keys // r)
            assert before is None or length <= before
            before = length
            seen[(e, row0[at])] = r
            first = sum(q_len[:e]) + row0[at]
            assert row_splits[first:first + rows].tolist() == [r] * rows
            at += r
        assert at == n and most == max(runs) and set(seen) == {(e, t) for e, m in enumerate(q_len) for t in range(0, m, 16)}
    tiles = [-(-min(r + 16, 1500) // 32) for r in range(0, 1500, 16)]
    assert 200 < sum(ops.mixed_tile_runs(tiles, 256, 2)) <= 256


def _runs_cut_by_cut(key_tiles, units, slices):
    """`mixed_tile_runs` as it is defined: every cut's rounds walked one after the other."""
    longest, best = max(key_tiles), None
    for most in range(1, min(ops.MIXED_MOST_RUNS, longest) + 1):
        chunk = -(-longest // most)
        items = {}
        for n in key_tiles:
            runs = -(-n // chunk)
            items[-(-n // runs)] = items.get(-(-n // runs), 0) + runs
        total, at, turn = sum(items.values()), 0, 0
        cost = ops.MIXED_ITEM * total + (ops.MIXED_SUMS if most > 1 else 0.0)
        start = ops.MIXED_ROUND_SLICED if slices > 1 and total * slices <= units else ops.MIXED_ROUND
        for length in sorted(items, reverse=True):
            at += items[length]
            while turn < at:
                cost += start + length
                turn += units
        if best is None or cost < best[0] - 1e-9:
            best = (cost, chunk)
    return [-(-n // best[1]) for n in key_tiles]


def _key_tiles(rows, behind, window=None):
    ends = [(behind + at, behind + min(at + 16, rows) - 1) for at in range(0, rows, 16)]
    return [last // 32 - (max(0, first - window + 1) // 32 if window else 0) + 1 for first, last in ends]


def test_runs_of_tiles_are_the_cheapest_cut():
    rng = random.Random(3)
    for _ in range(300):
        tiles = sum((_key_tiles(rng.randint(1, int(2 ** rng.uniform(1, 11))), rng.choice([0, rng.randint(0, 9000)]), rng.choice([None, 512]))
                     for _ in range(rng.randint(1, 3))), [])
        slices = rng.choice([1, 2, 4])
        assert ops.mixed_tile_runs(tiles, 256, slices) == _runs_cut_by_cut(tiles, 256, slices)


def test_runs_of_a_long_prompt_are_found_quickly():
    """Host work between a step's first launches: all cuts at once take a fraction of one cut after the other (a fifth here; half is asked for)."""
    tiles = _key_tiles(2048, 6000)

    def least(f):
        took = []
        for _ in range(20):
            start = time.perf_counter()
            f(tiles, 256, 2)
            took.append(time.perf_counter() - start)
        return min(took)
    assert least(ops.mixed_tile_runs) < 0.5 * least(_runs_cut_by_cut)


def test_runs_fill_a_round():
    """One round of workgroups where a window's few tiles of keys are cut further, and a context of two tiles is not cut."""
    assert sum(ops.mixed_tile_runs(_key_tiles(1000, 3000, 512), 256, 1)) == 252
    assert ops.mixed_tile_runs(_key_tiles(64, 0), 256, 1) == [1] * 4
