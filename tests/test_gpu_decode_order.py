"""Decode attention over whole contexts where a launch has more than 256 workgroups: its tokens are folded (every second run of 256 workgroups the
other way round), and neither that nor the order of the rows changes a bit."""
import math

import numpy as np
import pytest
import torch

from kipp_amd.engine.batch import StepEntry, build_batch

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("n_q,n_kv,tokens", [(32, 8, 33), (32, 8, 64), (32, 8, 65), (8, 2, 129), (12, 3, 90), (16, 16, 37)])
def test_folded_launches_give_every_token_its_own_bits(n_q, n_kv, tokens):
    """Against launches of few enough tokens that nothing is folded; rows as they come, by length, and in no order."""
    from kipp_amd.csrc import ops
    d, page, group = 128, 16, n_q // n_kv
    assert ops.attention_decode_streams(tokens, n_kv, d, group, page, 700, 0)
    rng = np.random.default_rng(tokens + n_kv)
    lens = rng.integers(1, 700, tokens)
    blocks = [-(-int(n) // page) for n in lens]
    pages = rng.permutation(sum(blocks)).tolist()
    table = np.zeros((tokens, max(blocks)), dtype=np.int32)
    for i, b in enumerate(blocks):
        table[i, :b] = [pages.pop() for _ in range(b)]
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    k, v = (torch.randn((sum(blocks), n_kv, page, d), device=DEV, generator=gen).bfloat16() for _ in range(2))
    q = torch.randn((tokens, n_q * d), device=DEV, generator=gen).bfloat16()
    i32 = lambda a: torch.tensor(np.asarray(a), dtype=torch.int32, device=DEV)
    positions, seq_of, tables = i32(lens - 1), i32(np.arange(tokens)), i32(table)

    def run(rows, out):
        ws = ops.attention_decode_workspace(len(rows), n_q, d, 700, DEV)
        return ops.attention_decode(q, k, v, out, i32(rows), positions, seq_of, tables, n_q, n_kv, d, 1 / math.sqrt(d), 0, 700, ws)
    few = -(-160 // n_kv)               # tokens that a launch over whole contexts needs at least
    assert few * n_kv <= 256
    want = torch.zeros((tokens, n_q * d), dtype=torch.bfloat16, device=DEV)
    for at in range(0, tokens, few):
        run([min(i, tokens - 1) for i in range(at, at + few)], want)       # (the last row again: the same bits)
    for rows in (np.arange(tokens), np.argsort(-lens, kind="stable"), rng.permutation(tokens)):
        assert torch.equal(run(rows, torch.zeros_like(want)), want)


class _Request:
    def __init__(self, length):
        self.length, self.slot, self.tables = length, 0, [[0] * (length // 16 + 1)]


def test_a_batch_lists_single_tokens_by_their_contexts():
    lengths = [5, 90, 17, 90, 3, 40]
    entries = [StepEntry(str(i), [1] * (3 if i == 2 else 1), [0]) for i in range(len(lengths))]
    batch = build_batch(entries, [_Request(n) for n in lengths], 1, torch.device("cpu"))
    assert batch.decode_rows.tolist() == [1, 5, 7, 0, 6]         # (entry 2 brings rows 2, 3 and 4)
    assert [int(batch.positions[r]) for r in batch.decode_rows] == [90, 90, 40, 5, 3] and batch.n_decode == 5
