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


@pytest.mark.gpu
@pytest.mark.parametrize("arrivals", [True, False])
@pytest.mark.parametrize("n_q,n_kv,tokens,longest,window", [
    (32, 8, 33, 900, 0), (32, 8, 65, 800, 0), (16, 16, 37, 600, 0),             # whole contexts, a last run of one token, of one and two, of five
    (32, 8, 40, 2500, 600), (12, 3, 90, 1500, 520),                             # a window that straddles an edge of its ranges of 1,024 keys
    (8, 8, 33, 4700, 0), (16, 16, 17, 9000, 5000)])                             # two ranges and more
def test_folded_launches_in_every_form(n_q, n_kv, tokens, longest, window, arrivals):
    """From the projection (norm, rotation, the new keys and values written) and from queries, ranges merged by the last workgroup or by a launch,
    rows in either order: the bits of launches of few enough tokens that nothing is folded."""
    from kipp_amd.csrc import ops
    d, page = 128, 16
    few = -(-160 // n_kv)
    assert ops.attention_decode_streams(tokens, n_kv, d, n_q // n_kv, page, longest, window) and tokens * n_kv > 256 >= few * n_kv
    rng = np.random.default_rng(tokens + longest)
    lens = rng.integers(longest // 4, longest + 1, tokens)
    lens[:3] = 1, longest, min(longest, 4097)
    blocks = [-(-int(n) // page) for n in lens]
    pages = rng.permutation(sum(blocks)).tolist()
    table = np.zeros((tokens, max(blocks)), dtype=np.int32)
    for i, b in enumerate(blocks):
        table[i, :b] = [pages.pop() for _ in range(b)]
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    rand = lambda *shape: torch.randn(shape, device=DEV, generator=gen)  # noqa: E731
    k, v = (rand(sum(blocks), n_kv, page, d).bfloat16() for _ in range(2))
    qkv, norms = rand(tokens, (n_q + 2 * n_kv) * d), 1 + 0.1 * rand(2, d)
    inv_freq = torch.tensor(np.power(1e6, -(2.0 * np.arange(d // 2)) / d), dtype=torch.float32, device=DEV)
    i32 = lambda a: torch.tensor(np.asarray(a), dtype=torch.int32, device=DEV)  # noqa: E731
    args = (i32(lens - 1), i32(np.arange(tokens)), i32(table), n_q, n_kv, d)
    new = lambda: torch.zeros((tokens, n_q * d), dtype=torch.bfloat16, device=DEV)  # noqa: E731

    def space(n):
        return ops.attention_decode_workspace(n, n_q, d, longest, DEV)[:3 if arrivals else 2]
    k1, v1 = k.clone(), v.clone()
    q = ops.qk_norm_rope_kv_write(qkv, new(), k1, v1, *args, norms[0], norms[1], 1e-6, inv_freq, d, write_kv=True)
    run = lambda rows, out: ops.attention_decode(q, k1, v1, out, i32(rows), *args, 1 / math.sqrt(d), window, longest, space(len(rows)))  # noqa: E731
    want = new()
    for at in range(0, tokens, few):
        run([min(i, tokens - 1) for i in range(at, at + few)], want)
    for rows in (np.argsort(-lens, kind="stable"), rng.permutation(tokens)):
        assert torch.equal(run(rows, new()), want)
        for major in (False, True):
            k2, v2 = k.clone(), v.clone()
            got = ops.attention_decode_fused(qkv, k2, v2, new(), i32(rows), *args, norms[0], norms[1], 1e-6, inv_freq, d, True, 1 / math.sqrt(d), window,
                                             longest, space(tokens), out_steps_major=major)
            assert torch.equal(ops.from_steps_major(got) if major else got, want) and torch.equal(k2, k1) and torch.equal(v2, v1)


class _Request:
    def __init__(self, length):
        self.length, self.slot, self.tables = length, 0, [[0] * (length // 16 + 1)]


def test_a_batch_lists_single_tokens_by_their_contexts():
    lengths = [5, 90, 17, 90, 3, 40]
    entries = [StepEntry(str(i), [1] * (3 if i == 2 else 1), [0]) for i in range(len(lengths))]
    batch = build_batch(entries, [_Request(n) for n in lengths], 1, torch.device("cpu"))
    assert batch.decode_rows.tolist() == [1, 5, 7, 0, 6]         # (entry 2 brings rows 2, 3 and 4)
    assert [int(batch.positions[r]) for r in batch.decode_rows] == [90, 90, 40, 5, 3] and batch.n_decode == 5
