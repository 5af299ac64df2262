"""The mixed-head attention's form for single tokens, by itself: against the written-out float64 form, over groupings, windows with
kept first keys, contexts of one tile of keys to many, and cuts into more runs than there are tiles."""
import numpy as np
import pytest

from tests.test_gpu_tobinex import KERNEL_TOL, MixerCase, close

pytestmark = pytest.mark.gpu


def single_run(case, monkeypatch, queries, runs=None, slabs=1, longest=None):
    """`case.run` for single tokens with the form for them in the place of the tiles of rows."""
    import torch
    from kipp_amd.csrc import ops

    def single(q, k_cache, v_cache, out, items, n_items, row_splits, most, q_start, q_len, ctx_len, table, n_q, n_kv, d, dv, scale, window,
               keep, r1, r2, sink, mix, space, gate=None, gate_at=0):
        n = q.shape[0]
        tiles, planned = ops.mixed_single_plan(n, longest or int(ctx_len.max()), window, keep)
        assert ops.mixed_single_ok(n_q, n_kv, n, tiles)
        work = ops.mixed_single_workspace(n, n_q, dv, tiles, runs or planned, q.device)
        for t in work:
            t.fill_(float("nan"))               # nothing unwritten is read
        rows = torch.arange(n, dtype=torch.int32, device=q.device)
        return ops.mixed_attention_single(q, k_cache, v_cache, out, rows, ctx_len - 1, rows, table, n_q, n_kv, d, dv, scale, window,
                                          keep, r1, r2, sink, mix, work, gate=gate, gate_at=gate_at)

    monkeypatch.setattr(ops, "mixed_attention_mfma", single)
    return case.run("bfloat16", True, queries=queries, slabs=slabs)


# (12 heads over 12: key/value heads beyond the waves; 16 over 1: a whole product's columns)
@pytest.mark.parametrize("runs", [None, 1, 7])
@pytest.mark.parametrize("geometry", [(4, 4, 32, 32, None, 0), (32, 8, 32, 16, 50, 2), (12, 12, 32, 64, 90, 70), (16, 1, 32, 16, None, 0),
                                      (6, 3, 32, 16, 64, 5), (2, 1, 96, 16, 16, 20), (9, 9, 32, 64, 1, 0)])
def test_single_tokens(monkeypatch, geometry, runs):
    H_, G, d, dv, window, keep = geometry
    case = MixerCase(H_, G, d, dv, window, keep, T=260, seed=H_)
    ref = case.plain(True)
    got, rows = single_run(case, monkeypatch, [0, 1, 15, 16, 62, 63, 64, 65, 127, 128, 129, 191, 192, 259], runs, slabs=3)
    close(got, ref[rows], KERNEL_TOL["bfloat16"], f"{geometry}/{runs}")


@pytest.mark.parametrize("off", ["bias", "sink", "mix", "gate"])
def test_each_mechanism_off(monkeypatch, off):
    case = MixerCase(6, 3, 32, 16, window=150, keep=4, T=200, seed=3, **{n: n != off for n in ("bias", "sink", "mix", "gate")})
    got, rows = single_run(case, monkeypatch, [0, 70, 199], longest=4000)       # planned for a longer context, as a recorded step is
    close(got, case.plain(True)[rows], KERNEL_TOL["bfloat16"], off)


def test_a_key_that_stands_out_at_every_edge(monkeypatch):
    window, keep, query = 70, 5, 199
    for key in sorted({query - window + 1, query - window, keep - 1, keep, 0, query, query - 1, 63, 64, 127, 128, 191, 192}):
        case = MixerCase(4, 2, 32, 16, window, keep, 260, seed=key).stand_out(key)
        ref = case.plain(True)
        assert (np.abs(ref[query]).max() > 20.0) == (query - key < window or key < keep)
        got, rows = single_run(case, monkeypatch, [query])
        close(got, ref[rows], KERNEL_TOL["bfloat16"] * 10, f"key {key}")


@pytest.mark.parametrize("tokens", [1, 3, 13, 14])
def test_some_tokens_at_a_time(monkeypatch, tokens):
    """Space for the scores of a few tokens only: they go one after another through it (14 tokens of up to five tiles of keys here)."""
    from kipp_amd.csrc import ops
    monkeypatch.setattr(ops, "MIXED_SINGLE_BYTES", tokens * 5 * 64 * 32 * 4)
    assert ops.mixed_single_tokens(14, 5) == {1: 1, 3: 3, 13: 7, 14: 14}[tokens]
    case = MixerCase(6, 3, 32, 16, None, 0, T=260, seed=5)
    got, rows = single_run(case, monkeypatch, [0, 1, 15, 16, 62, 63, 64, 65, 127, 128, 129, 191, 192, 259], slabs=2)
    close(got, case.plain(True)[rows], KERNEL_TOL["bfloat16"], tokens)
