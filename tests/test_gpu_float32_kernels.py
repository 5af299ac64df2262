"""The 32-bit product and the generic attention kernel where their forms meet: edges of tiles and of the runs of K, one
token among few and among many.  References in float64; bounds are those of float32 sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 2.0 ** -24


def _run_of(k):
    each = -(-k // 8)
    return -(-each // 32) * 32


@pytest.mark.parametrize("n, k", [(16, 32), (17, 31), (200, 256), (130, 257), (65, 1028), (2560, 640), (333, 2562)])
def test_product_rows_are_the_same_in_both_kernels(n, k):
    """Rows in every class of the dispatch (16, 32, 64 rows, several of 64, tiles) give the bits they have alone, within the
    bound of sums of `_run_of(k)` products and eight of those sums."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(n + k)
    rows = 700
    x, w = rng.normal(size=(rows, k)).astype(np.float32), rng.normal(size=(n, k)).astype(np.float32)
    xd, wd = torch.tensor(x, device=DEV), torch.tensor(w, device=DEV)
    full = ops.gemm_f32(xd, wd, torch.empty((rows, n), device=DEV))
    for lo, hi in [(0, 1), (5, 21), (30, 47), (100, 132), (7, 40), (600, 664), (63, 128), (0, 257), (699, 700)]:
        part = ops.gemm_f32(xd[lo:hi].contiguous(), wd, torch.empty((hi - lo, n), device=DEV))
        assert torch.equal(part, full[lo:hi]), (lo, hi)
    exact = x.astype(np.float64) @ w.astype(np.float64).T
    size = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert np.all(np.abs(full.cpu().numpy() - exact) <= (min(k, _run_of(k)) + 8) * EPS * size)
    wb = wd.bfloat16()
    got = ops.gemm_f32(xd[:70].contiguous(), wb, torch.empty((70, n), device=DEV))
    again = ops.gemm_f32(xd[:70].contiguous(), wb.float(), torch.empty((70, n), device=DEV))
    assert torch.equal(got, again)          # a weight in bfloat16 is widened exactly


@pytest.mark.parametrize("pieces", [0, 1, 2, 3, 5, 6, 7, 8, 11, 12, 13, 18, 19, 24, 25])
@pytest.mark.parametrize("m", [1, 16, 20])
def test_few_rows_over_every_number_of_pieces(m, pieces):
    """The kernel for few rows with up to twice and more of the 16-number pieces that it asks for ahead in the last run of K, whole and with a part
    of one behind them.  Bound as above."""
    import torch
    from kipp_amd.csrc import ops
    part = -(-max(pieces, 1) // 2) * 32
    for rest in (0, 4, 5):
        k = 7 * part + min(16 * pieces + rest, part) if pieces else rest + 1
        rng = np.random.default_rng(pieces + rest + m)
        x, w = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(37, k)).astype(np.float32)
        got = ops.gemm_f32(torch.tensor(x, device=DEV), torch.tensor(w, device=DEV), torch.empty((m, 37), device=DEV)).cpu().numpy()
        exact = x.astype(np.float64) @ w.astype(np.float64).T
        size = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
        assert np.all(np.abs(got - exact) <= (min(k, _run_of(k)) + 8) * EPS * size), k


@pytest.mark.parametrize("k", [1, 17, 31, 33, 127, 128, 129, 131, 190, 255, 256])
@pytest.mark.parametrize("m", [1, 16, 20, 40])
def test_few_rows_over_short_runs(m, k):
    """Both sides of where a run's pieces are asked for ahead, in either kind of weight, numbers four at a time and one at a time.  Bound as above."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(k + m)
    x, w = rng.normal(size=(m, k)).astype(np.float32), torch.tensor(rng.normal(size=(37, k)).astype(np.float32)).bfloat16().float().numpy()
    exact = x.astype(np.float64) @ w.astype(np.float64).T
    size = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    outs = []
    for dtype in (torch.float32, torch.bfloat16):
        outs.append(ops.gemm_f32(torch.tensor(x, device=DEV), torch.tensor(w, device=DEV, dtype=dtype), torch.empty((m, 37), device=DEV)).cpu().numpy())
    assert np.all(np.abs(outs[0] - exact) <= (min(k, _run_of(k)) + 8) * EPS * size)
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("m, n", [(17, 32), (33, 47), (49, 2579), (97, 2570), (350, 3001), (333, 2570), (200, 6155)])
@pytest.mark.parametrize("k", [40, 268])
def test_product_in_every_shape_of_tiles(m, n, k):
    """Sizes around the tiles of every kernel at a K of a step or two a run, with parts of tiles at both ends and of a step of K: every row
    as the kernel for up to 16 rows makes it, whose sums the test above holds to float64.  (The test below names every shape of tiles.)"""
    import torch
    from kipp_amd.csrc import ops
    gen = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=gen).to(DEV), torch.randn((n, k), generator=gen).to(DEV)
    full = ops.gemm_f32(x, w, torch.empty((m, n), device=DEV))
    for lo in sorted({0, m // 2, m - 16}):
        assert torch.equal(ops.gemm_f32(x[lo:lo + 16].contiguous(), w, torch.empty((min(16, m - lo), n), device=DEV)), full[lo:lo + 16]), lo


@pytest.mark.parametrize("m, n, form", [(33, 47, 22), (97, 2570, 23), (64, 6144, 42), (31, 9731, 42), (200, 6155, 43), (333, 2570, 44)])
@pytest.mark.parametrize("k", [1068, 1069])
def test_tiles_over_several_steps_of_k(m, n, form, k):
    """Every shape of tiles where a wave's run has more steps than are asked for ahead and the last run ends inside one; weights in both
    types, rows that begin anywhere (K of 1,069): every row as the kernel for up to 16 rows makes it."""
    import torch
    from kipp_amd.csrc import ops
    assert ops.gemm_f32_form(m, n, k) == form
    gen = torch.Generator().manual_seed(m + n + k)
    x, wf = torch.randn((m, k), generator=gen).to(DEV), torch.randn((n, k), generator=gen).to(DEV)
    for w in (wf, wf.bfloat16()):
        full = ops.gemm_f32(x, w, torch.empty((m, n), device=DEV))
        for lo in range(0, m, 16):
            part = x[lo:lo + 16].contiguous()
            assert torch.equal(ops.gemm_f32(part, w, torch.empty((len(part), n), device=DEV)), full[lo:lo + 16]), (w.dtype, lo)


@pytest.mark.parametrize("m, n, k, form", [(17, 32, 40, 2), (32, 2563, 268, 2), (31, 100, 500, 2), (19, 100, 201, 2), (33, 130, 31, 4), (130, 1000, 16, 4), (350, 3001, 40, 0), (333, 2570, 268, 0),
                                           (700, 2561, 257, 0), (2000, 1030, 33, 0)])
def test_products_of_a_short_k(m, n, k, form):
    """The kernels that short K goes through, at ends of tiles, steps and runs: every row as the kernel for up to 16 rows makes it."""
    import torch
    from kipp_amd.csrc import ops
    assert ops.gemm_f32_form(m, n, k) == form
    gen = torch.Generator().manual_seed(m + n + k)
    x, wf = torch.randn((m, k), generator=gen).to(DEV), torch.randn((n, k), generator=gen).to(DEV)
    for w in (wf, wf.bfloat16()):
        full = ops.gemm_f32(x, w, torch.empty((m, n), device=DEV))
        for lo in sorted({0, m // 32 * 16, m - 16}):
            part = x[lo:lo + 16].contiguous()
            assert torch.equal(ops.gemm_f32(part, w, torch.empty((16, n), device=DEV)), full[lo:lo + 16]), (w.dtype, lo)


def test_product_of_rows_that_begin_anywhere():
    """Operands at addresses that 16-byte loads do not take."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(0)
    m, n, k = 70, 50, 64
    store = torch.tensor(rng.normal(size=m * k + n * k + 8).astype(np.float32), device=DEV)
    x, w = store[1:1 + m * k].view(m, k), store[3 + m * k:3 + m * k + n * k].view(n, k)
    got = ops.gemm_f32(x, w, torch.empty((m, n), device=DEV))
    assert torch.equal(got, ops.gemm_f32(x.clone(), w.clone(), torch.empty((m, n), device=DEV)))


@pytest.mark.parametrize("n_q, n_kv, d, dv, shared, page, window, chunk", [
    (8, 2, 128, 128, False, 16, 0, 0), (6, 3, 20, 20, False, 8, 0, 0), (3, 1, 33, 17, False, 16, 70, 0), (16, 1, 576, 512, True, 16, 0, 0),
    (4, 1, 256, 256, False, 32, 0, 0), (6, 1, 64, 130, False, 16, 0, 100), (2, 2, 40, 1000, False, 16, 0, 0)])
def test_attention_of_a_token_alone_and_among_others(n_q, n_kv, d, dv, shared, page, window, chunk):
    """Tokens at the edges of the blocks of 64 keys, alone (several waves share the keys), among a few and among enough
    for a wave each: the same bits, against the softmax in float64."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(d + dv)
    length = 450
    blocks = -(-length // page)
    order = rng.permutation(blocks + 2)[:blocks]
    pages = blocks + 2
    k = rng.normal(size=(pages, n_kv, page, d)).astype(np.float32)
    v = k if shared else rng.normal(size=(pages, n_kv, page, dv)).astype(np.float32)
    keys = k[order].transpose(0, 2, 1, 3).reshape(-1, n_kv, d)[:length].astype(np.float64)
    values = v[order].transpose(0, 2, 1, 3).reshape(-1, n_kv, v.shape[3])[:length, :, :dv].astype(np.float64)
    where = [0, 1, 62, 63, 64, 127, 128, 200, 319, 320, 448, 449]
    many = -(-8200 // (n_q // 4 or 1))
    positions = np.array(where + [int(p) for p in rng.integers(0, length, many)], dtype=np.int32)
    q = rng.normal(size=(len(positions), n_q * d)).astype(np.float32)
    kd = torch.tensor(k, device=DEV)
    vd = kd if shared else torch.tensor(v, device=DEV)
    table = torch.tensor(order[None], dtype=torch.int32, device=DEV)
    scale = d ** -0.5

    def run(rows):
        pos = torch.tensor(positions[rows], device=DEV)
        return ops.paged_attention_wide(torch.tensor(q[rows], device=DEV), kd, vd, torch.empty((len(rows), n_q * dv), device=DEV), pos,
                                        torch.zeros_like(pos), table, n_q, n_kv, d, dv, scale, window=window, chunk=chunk, sink=True).cpu().numpy()
    every = run(np.arange(len(positions)))
    few = run(np.arange(300))
    assert np.array_equal(few, every[:300])
    for i, p in enumerate(where):
        assert np.array_equal(run(np.array([i])), every[i:i + 1]), p
        lo = p - p % chunk if chunk else (max(0, p - window + 1) if window else 0)
        for h in range(n_q):
            g = h // (n_q // n_kv)
            s = keys[lo:p + 1, g] @ q[i, h * d:(h + 1) * d].astype(np.float64) * scale
            top = max(s.max(), 0.0)
            e = np.exp(s - top)
            p_ = e / (e.sum() + np.exp(-top))
            # a score is off by d products of float32, which moves a weight by as much; then p + 1 weighted values
            moved = 2 * d * EPS * scale * (np.abs(keys[lo:p + 1, g]) @ np.abs(q[i, h * d:(h + 1) * d])).max() + (p + 20) * EPS
            bound = 2 * moved * (p_ @ np.abs(values[lo:p + 1, g]))
            assert np.all(np.abs(every[i, h * dv:(h + 1) * dv] - p_ @ values[lo:p + 1, g]) <= bound + 1e-30), (p, h)


@pytest.mark.parametrize("block", [0, 1, 3, 6])
@pytest.mark.parametrize("tokens", [1, 300, 4200])
def test_a_block_of_keys_whose_scores_overflow(block, tokens):
    """64 keys of one block score -inf: they weigh nothing, wherever the block lies and however many waves share the keys."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(block)
    length, d, n_q, page = 450, 16, 2, 16
    k, v = rng.normal(size=(length, d)).astype(np.float32), rng.normal(size=(length, d)).astype(np.float32)
    q = rng.normal(size=(tokens, n_q, d)).astype(np.float32)
    k[:, 0], q[:, :, 0] = 0.0, 2e38
    k[64 * block:64 * (block + 1), 0] = -2e38
    seen = np.arange(length) // 64 != block
    cache = lambda a: torch.tensor(np.concatenate([a, np.zeros((-length % page, d), dtype=np.float32)]).reshape(-1, 1, page, d), device=DEV)  # noqa: E731
    i32 = lambda a: torch.tensor(np.asarray(a), dtype=torch.int32, device=DEV)  # noqa: E731
    out = ops.paged_attention_wide(torch.tensor(q.reshape(tokens, -1), device=DEV), cache(k), cache(v), torch.empty((tokens, n_q * d), device=DEV),
                                   i32(np.full(tokens, length - 1)), i32(np.zeros(tokens)), i32(np.arange(-(-length // page)))[None], n_q, 1, d, d, 0.25)
    s = q[:, :, 1:].astype(np.float64) @ k[seen, 1:].astype(np.float64).T * 0.25
    p = np.exp(s - s.max(axis=-1, keepdims=True))
    ref = p / p.sum(axis=-1, keepdims=True) @ v[seen].astype(np.float64)
    # scores of size up to ~ 10, off by d float32 products; weights likewise, then `length` weighted values of size up to ~ 4
    assert np.all(np.abs(out.cpu().numpy().reshape(ref.shape) - ref) <= (10 * d + length) * EPS * 4)
