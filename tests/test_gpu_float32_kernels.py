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
