"""Attention of single tokens over rows that are key and value at once: against the written-out float64 form."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def attend(q, rows, pos, window, scale):
    lo = max(0, pos - window + 1) if window else 0
    k = rows[lo:pos + 1]
    s = q @ k.T * scale
    p = np.exp(s - s.max(axis=1, keepdims=True))
    return (p / p.sum(axis=1, keepdims=True)) @ k


# rows of half a product step, of odd steps, of the widest; every count of heads' edge; positions on both sides of tile and page edges
@pytest.mark.parametrize("d", [16, 48, 80, 224, 256])
@pytest.mark.parametrize("heads", [1, 5, 16])
@pytest.mark.parametrize("window,page", [(0, 16), (100, 32), (1, 8), (64, 64)])
def test_shared_rows(d, heads, window, page, runs=None):
    from kipp_amd.csrc import ops
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(d + heads + window)
    T = 700
    at = [0, 1, 62, 63, 64, 65, 127, 128, 191, 192, 300, 511, 640, 699]
    blocks = -(-T // page)
    pages = rng.permutation(blocks + 3)[:blocks]
    rows = torch.tensor(rng.normal(size=(T, d)), dtype=torch.bfloat16)
    q = torch.tensor(rng.normal(size=(len(at), heads * d)), dtype=torch.bfloat16)
    cache = torch.full((blocks + 3, 1, page, d), float("nan"), dtype=torch.bfloat16)        # what is not written is not read
    for t in range(T):
        cache[pages[t // page], 0, t % page] = rows[t]
    i32 = lambda a: torch.tensor(np.asarray(a), dtype=torch.int32, device=dev)  # noqa: E731
    table = i32(np.tile(pages, (len(at), 1)))
    scale = 1.5 / np.sqrt(d)
    exact = np.stack([attend(q[i].double().numpy().reshape(heads, d), rows.double().numpy(), p, window, scale) for i, p in enumerate(at)])
    order = np.arange(len(at))[::-1].copy()         # the tokens' rows of the batch in another order than the items
    # one rounding to bfloat16; scores of size ~ 6 in float32 sums of d products: d 2^-24 of that in the exponent, twice over
    bound = 2.0 ** -8 * np.abs(exact) + 12 * d * 2.0 ** -24 * np.abs(rows.double().numpy()).max()
    for n_runs in (None, 1, 3, 64):
        work = ops.attention_shared_workspace(len(at), d, T, window, dev)
        if n_runs is not None:
            work = torch.empty((len(at), n_runs, 16, d), device=dev), torch.empty((len(at), n_runs, 16, 2), device=dev)
        for t in work:
            t.fill_(float("nan"))
        out = torch.zeros((len(at), heads * d), dtype=torch.bfloat16, device=dev)
        ops.attention_shared(q.to(dev), cache.to(dev), out, i32(order), i32(at), i32(np.arange(len(at))), table, heads, d, scale, window, work)
        got = out.double().cpu().numpy().reshape(len(at), heads, d)
        assert (np.abs(got - exact) <= bound).all(), (n_runs, np.abs(got - exact).max())


def test_refusals():
    from kipp_amd.csrc import ops
    dev = torch.device("cuda:0")
    i32 = torch.zeros(1, dtype=torch.int32, device=dev)
    bf = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16, device=dev)  # noqa: E731
    work = ops.attention_shared_workspace(1, 32, 64, 0, dev)
    with pytest.raises(ops.KernelError):
        ops.attention_shared(bf(1, 17 * 32), bf(1, 1, 16, 32), bf(1, 17 * 32), i32, i32, i32, i32.view(1, 1), 17, 32, 1.0, 0, work)
    with pytest.raises(ops.KernelError):
        ops.attention_shared(bf(1, 32), bf(1, 1, 12, 32), bf(1, 32), i32, i32, i32, i32.view(1, 1), 1, 32, 1.0, 0, work)
