"""Matrix memories over prompt portions, 64 tokens at a time, against the recurrence in float64 and beside the walk token by
token: entries shorter and longer than a chunk, from states kept in slots, every key size the kernel takes, columns that do
not fill a workgroup, decays of zero and one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = [64, 1, 65, 15, 16, 130, 17, 63, 200]


@pytest.fixture(autouse=True)
def chunks_wherever_an_entry_may_take_them(monkeypatch):
    """Here chunks are taken from their first token count on, not from where they are the faster way."""
    from kipp_amd.csrc import ops
    monkeypatch.setattr(ops, "matrix_chunks_from", lambda mode, d, state: ops.CHUNKS_FROM)


def _plain(mode, q, k, v, beta, g, s):
    """The recurrence over one head's tokens in float64: (o [T, dv], S [d, dv])."""
    out = np.zeros(v.shape)
    for t in range(len(v)):
        s = g[t] * s
        u = beta[t] * (v[t] - s.T @ k[t]) if mode == "delta" else v[t]
        s = s + np.outer(k[t], u)
        out[t] = s.T @ q[t]
    return out, s


def _off(got, ref):
    return np.linalg.norm(got - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("d, dv, heads, rep", [(64, 16, 3, 1), (128, 40, 4, 2), (192, 8, 2, 2), (256, 33, 2, 1)])
@pytest.mark.parametrize("mode", ["decay", "delta", "gated"])
def test_chunks_beside_the_walk(mode, d, dv, heads, rep):
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(d + dv)
    rep = 1 if mode == "decay" else rep
    kv, tokens, n = heads // rep, sum(LENGTHS), len(LENGTHS)
    starts = np.concatenate([[0], np.cumsum(LENGTHS)[:-1]])
    q, k = rng.normal(size=(tokens, kv, d)), rng.normal(size=(tokens, kv, d))
    v = rng.normal(size=(tokens, heads, dv))
    beta = rng.uniform(0.05, 1.0, size=(tokens, heads))
    g = np.exp(-np.exp(rng.normal(size=heads) - 2.0) * rng.uniform(0.0, 1.5, size=(tokens, heads)))
    g[rng.integers(0, tokens, 6)] = 0.0
    g[rng.integers(0, tokens, 20)] = 1.0
    if mode == "decay":
        g = np.broadcast_to(rng.uniform(0.8, 1.0, size=heads), g.shape)
        g = np.where(np.arange(heads) == 0, 1.0, g)
    else:
        q, k = (x / np.linalg.norm(x, axis=-1, keepdims=True) for x in (q, k))
    columns = {"decay": [q, k, v], "delta": [q, k, v, beta[..., None], g[..., None]], "gated": [q, k, v, v, g[..., None]]}[mode]
    src = np.concatenate([c.reshape(tokens, -1) for c in columns], axis=1).astype(np.float32)
    src = np.concatenate([src, np.zeros((tokens, -src.shape[1] % 4), dtype=np.float32)], axis=1)
    if mode == "decay":
        silu = lambda x: np.float32(x).astype(np.float64) / (1.0 + np.exp(-np.float32(x).astype(np.float64)))  # noqa: E731
        qe, ke, ve = silu(q), silu(k), silu(v)
    else:
        qe, ke, ve = (np.float32(x).astype(np.float64) for x in (q, k, v))
    ge, be = np.float32(g).astype(np.float64), np.float32(beta).astype(np.float64)
    size = -(-heads * d * dv // 4) * 4 + 8
    kept = np.zeros((n + 1, size), dtype=np.float32)
    slots = rng.permutation(n + 1)[:n]
    kept[slots[1:], :heads * d * dv] = rng.normal(size=(n - 1, heads * d * dv))         # the first entry starts from zeros
    dev = lambda a, ty: torch.tensor(a, dtype=ty, device=DEV)  # noqa: E731
    i32 = torch.int32
    results = {}
    for chunks in (False, True):
        state, o = dev(kept, torch.float32), torch.full((tokens, heads * dv), float("nan"), device=DEV)
        where = (state, dev(starts, i32), dev(LENGTHS, i32), dev(slots, i32), o)
        if mode == "decay":
            ops.decay_scan(dev(src, torch.float32), dev(g[0], torch.float32), *where, heads, d, dv, longest=max(LENGTHS), chunks=chunks)
        elif mode == "delta":
            ops.delta_scan(dev(src, torch.float32), *where, heads, kv, d, dv, longest=max(LENGTHS), chunks=chunks)
        else:
            ops.gated_scan(dev(src, torch.float32), *where, heads, kv, d, dv, longest=max(LENGTHS), chunks=chunks)
        results[chunks] = o.cpu().numpy().astype(np.float64).reshape(tokens, heads, dv), state.cpu().numpy().astype(np.float64)
    for e in range(n):
        rows = slice(starts[e], starts[e] + LENGTHS[e])
        for h in range(heads):
            s0 = kept[slots[e], :heads * d * dv].astype(np.float64).reshape(heads, dv, d)[h].T
            ref, s = _plain(mode, qe[rows, h // rep], ke[rows, h // rep], ve[rows, h], be[rows, h], ge[rows, h], s0)
            off = {c: (_off(results[c][0][rows, h], ref), _off(results[c][1][slots[e], :heads * d * dv].reshape(heads, dv, d)[h].T, s)) for c in results}
            # both are float32 sums of d products and of the tokens so far: a few hundred roundings of 2^-24, half of them
            # cancelled; the chunks add in shorter chains than the walk
            for i in range(2):
                assert off[True][i] < 4e-6 and off[True][i] < 2.0 * off[False][i] + 3e-7, (e, h, off)
    spare = [i for i in range(n + 1) if i not in slots][0]
    assert not results[True][1][spare].any() and np.array_equal(results[True][1][:, heads * d * dv:], kept[:, heads * d * dv:])


def test_few_tokens_and_other_sizes_walk():
    """Entries of fewer tokens than a chunk pays for, and key sizes it does not take, give the walk's bits."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(0)
    for d, n in ((128, ops.CHUNKS_FROM - 1), (96, 70)):
        heads, dv = 2, 16
        src = torch.tensor(rng.normal(size=(n, heads * (2 * d + dv))).astype(np.float32), device=DEV)
        one = lambda v: torch.tensor([v], dtype=torch.int32, device=DEV)  # noqa: E731
        got = []
        for chunks in (False, True):
            state = torch.zeros((1, heads * d * dv), device=DEV)
            got.append(ops.decay_scan(src, torch.tensor([0.9, 1.0], device=DEV), state, one(0), one(n), one(0), torch.empty((n, heads * dv), device=DEV),
                                      heads, d, dv, longest=n, chunks=chunks))
        assert torch.equal(*got)


@pytest.mark.parametrize("mode", ["decay", "delta", "gated"])
def test_an_entry_beside_others_is_as_alone(mode):
    """Every entry of a launch by chunks, short or long, in any order of the entries, gives the bits it gives alone: the walk's below
    `CHUNKS_FROM` tokens, the chunks' from there on."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(1)
    d, dv, heads = 64, 24, 2
    lengths = [1, 70, 15, 16, 1, 1, 129, 0, 3] + [1] * 70 + [64]       # (more entries than a wave has lanes)
    tokens, n = sum(lengths), len(lengths)
    starts = np.concatenate([[0], np.cumsum(lengths)[:-1]])
    width = {"decay": heads * (2 * d + dv), "delta": heads * (2 * d + dv + 2), "gated": heads * (2 * d + 2 * dv + 1) + 2}[mode]
    src = rng.normal(size=(tokens, width)).astype(np.float32) * 0.3
    src[:, heads * (2 * d + dv):] = rng.uniform(0.3, 1.0, size=src[:, heads * (2 * d + dv):].shape)
    kept = rng.normal(size=(n, heads * d * dv)).astype(np.float32)
    dev = lambda a, ty=torch.float32: torch.tensor(np.asarray(a), dtype=ty, device=DEV)  # noqa: E731

    def run(rows, starts, lens, slots, chunks, portions):
        state, o = dev(kept), torch.zeros((len(rows), heads * dv), device=DEV)
        where = [state] + [dev(a, torch.int32) for a in (starts, lens, slots)] + [o]
        said = dict(longest=max(lens), chunks=chunks, portions=portions)
        if mode == "decay":
            ops.decay_scan(dev(src[rows]), dev([0.9, 0.99]), *where, heads, d, dv, **said)
        else:
            (ops.delta_scan if mode == "delta" else ops.gated_scan)(dev(src[rows]), *where, heads, heads, d, dv, **said)
        return o.cpu().numpy(), state.cpu().numpy()
    many = sum(m >= ops.CHUNKS_FROM for m in lengths)
    order = rng.permutation(n)
    together = [run(np.arange(tokens), starts[o], np.array(lengths)[o], o, True, portions) for o in (np.arange(n), order) for portions in (None, many)]
    for o, state in together[1:]:
        assert np.array_equal(o, together[0][0]) and np.array_equal(state, together[0][1])
    for e in [0, 1, 2, 3, 6, 8, 40, n - 1]:
        rows = np.arange(starts[e], starts[e] + lengths[e])
        o, state = run(rows, [0], [lengths[e]], [e], lengths[e] >= ops.CHUNKS_FROM, None)
        assert np.array_equal(o, together[0][0][rows]) and np.array_equal(state[e], together[0][1][e]), e
