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


@pytest.mark.parametrize("d, dv, heads", [(64, 16, 3), (128, 40, 2), (192, 31, 2), (256, 33, 1)])
def test_mlstm_chunks_beside_the_walk(d, dv, heads):
    """The mLSTM's running maximum, normalizer and floor by chunks: entries longer than the gates' turn of 1,024 tokens and shorter than
    what chunks take, from states that the walk left, a column of n beside whole and partial tiles of columns.  Both forms against
    float64; S, every copy of n and m as the walk leaves them."""
    import torch
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(d)
    cap, lengths = 15.0, [64, 1, 65, 15, 16, 1100]
    tokens, n = sum(lengths), len(lengths)
    starts = np.concatenate([[0], np.cumsum(lengths)[:-1]]).astype(np.int32)
    width = 2 * heads * d + 2 * heads * dv + 2 * heads
    proj = rng.normal(size=(tokens, width + -width % 4)).astype(np.float32)
    proj[:, width - 2 * heads:width] *= 4.0
    bi, bf = rng.normal(size=heads).astype(np.float32), (2.0 + rng.normal(size=heads)).astype(np.float32)
    to = lambda x: torch.tensor(x, device=DEV)  # noqa: E731
    args = lambda p, state, o, at, count, slots: (to(p), to(bi), to(bf), cap, state, to(at), to(count), to(slots), o, heads, d, dv)  # noqa: E731
    size, slots = ops.mlstm_state_size(heads, d, dv), np.arange(n, dtype=np.int32)[::-1].copy()
    before = torch.zeros((n, size), device=DEV)
    lead = rng.normal(size=(n, proj.shape[1])).astype(np.float32)
    ops.mlstm_scan(*args(lead, before, torch.empty((n, heads * dv), device=DEV), np.arange(n, dtype=np.int32), np.ones(n, dtype=np.int32), slots))
    walked, chunked = before.clone(), before.clone()
    o_walk, o = (torch.full((tokens, heads * dv), np.nan, device=DEV) for _ in range(2))
    lens = np.array(lengths, dtype=np.int32)
    ops.mlstm_scan(*args(proj, walked, o_walk, starts, lens, slots))
    den, below = ops.mlstm_chunks(*args(proj, chunked, o, starts, lens, slots), longest=max(lengths), portions=4)
    assert below == ops.CHUNKS_FROM
    ops.mlstm_scan(*args(proj, chunked, o, starts, lens, slots), below=below)
    got = (o.view(tokens, heads, dv) / den[:, :, None]).double().cpu().numpy()
    o_walk, walked, chunked = o_walk.view(tokens, heads, dv).double().cpu().numpy(), walked.double().cpu().numpy(), chunked.double().cpu().numpy()
    q, k, v = (proj[:, a:b].reshape(tokens, heads, -1).astype(np.float64) for a, b in ((0, heads * d), (heads * d, 2 * heads * d), (2 * heads * d, 2 * heads * d + heads * dv)))
    z = proj[:, width - 2 * heads:width].astype(np.float64)
    li, lf = (cap * np.tanh((z[:, a:a + heads] + b) / cap) for a, b in ((0, bi), (heads, bf)))
    lf = -np.logaddexp(0.0, -lf)
    copies = (size - heads * d * dv) // (heads * d + heads)
    before = before.double().cpu().numpy()
    for i in range(n):
        at, state, row = slice(starts[i], starts[i] + lengths[i]), before[slots[i]], slots[i]
        n_all, m_all = heads * d * dv, heads * d * dv + copies * heads * d
        for h in range(heads):
            size_s, size_n = 0.0, 0.0       # the same sums over the numbers' sizes
            s, nv, m = state[h * dv * d:(h + 1) * dv * d].reshape(dv, d).T, state[n_all + h * d:n_all + (h + 1) * d], state[m_all + h]
            ref, bound = np.zeros((lengths[i], dv)), np.zeros((lengths[i], dv))
            for j, t in enumerate(range(at.start, at.stop)):
                new = max(lf[t, h] + m, li[t, h])
                keep, take, m = np.exp(lf[t, h] + m - new), np.exp(li[t, h] - new), new
                s, nv = keep * s + take * np.outer(k[t, h], v[t, h]), keep * nv + take * k[t, h]
                qt = q[t, h] * d ** -0.5
                size_s, size_n = keep * size_s + take * np.abs(np.outer(k[t, h], v[t, h])), keep * size_n + take * np.abs(k[t, h])
                den = max(abs(nv @ qt), np.exp(-m)) + 1e-6
                ref[j] = s.T @ qt / den
                # numerator and denominator each off by less than 64 roundings of the sums of their terms' sizes (runs of up to 32
                # terms in one chain, 16 in the next, and the roundings of gates and decays)
                bound[j] = 64 * 2.0 ** -24 * (size_s.T + np.abs(ref[j])[:, None] * size_n) @ np.abs(qt) / den + 1e-6 * np.abs(ref[j])
            assert np.all(np.abs(got[at, h] - ref) <= bound), (i, h)
            assert np.all(np.abs(o_walk[at, h] - ref) <= bound), (i, h)
            for c in range(copies):
                assert _off(chunked[row, n_all + (c * heads + h) * d:n_all + (c * heads + h + 1) * d], nv) <= 4e-6, (i, h, c)
                assert abs(chunked[row, m_all + c * heads + h] - m) <= 4e-6 * max(1.0, abs(m)), (i, h, c)
            assert _off(chunked[row, h * dv * d:(h + 1) * dv * d].reshape(dv, d), s.T) <= 4e-6, (i, h)


@pytest.mark.parametrize("d, dv, heads", [(40, 5, 2), (64, 16, 3), (128, 320, 2), (96, 33, 1), (88, 300, 8)])
def test_mlstm_single_tokens_have_the_walks_bits(d, dv, heads):
    """Steps of single tokens, an entry without one among them: results, S, every copy of n and of m as the walk leaves them."""
    import torch
    from kipp_amd.csrc import ops
    gen = torch.Generator().manual_seed(d)
    n, size = 5, ops.mlstm_state_size(heads, d, dv)
    width = 2 * heads * d + 2 * heads * dv + 2 * heads
    width += -width % 4
    b = torch.randn((2, heads), generator=gen).to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    states = [torch.zeros((n + 1, size), device=DEV) for _ in range(2)]
    for step in range(3):
        proj = torch.randn((n, width), generator=gen).to(DEV)
        got = []
        for state, single in zip(states, (False, True)):
            o = torch.zeros((n, heads * dv), device=DEV)
            # (the walk takes every entry with a token; an entry without one is left alone by the other form)
            entries = [0, 1, 3, 4] if not single else [0, 1, 2, 3, 4]
            lens = [0 if e == 2 else 1 for e in entries]
            got.append(ops.mlstm_scan(proj, b[0], b[1], 15.0, state, i32(entries), i32(lens), i32([5 - e for e in entries]), o, heads, d, dv, few=True, single=single))
        assert torch.equal(*got) and torch.equal(*states), step


@pytest.mark.parametrize("d", [64, 128])
def test_mlstm_entries_beyond_the_portions_are_left_alone(d):
    """Fewer `portions` than entries that bring so many tokens: the first are as they are without the others, and of the others neither
    S nor n nor m moves."""
    import torch
    from kipp_amd.csrc import ops
    heads, dv, lens = 2, 20, [64, 1, 65, 64]
    gen = torch.Generator().manual_seed(d)
    proj = torch.randn((sum(lens), 2 * heads * (d + dv) + 2 * heads), generator=gen).to(DEV)
    bias = torch.randn((2, heads), generator=gen).to(DEV)
    kept = torch.randn((len(lens), ops.mlstm_state_size(heads, d, dv)), generator=gen).to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731

    def run(lens, portions):
        state, o = kept.clone(), torch.zeros((proj.shape[0], heads * dv), device=DEV)
        den, below = ops.mlstm_chunks(proj, bias[0], bias[1], 15.0, state, i32([0, 64, 65, 130][:len(lens)]), i32(lens), i32([3, 2, 1, 0][:len(lens)]), o, heads, d, dv,
                                      longest=65, portions=portions)
        assert below == ops.CHUNKS_FROM
        return state, o[:64], den[:65]
    some, alone = run(lens, 1), run(lens[:2], 1)
    for a, b in zip(some, alone):
        assert torch.equal(a, b)
    assert not torch.equal(some[0][3], kept[3]) and torch.equal(some[0][:3], kept[:3])


@pytest.mark.parametrize("heads, dv", [(1, 1), (5, 63), (8, 320), (3, 65)])
def test_mlstm_finish_with_and_without_a_division(heads, dv):
    """Sums that are still to be divided give the bits of divided ones, and those the norm, weight and gate of float64."""
    import torch
    from kipp_amd.csrc import ops
    gen = torch.Generator().manual_seed(dv)
    n, at = 7, 3
    o, proj, w = (torch.randn(shape, generator=gen).to(DEV) for shape in ((n, heads * dv), (n, at + heads * dv + 2), (heads * dv,)))
    den = torch.empty((n, heads)).uniform_(0.1, 20.0, generator=gen).to(DEV)
    o[0] = 0.0
    divided = (o.view(n, heads, dv) / den[:, :, None]).view(n, heads * dv)
    for dtype in (torch.float32, torch.bfloat16):
        out = [ops.mlstm_finish(sums, proj, at, w, 1e-6, torch.empty((n, heads * dv), dtype=dtype, device=DEV), heads, dv, den=d)
               for sums, d in ((o, den), (divided, None))]
        assert torch.equal(*out), dtype
        x = divided.double().view(n, heads, dv)
        ref = (x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt()).view(n, heads * dv) * w.double() * torch.sigmoid(proj.double()[:, at:at + heads * dv])
        # ten numbers a lane and six exchanges of the square's sum, a root, two quotients, an exponential and four products
        assert torch.all((out[0].double() - ref).abs() <= ref.abs() * (32 * 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -8))


@pytest.mark.parametrize("d, dv", [(20, 9), (128, 40), (200, 17), (300, 5), (600, 6)])
@pytest.mark.parametrize("few", [False, True])
def test_mlstm_walk_of_some_entries(d, dv, few):
    """`below`: the short entries' bits are those of a walk over every entry, the others' rows and states stay."""
    import torch
    from kipp_amd.csrc import ops
    gen = torch.Generator().manual_seed(d)
    heads, lens = 2, [3, 10, 9, 40]
    proj = torch.randn((sum(lens), 2 * heads * (d + dv) + 2 * heads), generator=gen).to(DEV)
    bias, kept = torch.randn((2, heads), generator=gen).to(DEV), torch.randn((len(lens), ops.mlstm_state_size(heads, d, dv)), generator=gen).to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    got = []
    for below in (0, 10):
        state, o = kept.clone(), torch.full((sum(lens), heads * dv), 7.0, device=DEV)
        ops.mlstm_scan(proj, bias[0], bias[1], 15.0, state, i32([0, 3, 13, 22]), i32(lens), i32([0, 1, 2, 3]), o, heads, d, dv, few=few and below > 0, below=below)
        got.append((o, state))
    (o, state), (o_some, state_some) = got
    for e, (at, n) in enumerate(zip((0, 3, 13, 22), lens)):
        if n < 10:
            assert torch.equal(o_some[at:at + n], o[at:at + n]) and torch.equal(state_some[e], state[e]), e
        else:
            assert bool((o_some[at:at + n] == 7.0).all()) and torch.equal(state_some[e], kept[e]), e


@pytest.mark.parametrize("mode, d", [("decay", 64), ("decay", 128), ("decay", 192), ("gated", 64), ("gated", 128), ("gated", 192), ("mlstm", 64), ("mlstm", 128),
                                     ("mlstm", 192), ("delta", 64)])
def test_many_portions_have_the_bits_of_few(mode, d):
    """Many workgroups of a walk go by four waves that do both, few by eight: the same bits, of portions of one, two and three chunks, whole
    and not."""
    import torch
    from kipp_amd.csrc import ops
    heads, dv = 40, 64
    lengths = [64, 65, 127, 128, 130, 150, 96, 192]
    tokens, n = sum(lengths), len(lengths)
    starts = np.concatenate([[0], np.cumsum(lengths)[:-1]])
    gen = torch.Generator(device=DEV).manual_seed(d)
    i32 = lambda x: torch.tensor(np.asarray(x), dtype=torch.int32, device=DEV)  # noqa: E731
    if mode == "mlstm":
        src = torch.randn(tokens, 2 * heads * d + 2 * heads * dv + 2 * heads, device=DEV, generator=gen)
        bias, size = torch.randn(heads, device=DEV, generator=gen), ops.mlstm_state_size(heads, d, dv)
    elif mode == "decay":
        src = torch.randn(tokens, 2 * heads * d + heads * dv, device=DEV, generator=gen)
        decays, size = torch.rand(heads, device=DEV, generator=gen), heads * d * dv
    elif mode == "delta":
        src = torch.randn(tokens, heads * d + heads * dv + 2 * heads, device=DEV, generator=gen)
        src[:, :heads * d] *= d ** -0.5
        src[:, heads * d + heads * dv:].uniform_(0.5, 1.0, generator=gen)
        size = heads * d * dv
    else:
        src = torch.randn(tokens, ops.ssd_prep_width(heads, 1, d, dv), device=DEV, generator=gen)
        src[:, 2 * d + 2 * heads * dv:].uniform_(0.5, 1.0, generator=gen)
        size = heads * d * dv
    begin = torch.randn(n, size, device=DEV, generator=gen)

    def run(entries):
        state, o = begin.clone(), torch.full((tokens, heads * dv), float("nan"), device=DEV)
        where = (state, i32(starts[entries]), i32(np.asarray(lengths)[entries]), i32(entries), o)
        longest, portions = max(lengths[e] for e in entries), len(entries)
        if mode == "mlstm":
            den, _ = ops.mlstm_chunks(src, bias, bias, 15.0, *where, heads, d, dv, longest=longest, portions=portions)
            return state, o, den
        if mode == "decay":
            ops.decay_scan(src, decays, *where, heads, d, dv, longest=longest, chunks=True, portions=portions)
        elif mode == "delta":
            ops.delta_scan(src, *where, heads, heads // 2, d, dv, longest=longest, chunks=True, portions=portions)
        else:
            ops.gated_scan(src, *where, heads, 1, d, dv, longest=longest, chunks=True, portions=portions)
        return state, o, torch.zeros(tokens, heads, device=DEV)
    kind = ["decay", "delta", "gated", "mlstm"].index(mode)
    assert ops.matrix_chunks_waves(kind, heads, d, dv, max(lengths), n) == 4 and all(ops.matrix_chunks_waves(kind, heads, d, dv, e, 1) == 8 for e in lengths)
    real, ops.matrix_chunks_from = ops.matrix_chunks_from, lambda *a: 16
    try:
        together = run(list(range(n)))
        for e in range(n):
            alone = run([e])
            rows = slice(starts[e], starts[e] + lengths[e])
            assert torch.equal(together[0][e], alone[0][e]) and torch.equal(together[1][rows], alone[1][rows]) and torch.equal(together[2][rows], alone[2][rows]), e
    finally:
        ops.matrix_chunks_from = real
