"""The kernels in front of the gated matrix memories: a step of single tokens (its filter keeps the inputs itself) gives bit for bit
what the same tokens give as portions of one and of two entries, with taps that are known to the kernel and others."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def tensors(rng, taps, channels, stride, heads):
    f = lambda *shape: torch.tensor(rng.normal(size=shape), dtype=torch.float32, device="cuda:0")  # noqa: E731
    return f(6, stride), f(channels, taps), f(channels), f(heads), f(heads)


# 6 tokens one after the other as steps of one entry; then 4 and 2 of them as portions (the portions' slot is filled by the kernel behind)
@pytest.mark.parametrize("taps", [1, 2, 4, 5])
@pytest.mark.parametrize("kind", ["delta", "ssd"])
@pytest.mark.parametrize("heads,groups,d,dv", [(4, 2, 24, 40), (6, 3, 128, 72), (2, 1, 300, 130)])
def test_single_tokens_are_portions_of_one(taps, kind, heads, groups, d, dv):
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(taps + d)
    if kind == "delta":
        channels = 2 * groups * d + heads * dv
        stride, width = channels + 2 * heads, channels + 2 * heads
    else:
        channels = heads * dv + 2 * groups * d
        stride, width = heads * dv + channels + heads, 2 * groups * d + 2 * heads * dv + heads
    proj, conv_w, conv_b, a_log, dt_bias = tensors(rng, taps, channels, stride, heads)
    i32 = lambda *a: torch.tensor(a, dtype=torch.int32, device="cuda:0")  # noqa: E731
    size = (ops.delta_state_size if kind == "delta" else ops.ssd_state_size)(heads, groups, d, dv, taps)
    kept = torch.tensor(rng.normal(size=(3, size)), dtype=torch.float32, device="cuda:0")

    def run(state, first, lens, slots, longest=None):
        n = sum(lens)
        prep = torch.full((n, width), float("nan"), dtype=torch.float32, device="cuda:0")
        starts = [sum(lens[:i]) for i in range(len(lens))]
        seq = i32(*[e for e, m in enumerate(lens) for _ in range(m)])
        rows = proj[first:first + n].contiguous()
        said = {} if longest == 0 else {"longest": longest or max(lens)}
        batch = (seq, i32(*starts), i32(*lens), i32(*slots))
        if kind == "delta":
            ops.delta_prepare(rows, conv_w, a_log, dt_bias, state, *batch, prep, heads, groups, d, dv, channels, channels + heads, 1e-6, **said)
        else:
            ops.ssd_prepare(rows, conv_w, conv_b, a_log, dt_bias, state, *batch, prep, heads, groups, d, dv, **said)
        return prep

    one, many, both = kept.clone(), kept.clone(), kept.clone()
    steps = torch.cat([run(one, t, [1], [1]) for t in range(6)])
    portions = torch.cat([run(many, 0, [4], [1]), run(many, 4, [2], [1])])
    assert torch.isfinite(steps[:, :channels]).all()
    assert torch.equal(steps, portions) and torch.equal(one, many)
    assert torch.equal(one[0], kept[0]) and torch.equal(one[2], kept[2])        # nobody else's slot
    pair = run(both, 0, [1, 1], [2, 0])                                          # two entries of one token each
    again = torch.cat([run(kept, 0, [1], [2]), run(kept, 1, [1], [0])])
    assert torch.equal(pair, again) and torch.equal(both, kept)
    # an entry without a token beside one of two: as many tokens as entries, and nothing said of the longest
    empty, plain = kept.clone(), kept.clone()
    assert torch.equal(run(empty, 0, [2, 0], [1, 2], longest=0), run(plain, 0, [2], [1])) and torch.equal(empty, plain)


# spans on both sides of what a thread's registers hold
@pytest.mark.parametrize("heads,dv,spans", [(4, 40, 2), (8, 128, 1), (20, 256, 1), (20, 272, 1), (4, 260, 1), (1, 256, 1), (1, 257, 1)])
def test_ssd_finish(heads, dv, spans):
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(heads * dv)
    f = lambda *shape: torch.tensor(rng.normal(size=shape), dtype=torch.float32, device="cuda:0")  # noqa: E731
    width = heads * dv
    o, prep, proj, skip, w = f(3, width), f(3, width + 5), f(3, width + 7), f(heads), f(width)
    out = ops.ssd_finish(o, prep, 5, proj, 7, skip, dv, w, 1e-5, width // spans, torch.empty((3, width), device="cuda:0"))
    y = (o.double() + skip.double().repeat_interleave(dv) * prep[:, 5:].double())
    z = proj[:, 7:].double()
    y = y * z * torch.sigmoid(z)
    ref = (y.view(3, spans, -1) / (y.view(3, spans, -1).square().mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(3, width) * w.double()
    # a handful of float32 roundings and a sum of `span` squares: its relative error at most span / 256 + 10 of them, halved by the root
    assert ((out.double() - ref).abs() <= (ref.abs() + 1e-3) * 2.0 ** -24 * (width / 256 + 30)).all()


def test_latent_prepare_without_a_row_to_write():
    """A run that reads another's cache brings no weights for the row it does not write: the query latent is what it is beside a row, and
    the cache stays as it was."""
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(5)
    f = lambda *shape: torch.tensor(rng.normal(size=shape), dtype=torch.float32, device="cuda:0")  # noqa: E731
    i32 = lambda *a: torch.tensor(a, dtype=torch.int32, device="cuda:0")  # noqa: E731
    proj, q_w, c_w, cache = f(3, 40 + 24 + 8), f(40), f(24), f(2, 1, 16, 32)
    positions, seq, table, freq = i32(3, 4, 17), i32(0, 0, 0), i32(1, 0).view(1, 2), f(4)
    there = ops.latent_prepare(proj, torch.empty((3, 40), device="cuda:0"), cache.clone(), positions, seq, table, 40, 24, 8, q_w, c_w, 1e-6, freq, 8, 1.0)
    before, cq = cache.clone(), torch.empty((3, 40), device="cuda:0")
    fn = ops._fn("latent", "kipp_latent_prepare", [ops._c_ptr, ops._c_int, ops._c_int, ops._c_ptr, ops._c_ptr, ops._c_float, ops._c_ptr, ops._c_int, ops._c_ptr,
                                                   ops._c_int, ops._c_ptr, ops._c_ptr, ops._c_ptr, ops._c_int, ops._c_ptr, ops._c_int, ops._c_float]
                 + [ops._c_int] * 8 + [ops._c_ptr])
    rc = fn(proj.data_ptr(), 1, proj.shape[1], q_w.data_ptr(), None, 1e-6, cq.data_ptr(), ops._code(cq), cache.data_ptr(), ops._code(cache), positions.data_ptr(),
            seq.data_ptr(), table.data_ptr(), 2, freq.data_ptr(), 8, 1.0, 0, 3, 40, 40, 24, 8, 16, 0, ops._stream())
    assert rc == 0 and torch.equal(cq, there) and torch.equal(cache, before)
