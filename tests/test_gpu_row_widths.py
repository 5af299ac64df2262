"""Kernels that hold a row in registers: every build of them, at the widths between which the dispatch changes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def f32(rng, *shape):
    return torch.tensor(rng.normal(size=shape), dtype=torch.float32, device=DEV)


def layer_norm64(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w + b


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("width", [1, 63, 256, 2560, 2561, 3072, 3073, 4096, 4097, 5120, 5121, 6144, 6145, 8191, 8192])
def test_layer_norm_and_step(width, parts):
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(width + parts)
    x, u, extra = f32(rng, 3, width), f32(rng, parts, 3, width), f32(rng, 3, width)
    w, b, w2, b2 = (f32(rng, width) for _ in range(4))
    delta = u if parts > 1 else u[0]
    total = u.double().sum(0)
    got = ops.layer_norm(delta, w, b, 1e-5, torch.empty((3, width), device=DEV), scale=0.7)
    ref = 0.7 * layer_norm64(total, w.double(), b.double(), 1e-5)
    # the slabs' sum, a mean and a variance of at most 32 numbers a lane and 16 waves, and a handful of roundings, of numbers up to ~ 5
    bound = (parts + 80) * 2.0 ** -24 * 25
    assert float((got.double() - ref).abs().max()) <= bound or width == 1
    assert width > 1 or torch.allclose(got.double(), 0.7 * b.double()[None].expand(3, 1))       # one number is its own mean
    before = x.double()
    out = ops.sandwich_step(x, delta, w, b, 1e-5, 0.5, extra, w2, b2, 1e-5, torch.empty((3, width), device=DEV))
    if width > 1:
        new = before + 0.5 * layer_norm64(total, w.double(), b.double(), 1e-5) + extra.double()
        assert float((x.double() - new).abs().max()) <= bound
        assert float((out.double() - layer_norm64(x.double(), w2.double(), b2.double(), 1e-5)).abs().max()) <= bound


@pytest.mark.parametrize("width", [4, 260, 2564, 3584, 3588, 4100, 8188])
def test_rows_at_multiples_of_16_bytes_and_elsewhere(width):
    """Widths of four columns a load: rows that begin elsewhere take a column a load, with the same result up to the order of the sums; a
    bfloat16 result is the float32 one rounded."""
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(width)

    def moved(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    x, u, w, b = f32(rng, 5, width), f32(rng, 2, 5, width), f32(rng, width), f32(rng, width)
    steps = []
    for place in (lambda t: t, moved):
        xs, out = place(x.clone()), torch.empty((5, width), device=DEV)
        ops.sandwich_step(xs, place(u), place(w), place(b), 1e-5, 0.5, None, place(w), place(b), 1e-5, out)
        steps.append((xs, out, ops.layer_norm(place(u), place(w), place(b), 1e-5, torch.empty((5, width), device=DEV))))
    for one, other in zip(*steps):      # both within the bound of the test above
        assert float((one - other).abs().max()) <= 2 * 82 * 2.0 ** -24 * 25 * (4.0 if width == 4 else 1.0)      # (four numbers can be close to each other)
    half, x2 = torch.empty((5, width), dtype=torch.bfloat16, device=DEV), x.clone()
    ops.sandwich_step(x2, u, w, b, 1e-5, 0.5, None, w, b, 1e-5, half)
    assert torch.equal(half, steps[0][1].bfloat16()) and torch.equal(x2, steps[0][0])
    assert torch.equal(ops.layer_norm(u, w, b, 1e-5, torch.empty((5, width), dtype=torch.bfloat16, device=DEV)), steps[0][2].bfloat16())


@pytest.mark.parametrize("width", [1, 4, 63, 512, 516, 2560, 2561])
def test_terms_of_a_weighted_sum_together(width):
    """One to six terms, in slabs and not, with biases and without: the bits of a launch a term, also where rows begin anywhere."""
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(width)
    x = f32(rng, 5, width)
    every = [(f32(rng, *((p,) if p > 1 else ()), 5, width), s, f32(rng, width) if b else None)
             for p, s, b in ((1, 1.25, False), (3, 0.8, True), (6, -0.5, False), (2, 1.0, True), (1, 0.3, True), (4, 2.0, False))]
    for count in range(1, 7):
        one, together = x.clone(), x.clone()
        for term in every[:count]:
            ops.residual_add_scaled(one, *term)
        ops.residual_add_terms(together, every[:count])
        assert torch.equal(one, together), count
        store = torch.zeros(x.numel() + 1, device=DEV)[1:].view(x.shape).copy_(x)
        assert torch.equal(ops.residual_add_terms(store, every[:count]), one), count
    ref = x.double()
    for delta, scale, bias in every:
        ref = ref + scale * ((delta.double().sum(0) if delta.dim() == 3 else delta.double()) + (0.0 if bias is None else bias.double()))
    assert float((one.double() - ref).abs().max()) <= 24 * 2.0 ** -24 * 30      # 24 additions of numbers up to about 30


@pytest.mark.parametrize("rows", [1, 33, 70])
@pytest.mark.parametrize("width", [3, 4, 8, 12, 16, 100, 255, 256, 260])
def test_terms_of_narrow_rows(rows, width):
    """Rows that share a workgroup, more and fewer than it holds, and numbers taken wherever rows end."""
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(rows * width)
    x, one, slabs, bias = f32(rng, rows, width), f32(rng, rows, width), f32(rng, 3, rows, width), f32(rng, width)
    ref = x.double() + 0.7 * (one.double() + bias.double()) - 0.4 * slabs.double().sum(0)
    got = ops.residual_add_terms(x.clone(), [(one, 0.7, bias), (slabs, -0.4, None)])
    assert float((got.double() - ref).abs().max()) <= 6 * 2.0 ** -24 * 16       # six additions of numbers up to about 16


def test_terms_without_rows_or_columns():
    """Nothing to add to is no error, with slabs and biases and without."""
    from kipp_amd.csrc import ops
    for shape in ((5, 0), (0, 5), (0, 0)):
        x, bias = torch.zeros(shape, device=DEV), torch.zeros(shape[1], device=DEV)
        assert ops.residual_add_scaled(x, torch.zeros(shape, device=DEV)) is x
        assert ops.residual_add_terms(x, [(torch.zeros((2, *shape), device=DEV), 0.5, bias), (torch.zeros(shape, device=DEV), 1.0, None)]) is x
    with pytest.raises(Exception, match="residual_add_terms"):
        ops.residual_add_terms(torch.zeros((2, 3), device=DEV), [(torch.zeros((3, 2), device=DEV), 1.0, None)])
    with pytest.raises(Exception, match="residual_add_scaled"):
        ops.residual_add_scaled(torch.zeros((2, 3), device=DEV), torch.zeros((3, 2), device=DEV))


@pytest.mark.parametrize("span", [1, 16, 64, 65, 256, 257, 512, 513, 1024, 1025, 1536, 1537, 2560, 2561, 4096, 4097, 5120, 5121, 11000])
@pytest.mark.parametrize("spans", [1, 3])
def test_state_space_finish(span, spans):
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(span)
    width = span * spans
    o, prep, proj, skip, w = f32(rng, 3, width), f32(rng, 3, width + 5), f32(rng, 3, width + 7), f32(rng, spans), f32(rng, width)
    out = ops.ssd_finish(o, prep, 5, proj, 7, skip, span, w, 1e-5, span, torch.empty((3, width), device=DEV))
    z = proj[:, 7:].double()
    y = (o.double() + skip.double().repeat_interleave(span) * prep[:, 5:].double()) * z * torch.sigmoid(z)
    ref = (y.view(3, spans, -1) / (y.view(3, spans, -1).square().mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(3, width) * w.double()
    # a handful of float32 roundings and a sum of `span` squares, at most `span` / 256 of them a thread: halved by the root
    assert ((out.double() - ref).abs() <= (ref.abs() + 1e-3) * 2.0 ** -24 * (span / 256 + 30)).all()


def fastest(run):
    """Milliseconds of 40 runs, the best of eight times."""
    marks = []
    for _ in range(8):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(40):
            run()
        end.record()
        marks.append((begin, end))
    torch.cuda.synchronize()
    return min(a.elapsed_time(b) for a, b in marks)


def test_wide_rows_take_their_share_of_the_time():
    """Rows of 8,192 are 3.2 times as many bytes as rows of 2,560, and take no more than four times as long."""
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(0)
    took = {}
    for width in (2560, 8192):
        x, u, w = torch.randn(2048, width, device=DEV), torch.randn(2048, width, device=DEV), f32(rng, width)
        out = torch.empty((2048, width), dtype=torch.bfloat16, device=DEV)
        took[width] = fastest(lambda: ops.sandwich_step(x, u, w, w, 1e-5, 0.01, next_w=w, next_b=w, next_eps=1e-5, out=out))
    assert took[8192] <= 4.0 * took[2560], took


def test_spans_take_their_share_of_the_time():
    """The same columns in spans of 1,280 take no more than one and a half times what they take in spans of 640."""
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(0)
    o, prep, proj, skip, w = f32(rng, 2048, 5120), f32(rng, 2048, 5120), f32(rng, 2048, 5120), f32(rng, 80), f32(rng, 5120)
    out = torch.empty((2048, 5120), dtype=torch.bfloat16, device=DEV)
    took = {span: fastest(lambda: ops.ssd_finish(o, prep, 0, proj, 0, skip, 64, w, 1e-5, span, out)) for span in (640, 1280)}
    assert took[1280] <= 1.5 * took[640], took
