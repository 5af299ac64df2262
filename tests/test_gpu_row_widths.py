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


def test_wide_rows_take_their_share_of_the_time():
    """Rows of 8,192 are 3.2 times as many bytes as rows of 2,560, and take no more than four times as long."""
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(0)
    took = {}
    for width in (2560, 8192):
        x, u, w = torch.randn(2048, width, device=DEV), torch.randn(2048, width, device=DEV), f32(rng, width)
        out = torch.empty((2048, width), dtype=torch.bfloat16, device=DEV)
        marks = []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(40):
                ops.sandwich_step(x, u, w, w, 1e-5, 0.01, next_w=w, next_b=w, next_eps=1e-5, out=out)
            end.record()
            marks.append((begin, end))
        torch.cuda.synchronize()
        took[width] = min(a.elapsed_time(b) for a, b in marks)
    assert took[8192] <= 4.0 * took[2560], took
