"""The many-rows product that ends in a gated activation with relu, or with biases: against the written-out float64 form."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# tiles and columns that end inside a tile, rows that begin at no multiple of 16 bytes (150 is no multiple of 8), whole rounds and a rest
@pytest.mark.parametrize("force", [0, 441, 221, 421, 2421])
@pytest.mark.parametrize("m,inner,k", [(257, 150, 64), (300, 24, 2560), (2050, 4804, 64)])
@pytest.mark.parametrize("activation,biased", [("relu", False), ("relu", True), ("silu", True), ("silu", False)])
def test_glu_end(m, inner, k, force, activation, biased):
    from kipp_amd.csrc import ops
    rng = np.random.default_rng(m + inner)
    dev = torch.device("cuda:0")
    x = torch.tensor(rng.normal(size=(m, k)), dtype=torch.bfloat16)
    w = torch.tensor(rng.normal(size=(2 * inner, k)) / np.sqrt(k), dtype=torch.bfloat16)
    bias = torch.tensor(rng.normal(size=2 * inner), dtype=torch.float32) if biased else None
    got = ops.gemm_tiles(x.to(dev), w.to(dev), "glu", force=force, activation=activation, bias=None if bias is None else bias.to(dev))
    both = x.double() @ w.double().T
    if biased:
        both = both + bias.double()
    gate, up = both[:, :inner], both[:, inner:]
    ref = ((gate.clamp(min=0) if activation == "relu" else gate * torch.sigmoid(gate)) * up).numpy()
    assert got.dtype == torch.bfloat16 and tuple(got.shape) == (m, inner)
    # one rounding to bfloat16 (2^-9 of the result), and of a sum of k float32 terms of total size ~ sqrt(k) |x||w| ~ 1 each
    # in any order at most k 2^-24 of that, through an activation of slope about 1 and a factor of at most ~ 6
    err = np.abs(got.double().cpu().numpy() - ref)
    assert (err <= 2.0 ** -8 * np.abs(ref) + 6 * k * 2.0 ** -24 + 1e-5).all()
    if activation == "silu" and not biased:
        assert torch.equal(got, ops.gemm_tiles(x.to(dev), w.to(dev), "swiglu", force=force))
