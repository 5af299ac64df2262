"""The mixed-head attention's tiles of rows where their places can go wrong: contexts that end in either half of a tile of keys or at its
edge, pages of several blocks of 16 keys, heads that leave a wave's share unfilled, both builds."""
import numpy as np
import pytest

from tests.test_gpu_tobinex import KERNEL_TOL, MixerCase, close

pytestmark = pytest.mark.gpu


# (heads, key/value heads, key size, value size, window, kept first keys, rows, page)
@pytest.mark.parametrize("whole", [False, True])
@pytest.mark.parametrize("geometry", [
    (32, 8, 128, 128, None, 0, 145, 16), (32, 8, 64, 64, None, 0, 129, 48), (32, 8, 32, 64, 50, 20, 177, 32), (32, 8, 32, 32, 40, 0, 15, 16),
    (20, 4, 32, 64, None, 0, 113, 32), (17, 17, 32, 16, None, 0, 97, 48), (24, 8, 64, 32, 33, 1, 161, 16), (12, 3, 32, 256, None, 0, 81, 16),
    (5, 5, 32, 48, None, 0, 1, 16), (16, 2, 96, 128, 70, 3, 129, 80)])
def test_tiles_of_rows(monkeypatch, geometry, whole):
    from kipp_amd.csrc import ops
    H_, G, d, dv, window, keep, T, page = geometry
    monkeypatch.setattr(ops, "COMPUTE_UNITS", 0 if whole else 1 << 20)         # which build takes a step follows from its items and the units
    case = MixerCase(H_, G, d, dv, window, keep, T, seed=T, page=page)
    got, _ = case.run("bfloat16", True, slabs=2)
    close(got, case.plain(True), KERNEL_TOL["bfloat16"], f"{geometry} whole {whole}")


@pytest.mark.parametrize("off", ["bias", "sink", "mix", "gate"])
def test_each_mechanism_off(off):
    case = MixerCase(18, 6, 32, 32, window=60, keep=4, T=131, seed=5, **{n: n != off for n in ("bias", "sink", "mix", "gate")})
    got, _ = case.run("bfloat16", True)
    close(got, case.plain(True), KERNEL_TOL["bfloat16"], off)


def _attend(case, rows, runs, single):
    """The last `rows` rows of the case: one portion whose tiles' keys go in `runs` runs each, or single tokens whose keys do."""
    import torch
    from kipp_amd.csrc import ops
    dev, H_, G, d, dv, T, page = torch.device("cuda:0"), case.H, case.G, case.d, case.dv, case.T, case.page
    t = lambda a, ty=None: torch.tensor(np.asarray(a), device=dev, dtype=ty)  # noqa: E731
    i32 = lambda a: t(a, torch.int32)  # noqa: E731
    blocks = -(-T // page)
    table = i32(np.random.default_rng(9).permutation(blocks)[None, :])
    k_cache, v_cache = (torch.zeros((blocks, G, page, n), dtype=torch.bfloat16, device=dev) for n in (d, dv))
    proj = t(case.proj)
    q = ops.mixed_prepare(proj, torch.empty((T, H_ * d), dtype=torch.bfloat16, device=dev), k_cache, v_cache, i32(range(T)), i32([0] * T), table,
                          H_, G, d, dv, t(case.qw), t(case.kw), case.eps)[T - rows:].contiguous()
    numbers = (H_, G, d, dv, case.scale, 0, 0, t(case.r1), t(case.r2), t(case.sink), t(case.mix))
    gate, out = proj[T - rows:].contiguous(), torch.empty((rows, H_ * dv), dtype=torch.bfloat16, device=dev)
    more = dict(gate=gate, gate_at=H_ * d + G * d + G * dv)
    if single:
        space = ops.mixed_single_workspace(rows, H_, dv, -(-T // ops.MIXED_SINGLE_KEYS), runs, dev)
        ops.mixed_attention_single(q, k_cache, v_cache, out, i32(range(rows)), i32(range(T - rows, T)), i32(range(rows)),
                                   table.repeat(rows, 1).contiguous(), *numbers, space, **more)
    else:
        tiles = range(0, rows, 16)
        items = tuple(i32(a) for a in ([0] * (runs * len(tiles)), np.repeat(tiles, runs), list(range(runs)) * len(tiles), [runs] * (runs * len(tiles))))
        space = ops.mixed_attention_workspace(len(items[0]), rows, H_, dv, runs, dev)
        ops.mixed_attention_mfma(q, k_cache, v_cache, out, items, len(items[0]), i32([runs] * rows), runs, i32([0]), i32([rows]), i32([T]), table,
                                 *numbers, space, **more)
    close(out.float().cpu().numpy(), case.plain(True)[T - rows:], KERNEL_TOL["bfloat16"], f"{runs} runs, single {single}")


@pytest.mark.parametrize("geometry", [(32, 8, 128, 128), (12, 4, 32, 64), (6, 3, 32, 16)])
def test_many_runs_of_keys(geometry):
    """Up to the sixteen runs that a plan makes, none of them empty (32 and 18 tiles of keys): statistics of several runs a quarter of a wave, sums
    beyond the first eight; single tokens over as many runs as they have tiles."""
    for T, counts in ((1010, (5, 8, 16)), (570, (9,))):
        case = MixerCase(*geometry, None, 0, T, seed=T)
        for runs in counts:
            _attend(case, 33, runs, False)
        _attend(case, 3, -(-T // 64), True)
