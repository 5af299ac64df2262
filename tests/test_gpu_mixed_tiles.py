"""The mixed-head attention's tiles of rows where their places can go wrong: contexts that end in either half of a tile of keys or at its
edge, pages of several blocks of 16 keys, heads that leave a wave's share unfilled, both builds."""
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
