"""How a prompt product is cut at rows that its class was not timed at: by the times of the rows it was timed at, in proportion to the rounds
of tiles over the compute units."""
import math
from types import SimpleNamespace

import pytest
import torch

from kipp_amd.runtime import Runtime


@pytest.mark.parametrize("m", [193, 256, 257, 1193, 2048])
@pytest.mark.parametrize("cols,pairs", [(12288, True), (4096, False), (100, False)])
def test_rounds(m, cols, pairs):
    half = 2 if pairs else 1
    big = 0.1 + 0.022 * 32
    tiles = math.ceil(m / 256) * math.ceil(cols * half / 256)
    assert Runtime._rounds_of(441, m, cols, pairs) == pytest.approx(math.ceil(tiles / 256) * big)
    assert Runtime._rounds_of(1423, m, cols, pairs) == pytest.approx(math.ceil(tiles * 3 / 256) * big)
    assert Runtime._rounds_of("library", m, cols, pairs) == math.ceil(m / 256)
    # whole rounds and a rest: as many columns in whole rounds as fit; one cut where there is none, or nothing left
    if tiles <= 256 or tiles % 256 == 0:
        assert Runtime._rounds_of(32421, m, cols, pairs) == pytest.approx(Runtime._rounds_of(1421, m, cols, pairs))
    else:
        rows = math.ceil(m / 256)
        first = tiles // 256 * 256 // rows
        rest = math.ceil(m / 128) * math.ceil((cols * half - first * 256) / 128)
        assert Runtime._rounds_of(32421, m, cols, pairs) == pytest.approx(math.ceil(rows * first / 256) * big + math.ceil(rest / 256) * (0.1 + 0.022 * 8))


def test_other_rows_take_the_times_in_proportion(monkeypatch):
    rt = Runtime.__new__(Runtime)
    rt.own_prompt_products, rt.for_a_graph, rt.prompt_product_choices = "auto", False, {}
    took = {"library": 0.4, "plan": 0.36, 1421: 0.351, 32421: 0.350}
    monkeypatch.setattr(Runtime, "_choices_of_process", {("auto", ("gated",)): (32421, 2048, took, {2048: 32421})})

    def never():
        raise AssertionError("nothing is run once a class has been timed")
    ways = {name: never for name in took}
    for _ in range(2):
        assert rt._fastest(("gated",), ways, (), 2048, 12288, pairs=True) == 32421       # level there: what was measured
        assert rt._fastest(("gated",), ways, (), 1193, 12288, pairs=True) == 1421        # two rounds of three, against one and four small ones
    assert rt.prompt_product_choices == {("gated",): 32421}


def test_own_products_keep_the_plans_bits_at_every_number_of_rows(monkeypatch):
    """A cut that gives the plan's bits at the rows a class was timed at is not taken at rows where the plan takes other parts of K."""
    rt = Runtime.__new__(Runtime)
    rt.own_prompt_products, rt.for_a_graph, rt.prompt_product_choices = True, False, {}
    took = {"plan": 0.4, 443: 0.1, 1423: 0.2}
    monkeypatch.setattr(Runtime, "_choices_of_process", {(True, ("linear",)): (443, 2048, took, {2048: 443})})
    assert rt._fastest(("linear",), {}, ("plan", 442, 1422), 1100, 4096) == "plan"
    assert rt._fastest(("linear",), {}, ("plan", 443, 1423), 1101, 4096) == 443


@pytest.mark.parametrize("own", [True, "auto"])
def test_own_products_are_timed_for_every_number_of_parts(monkeypatch, own):
    """Rows of one class that the plan cuts into one, two and three parts of K: each finds the cuts with its parts among the ways, timed; where
    any way may be taken, the class is timed once."""
    rt = Runtime.__new__(Runtime)
    rt.own_prompt_products, rt.for_a_graph, rt.prompt_product_choices = own, False, {}
    rt.staged_rows, rt.few_rows, rt.tile_products, rt.library_products = 192, 64, 0, 0
    parts = {1100: 1, 1300: 2, 1500: 3, 1101: 1}
    asked = []
    rt.ops = SimpleNamespace(gemm_rows_ok=lambda m, k: False, gemm_tiles_ok=lambda m, k, n: True, gemm_tiles_parts=lambda m, *a: parts[m],
                             gemm_tiles=lambda x, w, **k: torch.zeros(1, 1, 1))
    monkeypatch.setattr(Runtime, "_fastest", lambda self, key, ways, same, m, cols, **k: asked.append((key, same)) or "plan")
    w = torch.zeros((64, 32), dtype=torch.bfloat16)
    for m in parts:
        rt.linear(torch.zeros((m, 32), dtype=torch.bfloat16), w, slabs=True)
    keys = {m: key for m, (key, _) in zip(parts, asked)}
    assert keys[1100] == keys[1101] and len(set(keys.values())) == (3 if own is True else 1)
    for m, (_, same) in zip(parts, asked):
        assert all(cut % 10 == parts[m] for cut in same if cut != "plan")


def test_ways_whose_times_do_not_go_by_rounds_keep_their_rows():
    """[2,560 x 9,728] as measured at 2,048 rows, the library's the fastest: so it is at 1,536 (157 us; the plan 265).  One of our cuts is
    left for another where that promises more than 5 %."""
    took = {"library": 0.186, "plan": 0.205, 441: 0.363, 442: 0.233, 1421: 0.353, 1423: 0.209}
    for m in (1100, 1536, 1900):
        assert Runtime._at_rows("library", took, 2048, m, 2560, False) == "library"
        assert Runtime._at_rows("plan", took, 2048, m, 2560, False) == "plan"
    ours = {"library": 0.4, 442: 0.1, 444: 0.104}       # tiles in half a round and parts in one: 160 and 320 at 2,048 rows
    assert Runtime._at_rows(442, ours, 2048, 2047, 2560, False) == 442
    assert Runtime._at_rows(442, ours, 2048, 1500, 2560, False) == 444              # 240 in one round where 320 were two
    assert Runtime._at_rows(441, {"plan": 0.4}, 2048, 1500, 2560, False) == "plan"       # nothing else of the same bits
