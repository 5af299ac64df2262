"""Which rows a tile of the experts' products has, by what a step brings."""
import pytest
import torch

from kipp_amd.csrc import ops


@pytest.mark.parametrize("experts", [8, 32, 256])
def test_few_rows_an_expert(experts):
    for pairs, rows in ((1, 64), (6 * experts, 64), (6 * experts + 1, 128), (12 * experts, 128)):
        assert ops.moe_tile_rows(torch.bfloat16, 4096, 3072, pairs=pairs, experts=experts) == rows


def test_many_rows_an_expert():
    """Tiles of 256 from enough pairs an expert on, where the launch then still has workgroups for the chip."""
    rows = lambda experts, width, inner, pairs, gated: ops.moe_tile_rows(torch.bfloat16, width, inner, pairs=pairs, experts=experts, gated=gated)  # noqa: E731
    assert [rows(32, 2560, 2432, 32 * n, True) for n in (96, 97)] == [128, 256]
    assert [rows(32, 2560, 2432, 32 * n, False) for n in (240, 241)] == [128, 256]
    assert [rows(8, 1024, 1024, 8 * n, False) for n in (282, 512, 7000)] == [128, 128, 256]
    assert [rows(8, 1024, 1024, 8 * n, True) for n in (100, 282, 1024)] == [128, 128, 256]
    assert ops.moe_tile_rows(torch.bfloat16, 2560, 2432, pairs=1, experts=32, aligned=False) == 128
    assert ops.moe_tile_rows(torch.bfloat16, 2560, 2432, pairs=32 * 500, experts=32, aligned=False) == 128
