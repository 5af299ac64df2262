"""Which rows a tile of the experts' products has, by what a step brings."""
import pytest
import torch

from kipp_amd.csrc import ops


@pytest.mark.parametrize("experts", [8, 32, 256])
def test_few_rows_an_expert(experts):
    for pairs, rows in ((1, 64), (6 * experts, 64), (6 * experts + 1, 128), (12 * experts, 128)):
        assert ops.moe_tile_rows(torch.bfloat16, 4096, 3072, pairs=pairs, experts=experts) == rows
