"""Which rows a tile of the experts' products has, by what a step brings."""
import pytest
import torch

from kipp_amd.csrc import ops


@pytest.mark.parametrize("experts,width,inner,gated,most,then", [(32, 2560, 2432, False, 192, 256), (32, 2560, 2432, True, 192, 256), (8, 4096, 3584, False, 96, 128),
                                                                 (32, 4096, 3072, False, 190, 256), (32, 4096, 3072, True, 158, 256), (32, 5120, 6400, False, 96, 256),
                                                                 (256, 2560, 512, False, 1536, 256), (1, 64, 64, True, 12, 128), (32, 1024, 1024, False, 384, 128)])
def test_few_rows_an_expert(experts, width, inner, gated, most, then):
    """Up to a number of pairs that falls with the experts' sizes: by pairs an expert, by the work, never below three an expert."""
    for pairs, rows in ((1, 64), (most, 64), (most + 1, then)):
        assert ops.moe_tile_rows(torch.bfloat16, width, inner, pairs=pairs, experts=experts, gated=gated) == rows


def test_identity_experts_take_a_share_of_the_pairs():
    rows = [ops.moe_tile_rows(torch.bfloat16, 2560, 2432, pairs=n, experts=32, identity=8) for n in (240, 241)]
    assert rows == [64, 256]


def test_many_rows_an_expert():
    """Tiles of 256 where the launch then still has workgroups for the chip."""
    rows = lambda experts, width, inner, pairs, gated: ops.moe_tile_rows(torch.bfloat16, width, inner, pairs=pairs, experts=experts, gated=gated)  # noqa: E731
    assert [rows(32, 2560, 2432, 32 * n, g) for g in (True, False) for n in (7, 96, 241)] == [256] * 6
    assert [rows(8, 1024, 1024, 8 * n, False) for n in (282, 512, 896, 897, 7000)] == [128, 128, 256, 256, 256]
    assert [rows(8, 1024, 1024, 8 * n, True) for n in (100, 282, 384, 1024)] == [128, 128, 256, 256]
    assert ops.moe_tile_rows(torch.bfloat16, 2560, 2432, pairs=1, experts=32, aligned=False) == 128
    assert ops.moe_tile_rows(torch.bfloat16, 2560, 2432, pairs=32 * 500, experts=32, aligned=False) == 128
    assert ops.moe_tile_rows(torch.bfloat16, 2560, 2432) == 128 and ops.moe_tile_rows(torch.bfloat16, 2560, 2440) == 16
    assert rows(3, 32768, 32768, 3 * 5000, False) == 128        # offsets of 32 bits


def test_rows_of_a_step():
    """The kernel for few rows up to six pairs an expert, or as long as it may where the experts have few numbers; then the walk, in tiles of 256
    where those are workgroups enough; what begins at no multiple of 16 bytes, and float32, as ever."""
    rows = lambda experts, width, inner, pairs, gated, **k: ops.moe_tile_rows(k.pop("dtype", torch.bfloat16), width, inner, pairs=pairs, experts=experts, gated=gated, **k)  # noqa: E731
    assert [rows(32, 2560, 2432, n, g) for g in (False, True) for n in (192, 193)] == [64, 256, 64, 256]
    assert [rows(32, 2560, 2432, n, False, identity=8) for n in (240, 241)] == [64, 256]
    assert [rows(64, 2048, 704, 64 * 6 + n, g) for g in (False, True) for n in (0, 1)] == [64, 128, 64, 256]
    assert [rows(32, 2048, 1408, 32 * n, g) for g in (False, True) for n in (12, 13)] == [64, 128, 64, 256]      # 92 million numbers
    assert [rows(8, 1024, 1024, n, False) for n in (30, 96, 97, 8 * 512, 8 * 900)] == [64, 64, 128, 128, 256]
    assert [rows(32, 2560, 2432, n, True, aligned=False) for n in (1, 500, 9000)] == [128, 128, 128]
    assert rows(32, 2560, 2432, 9000, True, dtype=torch.float32) == 16


@pytest.mark.parametrize("experts, width, inner, pairs", [(1, 4096, 3072, 6), (3, 4096, 768, 26), (1, 64, 96, 7), (16, 512, 4096, 88), (8, 4096, 96, 36), (2, 5120, 4096, 20), (16, 2048, 2432, 130)])
@pytest.mark.parametrize("gated", [False, True])
def test_few_or_small_experts_keep_the_kernel_for_few_rows(experts, width, inner, pairs, gated):
    """Sizes at which the walk took 1.1 to 2.1 times as long."""
    assert ops.moe_tile_rows(torch.bfloat16, width, inner, pairs=pairs, experts=experts, gated=gated) == 64
