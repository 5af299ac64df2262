"""Which steps take a matrix memory by chunks."""
import pytest

from kipp_amd.csrc import ops

DECAY, DELTA, GATED, MLSTM = 0, 1, 2, 3


@pytest.mark.parametrize("mode, heads, d, dv, entries, walks, chunks", [
    (DECAY, 8, 128, 320, 1, 64, 96), (DELTA, 8, 128, 320, 1, 112, 128), (DELTA, 8, 128, 320, 4, 176, 256), (GATED, 40, 128, 64, 1, 64, 96), (GATED, 40, 128, 64, 16, 32, 48),
    (DECAY, 8, 64, 128, 16, 112, 160), (DELTA, 8, 64, 128, 16, 192, 256), (DECAY, 16, 256, 256, 1, 48, 64), (DELTA, 16, 256, 256, 4, 32, 48),
    (DELTA, 4, 192, 64, 1, 96, 128), (DELTA, 32, 128, 128, 4, 160, 256),
    (GATED, 16, 192, 128, 16, 16, 32), (DECAY, 16, 192, 128, 48, 0, 24), (DECAY, 16, 256, 256, 2, 24, 32), (MLSTM, 16, 192, 128, 4, 16, 24), (MLSTM, 16, 192, 128, 48, 0, 16),
    (MLSTM, 8, 64, 128, 48, 0, 24), (DELTA, 16, 192, 128, 4, 32, 48), (DELTA, 8, 256, 512, 16, 16, 40)])
def test_where_chunks_were_the_faster_way(mode, heads, d, dv, entries, walks, chunks):
    """Steps whose longest entry has `walks` tokens walk, with `chunks` they take chunks: at those the chunks were the faster way, and no
    slower with a walk of single tokens beside them; at a few of the former they were by themselves."""
    start = ops.matrix_chunks_from(mode, d, entries * heads * d * dv)
    assert walks < start <= chunks and start >= ops.CHUNKS_FROM


@pytest.mark.parametrize("mode, heads, d, dv, longest, portions, waves", [
    (GATED, 16, 192, 128, 80, 64, 4), (GATED, 16, 192, 128, 80, 4, 4), (GATED, 16, 128, 128, 80, 4, 4), (DELTA, 32, 64, 64, 64, 64, 4), (DELTA, 32, 64, 64, 64, 4, 4),
    (MLSTM, 16, 192, 128, 64, 64, 4), (MLSTM, 4, 64, 64, 150, 16, 4), (MLSTM, 40, 128, 64, 150, 4, 4), (DECAY, 16, 192, 128, 80, 32, 4), (DECAY, 40, 128, 64, 80, 64, 4),
    (GATED, 40, 128, 64, 2048, 1, 8), (GATED, 16, 128, 128, 700, 10, 8), (DECAY, 8, 128, 320, 80, 4, 8), (DELTA, 8, 128, 320, 80, 64, 8), (DELTA, 4, 64, 64, 64, 16, 8),
    (MLSTM, 8, 128, 320, 2048, 1, 8), (MLSTM, 8, 256, 512, 64, 64, 8), (GATED, 16, 256, 256, 64, 64, 8), (DECAY, 4, 64, 64, 64, 64, 8)])
def test_the_waves_that_were_the_faster_ones(mode, heads, d, dv, longest, portions, waves):
    """Sizes at which four or eight waves a workgroup of the walk took 5 % less than the other (or eight alone were measured the faster at all)."""
    assert ops.matrix_chunks_waves(mode, heads, d, dv, longest, portions) == waves
