"""What the experts' products refuse before anything is launched."""
import ctypes

import pytest
import torch

from kipp_amd.csrc import build

BF16, REFUSED = 1, -2


@pytest.mark.skipif(torch.cuda.is_available(), reason="asks for the refusal alone, without operands")
@pytest.mark.parametrize("tile_rows", [128, 256])
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("gated", [True, False])
def test_sizes_that_32_bit_offsets_do_not_reach(tile_rows, aligned, gated):
    """Tiles of 128 and 256 rows go by 32-bit offsets into x and into an expert's matrix, whichever kernel takes them."""
    lib = build.library("moe")
    ptr, whole = ctypes.c_void_p, ctypes.c_int          # declared: a number of arguments that is not the entry's raises
    lib.kipp_moe_expert.argtypes = [ptr, whole, ptr, ptr, whole, ptr, whole, ptr] + [whole] * 9 + [ptr]
    lib.kipp_moe_expert_gated.argtypes = [ptr, whole, ptr, ptr, ptr, whole, ptr, whole, ptr] + [whole] * 8 + [ptr]
    null, at = ctypes.c_void_p(0), ctypes.c_void_p(0 if aligned else 4)

    def call(max_tiles, n_out, k, x_rows, sorted_rows):
        sizes = (max_tiles, null, BF16, n_out, k, 1, tile_rows, x_rows, sorted_rows, 8)
        if gated:
            return lib.kipp_moe_expert_gated(at, BF16, null, null, at, BF16, null, *sizes, null)
        return lib.kipp_moe_expert(at, BF16, null, at, BF16, null, *sizes, 0, null)
    k = 2432
    for sorted_rows in (8, 1 << 20):        # few rows an expert and many
        assert call((1 << 31) // (tile_rows * k) + 1, 64, k, 64, sorted_rows) == REFUSED
        assert call(8, (1 << 31) // ((2 if gated else 1) * 4096) + 1, 4096, 64, sorted_rows) == REFUSED
        assert call(8, 64, 4096, 1 << 20, sorted_rows) == REFUSED         # rows that the list may name
