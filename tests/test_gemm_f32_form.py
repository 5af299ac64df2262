"""Which kernel a 32-bit product takes."""
import pytest

from kipp_amd.csrc import ops


@pytest.mark.parametrize("m, n, k, form", [
    (16, 9728, 2560, 1), (2048, 31, 2560, 1),                                                                      # up to 16 rows, or too few rows of w for a tile
    (17, 2560, 768, 2), (24, 512, 256, 2), (32, 2560, 512, 2), (32, 6144, 64, 2), (48, 1024, 16, 4), (200, 512, 16, 4),     # few rows and short K
    (2048, 9728, 16, 0), (2048, 9728, 768, 0), (2048, 2560, 192, 0), (1024, 2560, 256, 0), (700, 1024, 64, 0),      # many tiles and short K
    (24, 2560, 768, 22), (333, 2560, 1024, 44), (2048, 512, 512, 44), (512, 1024, 256, 42), (333, 19456, 2560, 43), (1024, 6144, 2560, 44)])
def test_the_form_that_was_the_faster_one(m, n, k, form):
    """Sizes at which one kernel took 5 % less than the other, and the 4B shape's."""
    assert ops.gemm_f32_form(m, n, k) == form


@pytest.mark.parametrize("m, n, k, form", [
    (64, 6144, 1 << 26, 42), (20, 64, (1 << 26) + 4, 0), (64, 6144, (1 << 26) + 4, 0),      # 63 rows of x in 32 bits, and not
    (1 << 18, 1 << 16, 4096, 44), (1 << 18, 1 << 17, 4096, 0),                              # workgroups of 512 threads that one launch holds, and not
    (5_000_000, 64, 64, 44), (4_000_000, 64, 64, 0)])                                       # 64 x 64 tiles that a grid's second side holds, and not
def test_sizes_beyond_what_a_kernel_addresses(m, n, k, form):
    assert ops.gemm_f32_form(m, n, k) == form
