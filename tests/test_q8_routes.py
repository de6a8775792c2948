"""Which kernel takes a full-row Q8 product (nitro_q8_tile_rows), at the limits of its
rule: on the CPU, no product is run."""
import pytest

from nitrorag_amd import _native as N
from nitrorag_amd.q8 import MATMUL, QKV, RESIDUAL, SWIGLU, tile_rows


def test_small_batches_and_small_products_take_other_kernels():
    assert tile_rows(4, 4096, 32000) == 0
    assert tile_rows(96, 4096, 32000) in (64, 128)
    assert tile_rows(1024, 768, 64) == 0


@pytest.mark.parametrize("launch", [MATMUL, RESIDUAL, SWIGLU, QKV])
def test_offsets_past_32_bits_take_other_kernels(launch):
    # x in split form, 6 bytes a value in panels of 16 rows, below 2^32 bytes
    rows = (1 << 32) // (6 * 4096) // 16 * 16
    assert tile_rows(rows, 4096, 4096, launch, 4096) in (64, 128)
    assert tile_rows(rows + 1, 4096, 4096, launch, 4096) == 0
    # a matrix's tile layout, 576 bytes per 16 rows and 32 columns, below 2^32 bytes
    d = ((1 << 32) // (576 * 128) - 1) * 16
    assert tile_rows(2000, 4096, d, launch, 32) in (64, 128)
    assert tile_rows(2000, 4096, d + 32, launch, 32) == 0


def test_bad_arguments():
    for args in ((0, 64, 64), (8, 0, 64), (8, 40, 64), (8, 64, 0), (8, 64, 64, 4), (8, 64, 64, -1), (8, 64, 64, QKV, 0)):
        with pytest.raises(N.NitroError):
            tile_rows(*args)
