"""The rule that picks an expert tile's row limit, on both sides of its lines."""
import pytest
import torch

from kubernetes_cloud_amd.ops.moe import tile_rows


@pytest.mark.parametrize("T,top,E,d,F,rows", [
    (8, 2, 2, 4096, 4096, 8), (16, 2, 2, 4096, 4096, 8), (16, 4, 8, 4096, 4096, 8), (8, 1, 2, 4096, 8192, 8),  # long rows, more than 3 of an expert
    (6, 4, 8, 4096, 4096, 4), (16, 3, 16, 4096, 2048, 4), (5, 1, 2, 4096, 8192, 4),                            # up to 3
    (16, 4, 4, 2048, 2048, 4), (16, 8, 16, 2048, 1024, 4), (16, 8, 8, 1024, 512, 4),                          # rows that a block takes whole
    (4, 2, 2, 4096, 4096, 4), (2, 2, 2, 4096, 4096, 2), (1, 2, 2, 4096, 4096, 1)])
def test_few_tokens(T, top, E, d, F, rows):
    """An expert's weights are streamed once for 8 of its rows, or for 4 where that costs less."""
    assert tile_rows(T, top, E, d, F, torch.bfloat16) == rows
    assert tile_rows(T, top, E, d, F, torch.float32) == (rows if T <= 4 else 8)


@pytest.mark.parametrize("top,E,d,F,r,rows", [
    (5, 32, 2048, 768, 136, 192), (4, 32, 1536, 704, 136, 192), (6, 64, 1024, 448, 136, 192), (2, 12, 4096, 1920, 136, 192),
    (4, 40, 2048, 512, 136, 128), (4, 28, 2048, 640, 136, 128), (5, 32, 2048, 768, 121, 128), (5, 32, 2048, 768, 180, 256)])
def test_larger_tiles_by_blocks(top, E, d, F, r, rows):
    """Tiles of 192 rows past 130 expected rows where the blocks of 64 weight rows take two thirds of the 512 places."""
    assert tile_rows(round(r * E / top), top, E, d, F, torch.bfloat16) == rows


@pytest.mark.parametrize("E,d,F,rows", [(8, 4608, 2304, 256), (8, 5120, 2560, 256), (12, 3072, 2304, 256), (6, 5632, 2816, 256), (9, 4096, 2048, 256),
                                        (8, 4096, 2560, 128), (8, 4096, 2048, 128), (8, 6144, 2048, 128), (6, 5120, 5120, 128)])
def test_one_round_of_wide_blocks(E, d, F, rows):
    """Wide blocks at 50 rows an expert where both products' are one round of more than half of the CUs."""
    assert tile_rows(25 * E, 2, E, d, F, torch.bfloat16) == rows
