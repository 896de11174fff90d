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
