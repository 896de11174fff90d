"""Sizes past the kernels' 32-bit byte offsets: the entry points refuse them before any launch, and the dispatch does not send
them there."""
import pytest
import torch

from kubernetes_cloud_amd.ops import _lib

built = pytest.mark.skipif(not _lib.available(), reason="kernel library not built")
A = 1 << 20  # an aligned address that nothing reads


@built
@pytest.mark.parametrize("rows,n,k", [(128, 16, 1 << 25), (16, 128, 1 << 25), (128, 112, 1 << 24)])
def test_rows_product(rows, n, k):
    from kubernetes_cloud_amd.ops.linear import _rows_mm
    assert 2 * max(rows, n) * k >= 1 << 32
    assert _lib.call_rc("kca_rows_mm", 1, A, A, None, A, None, None, 0, 0, rows, n, k, 1, None) == 3
    t = lambda *s: torch.empty(*s, device="meta", dtype=torch.bfloat16)  # noqa: E731
    assert _rows_mm(t(rows, k), t(n, k), None) is None


@pytest.mark.parametrize("d,F,E,top", [(4096, 4096, 16, 2), (8192, 64, 4, 1), (16384, 65536, 2, 2), (2048, 768, 24, 5), (72, 200, 8, 2)])
def test_expert_tiles(d, F, E, top):
    """Whatever the number of tokens, the tiles are as many as the expert products take, and past 32-bit offsets they are of the
    one kind that has longer ones."""
    from kubernetes_cloud_amd.ops.moe import tile_rows
    for T in [1, 5, 17, 40, 300, 4096, 16384, 65536, 131072, 262144, 500000, 1000000 // top * 4]:
        mt, n = tile_rows(T, top, E, d, F, torch.bfloat16), T * top
        assert min(E, n) + n // mt <= 32767, T
        if 2 * T * d >= 1 << 31 or 4 * F * d >= 1 << 32:
            assert mt == 128 or (mt <= 8 and n <= 16 * E)
