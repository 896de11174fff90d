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
