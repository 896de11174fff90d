"""Long products without gradients run as whole waves of blocks and a rest: the rule, and the rows' values."""
import pytest
import torch
import torch.nn.functional as F

from kubernetes_cloud_amd.ops.linear import FEW_ROWS, TLinear, few_rows, linear_rows, wave_rows


@pytest.mark.parametrize("n,k", [(4096, 4096), (4096, 16384), (12288, 4096), (16384, 4096), (8192, 2048), (6144, 2048),
                                 (2048, 8192), (50400, 4096), (256, 4096), (100, 2048), (4096, 1024)])
def test_parts_cover_the_rows(n, k):
    for rows in list(range(1, 300, 37)) + list(range(1900, 20000, 61)) + [2048, 2049, 4096, 4097, 8192]:
        first = wave_rows(rows, n, k)
        assert 0 < first <= rows
        if first < rows:
            assert rows > 2048 and k >= 2048
            blocks = first // 256 * -(-n // 256)
            assert first % 256 == 0 and blocks % 256 == 0


@pytest.mark.parametrize("n,k,last", [(64, 64, 128), (1280, 1280, 128), (4096, 16384, 128), (12288, 4096, 128), (16384, 4096, 128),
                                      (14336, 14336, 64), (6144, 24576, 128), (18432, 6144, 24), (50400, 4096, 24)])
def test_few_rows(n, k, last):
    # eager calls up to a number of rows; a capture takes no other ones
    eager, graph = ([few_rows(r, n, k, c) for r in range(1, 200)] for c in (False, True))
    assert eager == [r <= last for r in range(1, 200)] and last <= FEW_ROWS
    assert all(e or not g for e, g in zip(eager, graph))


def test_other_calls_stay_one_product(monkeypatch):
    """Off the GPU, and with gradients, the module is F.linear."""
    lin = TLinear(2048, 4096)
    x = torch.randn(3, 2048)
    with torch.no_grad():
        assert torch.equal(lin(x), F.linear(x, lin.weight, lin.bias))
        assert torch.equal(torch.vmap(lin)(x), torch.vmap(lambda r: F.linear(r, lin.weight, lin.bias))(x))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,n,bias", [((2049, 2048), 16384, True), ((1, 4097, 2048), 4096, False),
                                          ((2, 2900, 2048), 4096, True), ((3, 1383, 4096), 4096, True),
                                          ((2304, 4096), 8192, False), ((2048, 4096), 16384, True)])
def test_rows_against_float32(dtype, shape, n, bias):
    g = torch.Generator(device="cuda").manual_seed(7)
    k = shape[-1]
    x = torch.empty(shape, device="cuda", dtype=dtype).normal_(generator=g)
    w = torch.empty(n, k, device="cuda", dtype=dtype).normal_(std=k ** -0.5, generator=g)
    b = torch.empty(n, device="cuda", dtype=dtype).normal_(generator=g) if bias else None
    with torch.no_grad():
        y = linear_rows(x, w, b)
        ref = F.linear(x.float(), w.float(), None if b is None else b.float())
    assert y.shape == ref.shape and y.dtype == dtype and y.is_contiguous()
    # one rounding to the type, of a sum whose own error in 32 bits is below sqrt(k) * 2^-24 of its terms' size
    eps = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11
    assert ((y.float() - ref).abs() <= eps * ref.abs() + 1e-4).all()
    # a call that may record gradients is F.linear
    assert torch.equal(linear_rows(x, w, b), F.linear(x, w, b))
