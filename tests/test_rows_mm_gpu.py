"""Products of few rows on the weight-streaming kernel (csrc/kernels/rows_mm.hip) against float32."""
import pytest
import torch
import torch.nn.functional as F

from kubernetes_cloud_amd.ops import _lib
from kubernetes_cloud_amd.ops.linear import _k_slices, _rows_mm, few_rows, few_rows_beside, linear_rows
from kubernetes_cloud_amd.utils import capture

pytestmark = pytest.mark.gpu


def _inputs(rows, n, k, dtype, bias, seed=3):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.empty(rows, k, device="cuda", dtype=dtype).normal_(generator=g)
    w = torch.empty(n, k, device="cuda", dtype=dtype).normal_(std=k ** -0.5, generator=g)
    b = torch.empty(n, device="cuda", dtype=dtype).normal_(generator=g) if bias else None
    return x, w, b, F.linear(x.float(), w.float(), None if b is None else b.float())


def _close(y, ref):
    # one rounding to the type; the 32-bit sums of terms of size k^-1/2 are good to well below 1e-4
    eps = 2.0 ** -8 if y.dtype is torch.bfloat16 else 2.0 ** -11
    return ((y.float() - ref).abs() <= eps * ref.abs() + 1e-4).all().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 15, 32, 33, 64, 65, 127, 128])
@pytest.mark.parametrize("n,k,bias", [(16, 64, True), (80, 192, False), (4096, 1024, True), (2048, 4160, True), (12304, 512, False)])
def test_rows_against_float32(dtype, rows, n, k, bias):
    x, w, b, ref = _inputs(rows, n, k, dtype, bias)
    before = _lib.LAUNCHES[0]
    with torch.no_grad():
        y = linear_rows(x, w, b)
        again = linear_rows(x, w, b)
    assert _lib.LAUNCHES[0] == before + 2 and _close(y, ref) and torch.equal(y, again)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 2, 3])
@pytest.mark.parametrize("n,k", [(16, 64), (4096, 1984), (4112, 1984), (4112, 2048), (1040, 8192), (1040, 8256), (272, 16448),
                                 (16384, 1984), (16384, 2048), (12288, 4096)])
def test_one_and_two_rows(dtype, rows, n, k, monkeypatch):
    """On both sides of the lines between the vector kernel and the rows' one; eager, and replayed where a capture takes them (the others are
    the library's there)."""
    x, w, b, ref = _inputs(rows, n, k, dtype, True)
    call, names = _lib.call, []
    monkeypatch.setattr(_lib, "call", lambda name, *a: (names.append(name), call(name, *a))[1])
    bf16 = dtype == torch.bfloat16
    vector = (rows == 1 or (rows == 2 and bf16 and k <= 8192)) and (k >= 2048 or n <= 4096)
    own = ("kca_skinny_gemm" if bf16 else "kca_skinny_gemm_f16") if vector else "kca_rows_mm"
    captured = few_rows(rows, n, k, True)
    assert captured == ((n, k) in [(16, 64), (16384, 1984), (16384, 2048), (12288, 4096)])
    with torch.no_grad():
        y = linear_rows(x, w, b)
        assert _close(y, ref) and _close(linear_rows(x, w), F.linear(x.float(), w.float())) and names == [own] * 2
        graph = torch.cuda.CUDAGraph()
        with capture.graph(graph, stream=torch.cuda.Stream()):
            z = linear_rows(x, w, b)
        assert names == [own] * (3 if captured else 2)
        for _ in range(3):
            z.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert _close(z, ref) and torch.equal(linear_rows(x, w, b), y) and (not captured or torch.equal(z, y))


@pytest.mark.parametrize("rows,n,k", [(61, 4096, 4096), (128, 4096, 4096)])
def test_slices_under_capture_and_on_streams(rows, n, k):
    """The slices' counters: two streams at once, and a graph beside eager calls of its stream."""
    assert _k_slices(n, k) > 1 and few_rows(rows, n, k) and few_rows(rows, n, k, True)
    x, w, b, ref = _inputs(rows, n, k, torch.bfloat16, True)
    main, side = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.no_grad():
        outs = []
        for _ in range(20):
            for s in (main, side):
                with torch.cuda.stream(s):
                    outs.append(linear_rows(x, w, b))
        torch.cuda.synchronize()
        assert all(torch.equal(o, outs[0]) for o in outs) and _close(outs[0], ref)
        for s in (main, torch.cuda.Stream()):  # a stream with a workspace, and one that has none yet
            graph = torch.cuda.CUDAGraph()
            with capture.graph(graph, stream=s):
                y = linear_rows(x, w, b)
            for _ in range(3):
                y.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, outs[0])
                assert torch.equal(linear_rows(x, w, b), outs[0])


def test_what_it_does_not_take():
    x, w, b, _ = _inputs(8, 96, 128, torch.bfloat16, True)
    with torch.no_grad():
        before = _lib.LAUNCHES[0]
        for args in ((x, w[:90], b[:90]), (x[:, :120], w[:, :120], b), (x.float(), w.float(), b.float()), (x[:0], w, b)):
            assert torch.allclose(linear_rows(*args).float(), F.linear(*args).float(), atol=0.05)
        assert _lib.LAUNCHES[0] == before
        assert _rows_mm(x, w[:90], b[:90]) is None
    p = torch.nn.Parameter(w)
    assert linear_rows(x, p, b).requires_grad
    with pytest.raises(RuntimeError):
        _lib.call("kca_rows_mm", 1, x.data_ptr(), w.data_ptr(), None, x.data_ptr(), None, None, 0, 0, 129, 96, 128, 1, _lib.stream())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [3, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k", [(16384, 320), (16400, 64), (16400, 192), (24560, 448), (32768, 320), (32784, 128), (49152, 64), (49168, 576)])
def test_blocks_of_64_and_128_weight_rows(dtype, rows, n, k):
    """On both sides of the lines between the blocks, their last ones partly filled, in walks shorter and longer than the stages in LDS that
    start at any of them."""
    x, w, b, ref = _inputs(rows, n, k, dtype, True)
    with torch.no_grad():
        y = _rows_mm(x, w, b)
        assert _close(y, ref) and torch.equal(y, _rows_mm(x, w, b))
        assert _close(_rows_mm(x, w, None), F.linear(x.float(), w.float()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [3, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(50400, 320), (51216, 64), (57344, 192), (57360, 128)])
def test_blocks_of_112_weight_rows(dtype, rows, n, k):
    """Seven waves, some of which request a piece of the activations that another one requests too; the last one is back at blocks of 128."""
    x, w, b, ref = _inputs(rows, n, k, dtype, True)
    x2, w2, b2, ref2 = _inputs(rows, 48, 64, dtype, True, 4)
    with torch.no_grad():
        y = _rows_mm(x, w, b)
        assert _close(y, ref) and torch.equal(y, _rows_mm(x, w, b))
        if rows <= 24:  # (more rows of so many outputs are the library's beside another product)
            for got, want in zip(few_rows_beside((x, w, b), (x2, w2, b2), None), (ref, ref2)):
                assert _close(got, want)


@pytest.mark.parametrize("rows", [5, 61, 100])
@pytest.mark.parametrize("n,k,n2,k2", [(12304, 192, 4096, 640), (8192, 64, 8208, 320), (16384, 320, 16, 64)])
def test_two_products_in_wide_blocks(rows, n, k, n2, k2):
    x, w, b, ref = _inputs(rows, n, k, torch.bfloat16, True)
    x2, w2, b2, ref2 = _inputs(rows, n2, k2, torch.bfloat16, True, 4)
    with torch.no_grad():
        y, y2 = few_rows_beside((x, w, b), (x2, w2, b2), None)
    assert _close(y, ref) and _close(y2, ref2)
