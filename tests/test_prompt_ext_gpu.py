"""A prompt layer's operators in the extension module: the bits of the same functions in Python over the forms that both take, and None
for what is Python's."""
import pytest
import torch

from kubernetes_cloud_amd import ops
from kubernetes_cloud_amd.ops import _lib
from kubernetes_cloud_amd.ops import linear as L
from kubernetes_cloud_amd.ops.norms import layer_norm
from kubernetes_cloud_amd.ops.rope import rope_tables

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available() or _lib.torch_ext() is None, reason="not built")]


def _rand(*shape, dtype=torch.bfloat16, seed=1):
    return torch.empty(shape, device="cuda", dtype=dtype).normal_(generator=torch.Generator(device="cuda").manual_seed(seed + sum(shape)))


def _both(monkeypatch, f, name):
    """f() on the module, which has to take it, and in Python."""
    ext, took = _lib.torch_ext(), []

    class Spy:
        def __getattr__(self, n):
            g = getattr(ext, n)
            return lambda *a: (lambda r: (took.append(n) if r is not None else None, r)[1])(g(*a))
    with torch.no_grad(), monkeypatch.context() as mp:
        mp.setattr(_lib, "_torch_ext", [Spy()])
        before = _lib.LAUNCHES[0]
        a = f()
        launches = _lib.LAUNCHES[0] - before
        assert took == ([name] if name else [])
        mp.setattr(_lib, "_torch_ext", [None])
        b = f()
        assert launches == _lib.LAUNCHES[0] - before - launches
    assert type(a) is type(b) or isinstance(a, tuple)
    for x, y in zip(a if isinstance(a, (tuple, list)) else [a], b if isinstance(b, (tuple, list)) else [b]):
        assert (x is None and y is None) or torch.equal(x, y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 33, 128])
@pytest.mark.parametrize("n,k,n2,k2", [(16, 64, 80, 64), (4096, 1024, 4096, 4096), (3072, 1024, 4096, 1024)])
def test_few_rows(monkeypatch, dtype, rows, n, k, n2, k2):
    a = _rand(1, rows, k, dtype=dtype), _rand(n, k, dtype=dtype), _rand(n, dtype=dtype)
    b = _rand(rows, k2, dtype=dtype), _rand(n2, k2, dtype=dtype), None
    _both(monkeypatch, lambda: L.few_rows_beside(a, b, "tanh"), "few_rows")
    _both(monkeypatch, lambda: L.few_rows_gelu(*a, "none"), "few_rows")
    _both(monkeypatch, lambda: L.few_rows_sum(a, b), "few_rows" if n == n2 else None)
    res = _rand(rows, n, dtype=dtype)
    _both(monkeypatch, lambda: L.few_rows_sum(a, b, res=res), "few_rows" if n == n2 else None)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [8, 512, 2040, 16384])
@pytest.mark.parametrize("residuals", [0, 1, 2])
def test_norm_rows(monkeypatch, dtype, d, residuals):
    x, *r = (_rand(1, 7, d, dtype=dtype, seed=i) for i in range(1 + residuals))
    w, b = _rand(d, dtype=dtype), _rand(d, dtype=dtype, seed=9)
    _both(monkeypatch, lambda: layer_norm(x, w, b, 1e-5, tuple(r)), "norm_rows")
    _both(monkeypatch, lambda: layer_norm(x, w, None, 1e-5, tuple(r)), "norm_rows")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,rot,inter,window", [(256, 64, True, 0), (64, 0, False, 40), (96, 24, False, 0)])
def test_rotation_and_attention(monkeypatch, dtype, D, rot, inter, window):
    lens, H = [30, 7, 65], 3
    T = sum(lens)
    cu = torch.tensor([0, 30, 37, 102], device="cuda", dtype=torch.int32)
    pos = torch.cat([torch.arange(n) for n in lens]).to("cuda", torch.int32)
    first = torch.tensor([0, 5, 10], device="cuda").repeat_interleave(torch.tensor(lens, device="cuda"))  # a sequence's first page
    page, off = (pos // 16 + first).int(), (pos % 16).int()
    page[-1] = -1
    cos, sin = rope_tables(rot, 128, 10000.0, "cuda") if rot else (None, None)
    qkv = _rand(T, 3, H, D, dtype=dtype)

    def go():
        x, kc = qkv.clone(), torch.zeros(20, H, 16, D, device="cuda", dtype=dtype)
        vc = kc.clone()
        assert ops.rope_append(*x.unbind(1), rot, inter, cos, sin, pos, page, off, kc, vc)
        return x, kc, vc
    _both(monkeypatch, go, "rope_append")
    _both(monkeypatch, lambda: ops.packed_attention(*qkv.unbind(1), cu, 65, None, None, window), "packed_attention")


def test_what_it_leaves(monkeypatch):
    ext = _lib.torch_ext()
    x, w, b = _rand(8, 128), _rand(96, 128), _rand(96)
    few = lambda x=x, w=w, b=b, rows=8: ext.few_rows(x, w, b, None, None, None, 0, 0, False, rows)  # noqa: E731
    norm = lambda x=x, w=_rand(128), b=None, r=None: ext.norm_rows(x, w, b, 1e-5, r, None)  # noqa: E731
    assert few() is None and norm() is None  # gradients
    with torch.no_grad():
        assert few() is not None and norm() is not None and norm(r=x) is not None
        for y in (few(x.float()), few(x[:, :64]), few(x, w[:90]), few(x, w[:, :64]), few(rows=7), few(x, w.half()), few(b=b[:90]), few(b=b.float()),
                  few(_rand(1025)[1:].view(8, 128)), few(x.cpu()),
                  norm(x.float()), norm(x.t()), norm(w=_rand(120)), norm(w=_rand(128).float()), norm(b=_rand(120)), norm(r=x[:4]), norm(r=x.half()),
                  norm(_rand(1025)[1:].view(8, 128)), norm(x[:0])):
            assert y is None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert few() is None and norm() is None
        import torch.autograd.forward_ad as fwAD
        with fwAD.dual_level():
            assert norm(fwAD.make_dual(x, x)) is None

        class Sub(torch.Tensor):
            pass
        assert few(x.as_subclass(Sub)) is None and norm(x.as_subclass(Sub)) is None
        assert torch.func.vmap(lambda t: layer_norm(t, x[0], None))(x[None].float()).shape == (1, 8, 128)


