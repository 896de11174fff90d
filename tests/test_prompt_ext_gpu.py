"""A prompt layer's operators in the extension module: the bits of the same functions in Python over the forms that both take, and None
for what is Python's."""
import ctypes

import pytest
import torch

from kubernetes_cloud_amd import ops
from kubernetes_cloud_amd.ops import _lib
from kubernetes_cloud_amd.ops import linear as L
from kubernetes_cloud_amd.ops.norms import layer_norm
from kubernetes_cloud_amd.ops.rope import rope_tables
from kubernetes_cloud_amd.utils import capture

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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 33, 128])
@pytest.mark.parametrize("n,k,k2", [(16, 64, 64), (4096, 1024, 4096)])
def test_few_rows_and_residual_rows(monkeypatch, dtype, rows, n, k, k2):
    a = _rand(1, rows, k, dtype=dtype), _rand(n, k, dtype=dtype), _rand(n, dtype=dtype)
    b, res = (_rand(rows, k2, dtype=dtype), _rand(n, k2, dtype=dtype), None), _rand(rows, n, dtype=dtype)
    _both(monkeypatch, lambda: L.few_rows_sum(a, b, res=res), "few_rows")


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


def test_modes_it_leaves():
    """Transforms, tracing, torch's modes and (few_rows) captures, on types that the module's functions take otherwise."""
    ext = _lib.torch_ext()
    x, w, b = _rand(8, 128), _rand(96, 128), _rand(96)
    few = lambda x=x: ext.few_rows(x, w, b, None, None, None, 0, 0, False, 8)  # noqa: E731
    norm = lambda x=x, w=_rand(128), r=None: ext.norm_rows(x, w, None, 1e-5, r, None)  # noqa: E731
    with torch.no_grad():
        assert few() is not None and norm() is not None

        def under(t):
            assert few(t) is None and norm(t) is None and norm(r=t) is None
            return t
        assert torch.equal(torch.func.vmap(under)(x[None]), x[None])
        torch.func.jvp(under, (x,), (x,))
        torch.jit.trace(under, (x,), check_trace=False)

        class Dispatch(torch.utils._python_dispatch.TorchDispatchMode):
            def __torch_dispatch__(self, f, types, args=(), kwargs=None):
                return f(*args, **(kwargs or {}))

        class Function(torch.overrides.TorchFunctionMode):
            def __torch_function__(self, f, types, args=(), kwargs=None):
                return f(*args, **(kwargs or {}))
        for mode in (Dispatch, Function):
            with mode():
                under(x)
        with capture.graph(torch.cuda.CUDAGraph(), stream=torch.cuda.Stream()):
            taken = few(), norm()
        assert taken[0] is None and taken[1] is not None  # (slices of K have the stream's counters)


def _prompt(T=40, H=2, D=64, dtype=torch.bfloat16):
    at = torch.arange(T, device="cuda", dtype=torch.int32)
    kc = torch.zeros(4, H, 16, D, device="cuda", dtype=dtype)
    return dict(zip("qkv", _rand(T, 3, H, D, dtype=dtype).unbind(1)), cos=_rand(64, 16).float(), sin=_rand(64, 16).float(), pos=at, page=at // 16,
                off=at % 16, kc=kc, vc=kc.clone(), cu=torch.tensor([0, T], device="cuda", dtype=torch.int32))


def test_what_rotation_and_attention_leave():
    ext, p = _lib.torch_ext(), _prompt()

    def rope(**kw):
        a = {**p, **kw}
        return ext.rope_append(a["q"], a["k"], a["v"], 32, False, *(a[n] for n in ("cos", "sin", "pos", "page", "off", "kc", "vc")))

    def attend(max_len=40, **kw):
        a = {**p, **kw}
        return ext.packed_attention(a["q"], a["k"], a["v"], a["cu"], max_len, 0.125, 0)

    def odd(t):  # its values, rows off 16 bytes
        s = torch.empty(t.shape[0], t.shape[1], t.shape[2] + 4, device="cuda", dtype=t.dtype)[..., 1:-3]
        s.copy_(t)
        return s
    assert rope() is None and attend() is None  # gradients
    with torch.no_grad():
        assert rope() is True and attend() is not None
        twice = torch.stack([p["pos"], p["pos"]], 1)[:, 0]
        for n in ("pos", "page", "off"):
            for bad in (p[n].long(), p[n][:-1], p[n].cpu(), twice, p[n].float()):
                assert rope(**{n: bad}) is None
        for n in "qkv":
            for bad in (p[n].float(), p[n].half(), p[n][:-1], p[n].cpu(), p[n].transpose(1, 2).contiguous().transpose(1, 2), p[n][..., :56], p[n][0]):
                assert rope(**{n: bad}) is None and attend(**{n: bad}) is None
        for bad in (p["kc"].float(), p["kc"][:2], p["kc"][:, :1], p["kc"].transpose(0, 1), p["kc"].cpu()):
            assert rope(kc=bad) is None and rope(vc=bad) is None
        assert rope(cos=None) is None and rope(sin=p["sin"].half()) is None and rope(cos=p["cos"][:, ::2]) is None
        for bad in (p["cu"].long(), p["cu"].cpu(), p["cu"][:1], torch.stack([p["cu"], p["cu"]], 1)[:, 0]):
            assert attend(cu=bad) is None
        assert attend(max_len=0) is None
        # the kernels' own checks: nothing is done, as for the same call from Python
        before = p["q"].clone(), p["kc"].clone()
        assert rope(k=odd(p["k"])) is False and torch.equal(p["q"], before[0]) and torch.equal(p["kc"], before[1])
        half = {n: p[n].half() for n in "qkv"}
        assert attend(**half) is not None
        with pytest.raises(RuntimeError, match="status"):
            attend(**{**half, "k": odd(half["k"])})
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert rope() is None and attend() is None

        def under(q):
            assert rope(q=q) is None and attend(q=q) is None
            return q
        torch.func.vmap(under)(p["q"][None])
        torch.jit.trace(under, (p["q"],), check_trace=False)


def test_alibi_is_python_s(monkeypatch):
    p, slopes = _prompt(), torch.tensor([0.5, 0.25], device="cuda")
    _both(monkeypatch, lambda: ops.packed_attention(p["q"], p["k"], p["v"], p["cu"], 40, None, slopes), None)


def test_stream_and_capture():
    """Launches go to the stream that is current, into a capture's graph too."""
    p, w = _prompt(), _rand(64)
    x, big = _rand(8, 64), _rand(4096, 1024)
    side = torch.cuda.Stream()
    with torch.no_grad():
        def go(x, q):
            kc = torch.zeros_like(p["kc"])
            assert ops.rope_append(q, p["k"].clone(), p["v"], 32, False, p["cos"], p["sin"], p["pos"], p["page"], p["off"], kc, kc.clone())
            return layer_norm(x, w, None), ops.packed_attention(q, p["k"], p["v"], p["cu"], 40), kc
        want = go(x, p["q"].clone())
        few = L.few_rows_gelu(_rand(8, 1024), big, None, "tanh")
        torch.cuda.synchronize()
        with torch.cuda.stream(side):  # (memory of its own)
            go(x, p["q"].clone()), L.few_rows_gelu(_rand(8, 1024), big, None, "tanh")
        torch.cuda.synchronize()
        torch.cuda._sleep(200_000_000)  # (the side stream's work is done before the default stream's)
        tail = torch.cuda.Event()
        tail.record()
        with torch.cuda.stream(side):
            got, z = go(x, p["q"].clone()), L.few_rows_gelu(_rand(8, 1024), big, None, "tanh")
        side.synchronize()
        assert not tail.query() and torch.equal(z, few) and all(torch.equal(a, b) for a, b in zip(got, want))
        graph, q = torch.cuda.CUDAGraph(), p["q"].clone()
        with capture.graph(graph, stream=torch.cuda.Stream()):
            out = layer_norm(x, w, None), ops.packed_attention(q, p["k"], p["v"], p["cu"], 40)
        for i in range(3):
            x.copy_(_rand(8, 64, seed=i))
            graph.replay()
            assert torch.equal(out[0], layer_norm(x, w, None)) and torch.equal(out[1], ops.packed_attention(q, p["k"], p["v"], p["cu"], 40))


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 64, 65, 128])
def test_both_ask_the_kernel_for_the_same(monkeypatch, rows):
    """The module works out a launch's slices, scratch and counters by itself: what it hands to the kernel is what Python hands to it."""
    ext, lib, asked = _lib.torch_ext(), _lib._load(), []
    types = lib.kca_rows_mm_two.argtypes
    stand_in = ctypes.CFUNCTYPE(ctypes.c_int, *types)(lambda *a: asked.append(a) or 0)
    address = lambda f: ctypes.cast(f, ctypes.c_void_p).value  # noqa: E731
    real = [address(getattr(lib, n)) for n in _lib._ROWS]
    monkeypatch.setattr(_lib, "call", lambda name, *a: asked.append(a))
    shapes = lambda a: [bool(v) if t is ctypes.c_void_p else v for t, v in zip(types, a)]  # noqa: E731
    try:
        ext.init_rows(address(stand_in), *real[1:], _lib.counters)
        with torch.no_grad():
            for n, k, n2, k2 in [(16, 64, 16, 64), (64, 512, 80, 1024), (1040, 2048, 1040, 576), (4096, 16384, 4096, 4096), (8128, 1088, 8320, 1024),
                                 (16384, 1024, 16384, 2048), (5120, 5120, 15360, 5120), (2048, 8192, 2048, 2048)]:
                a, b = ((torch.empty(rows, kk, device="cuda", dtype=torch.bfloat16), torch.empty(nn, kk, device="cuda", dtype=torch.bfloat16), None)
                        for nn, kk in ((n, k), (n2, k2)))
                res = torch.empty(rows, n, device="cuda", dtype=torch.bfloat16)
                for f in (lambda: L.few_rows_beside(a, b, "tanh"), lambda: L.few_rows_gelu(*a, "none"), lambda: L.few_rows_sum(a, b, res=res)):
                    asked.clear()
                    took = f() is not None
                    with monkeypatch.context() as mp:
                        mp.setattr(_lib, "_torch_ext", [None])
                        assert (f() is not None) == took
                    assert len(asked) == 2 * took
                    if took:
                        assert shapes(asked[0]) == shapes(asked[1])
    finally:
        ext.init_rows(*real, _lib.counters)


