"""``flash_attention``'s autograd function in C++ against the one in Python: the same kernels, so the same bits; and what stays
with the Python one or behaves as it did (hooks on saved tensors, transforms, tangents, freed graphs, changed inputs, streams,
threads)."""
import threading

import pytest
import torch
from torch.autograd import forward_ad

from kubernetes_cloud_amd.ops import _lib
from kubernetes_cloud_amd.ops import attention as A

pytestmark = pytest.mark.gpu


def _inputs(B=2, S=150, H=4, Hkv=4, D=64, seed=0, grad=True):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = [torch.randn(B, S, h, D, device="cuda", generator=g).bfloat16().requires_grad_(grad) for h in (H, Hkv, Hkv)]
    return t, torch.randn(B, S, H, D, device="cuda", generator=g).bfloat16()


def _python(q, k, v, causal=True, kv_len=None, alibi=None, window=0):
    return A._FlashAttnFn.apply(q, k, v, causal, q.shape[-1] ** -0.5, A.native_mask(kv_len, q.device), alibi, window)


def test_extension_is_there():
    assert _lib.torch_ext() is not None
    (q, k, v), _ = _inputs()
    assert "FlashAttnFn" not in type(A.flash_attention(q, k, v, causal=True).grad_fn).__name__


@pytest.mark.parametrize("kw", [{}, {"causal": False}, {"window": 40}, {"kv_len": [150, 33]}, {"alibi": True}, {"kv_len": "bitmap"},
                                {"Hkv": 2}, {"D": 256}, {"D": 80}])
def test_same_bits(kw):
    kw = dict(kw)
    shape = {n: kw.pop(n) for n in ("Hkv", "D") if n in kw}
    (q, k, v), do = _inputs(**shape)
    if kw.get("kv_len") == "bitmap":
        kw["kv_len"] = torch.rand(2, 150, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)) > 0.3
        kw["kv_len"][:, 0] = True
    elif "kv_len" in kw:
        kw["kv_len"] = torch.tensor(kw["kv_len"], device="cuda")
    if "alibi" in kw:
        kw["alibi"] = 2.0 ** -torch.arange(1, 5, device="cuda").float()
    causal = kw.pop("causal", True)
    for up in (do, do.transpose(1, 2).contiguous().transpose(1, 2), do[:, :1].expand_as(do)):
        o, p = A.flash_attention(q, k, v, causal=causal, **kw), _python(q, k, v, causal, **kw)
        assert torch.equal(o, p) and o.stride() == p.stride()
        for a, b in zip(torch.autograd.grad(o, (q, k, v), up, retain_graph=True), torch.autograd.grad(p, (q, k, v), up)):
            assert torch.equal(a, b) and a.stride() == b.stride()
    with torch.no_grad():
        n = A.flash_attention(q, k, v, causal=causal, **kw)
    assert torch.equal(n, o) and not n.requires_grad
    (gk,) = torch.autograd.grad(A.flash_attention(q.detach(), k, v.detach(), causal=causal, **kw), (k,), do)
    assert torch.equal(gk, torch.autograd.grad(o, (k,), do)[0])


def test_hooks_on_saved_tensors_and_checkpoints():
    (q, k, v), do = _inputs()
    want = torch.autograd.grad(A.flash_attention(q, k, v, causal=True), (q, k, v), do)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        o = A.flash_attention(q, k, v, causal=True)
    assert len(seen) >= 5
    for a, b in zip(torch.autograd.grad(o, (q, k, v), do), want):
        assert torch.equal(a, b)
    o = torch.utils.checkpoint.checkpoint(lambda *t: A.flash_attention(*t, causal=True), q, k, v, use_reentrant=False)
    for a, b in zip(torch.autograd.grad(o, (q, k, v), do), want):
        assert torch.equal(a, b)


def test_freed_graphs_and_changed_inputs():
    (q, k, v), do = _inputs()
    o = A.flash_attention(q, k, v, causal=True)
    torch.autograd.grad(o, (q, k, v), do)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, (q, k, v), do)
    x = q * 1.0
    o = A.flash_attention(x, k, v, causal=True)
    x.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(o, (q, k, v), do)


def test_what_is_not_plain_stays_with_the_python_function():
    (q, k, v), do = _inputs()

    def both(f):
        """Result or the kind of error of a call through either function."""
        out = []
        for g in (lambda *t: A.flash_attention(*t, causal=True), _python):
            try:
                out.append(f(g))
            except Exception as e:  # noqa: BLE001
                out.append(type(e))
        return out

    def tangent(g):
        with forward_ad.dual_level():
            return g(forward_ad.make_dual(q, torch.ones_like(q)), k, v)

    def mapped(g):
        return torch.vmap(lambda a: g(a, k, v))(torch.stack([q, q]))

    def gradient(g):
        return torch.func.grad(lambda a: g(a, k, v).float().sum())(q)

    class Sub(torch.Tensor):
        pass

    for f in (tangent, mapped, gradient, lambda g: g(q.as_subclass(Sub), k, v)):
        a, b = both(f)
        assert (a is b) if isinstance(a, type) else torch.equal(a, b)
    with pytest.raises(ValueError):
        A.flash_attention(*(t.detach()[..., :12] for t in (q, k, v)), causal=True)
    with pytest.raises(RuntimeError, match="status"):
        A.flash_attention(q, k[:, :, :3], v[:, :, :3], causal=True)  # 4 heads over 3


def test_streams_and_threads():
    (q, k, v), do = _inputs(S=700)
    want = [t.clone() for t in torch.autograd.grad(A.flash_attention(q, k, v, causal=True), (q, k, v), do)]
    torch.cuda.synchronize()
    bad = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(5):
                got = torch.autograd.grad(A.flash_attention(q, k, v, causal=True), (q, k, v), do)
                s.synchronize()
                bad.extend(not torch.equal(a, b) for a, b in zip(got, want))

    ts = [threading.Thread(target=work) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert len(bad) == 60 and not any(bad)
