"""fp16 prompts on the native kernels: packed attention with softmax weights of 24 bits, LayerNorm rows and GELU against
float64 or float32, and the gradient, strided and odd calls that stay torch's."""
import pytest
import torch
import torch.nn.functional as F

from kubernetes_cloud_amd import ops
from kubernetes_cloud_amd.ops import _lib

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -11  # half a unit of fp16


@pytest.mark.parametrize("D,alibi,window", [(64, False, 0), (80, False, 0), (96, False, 33), (128, True, 0), (160, False, 0), (256, False, 0),
                                            (256, True, 40)])
def test_packed_attention(D, alibi, window):
    lens, H = [1, 129, 31, 300, 256, 64], 3
    g = torch.Generator(device="cuda").manual_seed(D)
    qkv = torch.randn(sum(lens), 3, H, D, device="cuda", generator=g).half()
    q, k, v = qkv.unbind(1)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], device="cuda", dtype=torch.int32)
    sl = 2.0 ** (-torch.arange(1, H + 1, device="cuda").float()) if alibi else None
    o = ops.packed_attention(q, k, v, cu, max(lens), alibi=sl, window=window)
    for a, b in zip(cu.tolist(), cu.tolist()[1:]):
        n = b - a
        i = torch.arange(n, device="cuda")
        z = torch.einsum("qhd,khd->hqk", q[a:b].double(), k[a:b].double()) * D ** -0.5
        if alibi:
            z = z + sl.double()[:, None, None] * (i[None] - i[:, None])
        seen = (i[None] <= i[:, None]) & ((i[None] > i[:, None] - window) if window else True)
        p = z.masked_fill(~seen, -torch.inf).softmax(-1)
        want = torch.einsum("hqk,khd->qhd", p, v[a:b].double())
        # the result's rounding; scores in 32 bits (products of up to 256 terms) and weights of 24 bits under it
        size = torch.einsum("hqk,khd->qhd", p, v[a:b].double().abs())
        assert ((o[a:b].double() - want).abs() <= EPS * want.abs() + 2.0 ** -17 * size + 2.0 ** -24).all()


def test_weights_over_the_whole_range():
    """Scores from 2^-100 to 2^8 of the first tile's: what a running maximum moves, and what falls below fp16."""
    n = 300
    q = torch.zeros(n, 1, 64, device="cuda", dtype=torch.half)
    k, v = torch.zeros_like(q), torch.randn(n, 1, 64, device="cuda").half()
    q[..., 0] = 8.0
    k[:, 0, 0] = torch.linspace(-60, 12, n).half()
    cu = torch.tensor([0, n], device="cuda", dtype=torch.int32)
    o = ops.packed_attention(q, k, v, cu, n)
    z = (q[:, 0].double() @ k[:, 0].double().T) * 64 ** -0.5
    p = z.masked_fill(torch.ones(n, n, device="cuda").triu(1).bool(), -torch.inf).softmax(-1)
    want, size = p @ v[:, 0].double(), p @ v[:, 0].double().abs()
    assert ((o[:, 0].double() - want).abs() <= EPS * want.abs() + 2.0 ** -17 * size + 2.0 ** -24).all()


@pytest.mark.parametrize("rows,d", [(1, 64), (3, 768), (61, 4096), (700, 2048), (5, 16384)])
@pytest.mark.parametrize("residuals,bias", [(0, True), (1, True), (2, False)])
def test_layer_norm(rows, d, residuals, bias):
    g = torch.Generator(device="cuda").manual_seed(rows)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g).half()  # noqa: E731
    x, w, b, res = r(1, rows, d), r(d), r(d) if bias else None, tuple(r(1, rows, d) for _ in range(residuals))
    before = _lib.LAUNCHES[0]
    with torch.no_grad():
        out = ops.layer_norm(x, w, b, 1e-5, residual=res)
    assert _lib.LAUNCHES[0] == before + 1
    y, h = out if residuals else (out, x)
    s = x.double() + sum(t.double() for t in res)
    assert y.shape == x.shape and h.shape == x.shape
    assert ((h.double() - s).abs() <= EPS * s.abs() + 2.0 ** -22).all()  # one rounding of a sum in 32 bits
    want = F.layer_norm(h.double(), (d,), w.double(), None if b is None else b.double(), 1e-5)
    assert ((y.double() - want).abs() <= EPS * want.abs() + 2.0 ** -11 * w.double().abs() * EPS + 1e-4).all()


@pytest.mark.parametrize("kind", ["tanh", "none"])
def test_gelu(kind):
    u = torch.linspace(-12, 12, 8 * 4001, device="cuda").half()
    before = _lib.LAUNCHES[0]
    with torch.no_grad():
        y = ops.gelu(u, kind)
    assert _lib.LAUNCHES[0] == before + 1
    want = F.gelu(u.double(), approximate=kind)
    # one rounding; the 32-bit 1 + tanh cancels to a few 2^-23 of u
    assert ((y.double() - want).abs() <= EPS * want.abs() + 2.0 ** -21 * u.double().abs() + 2.0 ** -24).all()


def test_calls_that_stay_torch():
    x = torch.randn(4, 24, device="cuda").half()
    w = torch.randn(24, device="cuda").half()
    before = _lib.LAUNCHES[0]
    assert ops.gelu(x.clone().requires_grad_()).requires_grad
    assert ops.layer_norm(x.clone().requires_grad_(), w, None).requires_grad
    with torch.no_grad():
        odd = torch.randn(3, 20, device="cuda").half()
        ops.layer_norm(odd, odd[0].clone(), None)
        ops.layer_norm(x[:, ::2], w[::2], None)
        ops.gelu(x[:, :7])
        assert torch.allclose(torch.vmap(lambda r: ops.gelu(r, "tanh"))(x).float(), F.gelu(x.float(), approximate="tanh"), atol=2e-3)
    assert _lib.LAUNCHES[0] == before
