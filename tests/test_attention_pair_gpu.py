"""256-wide heads: the backward, whose waves work in pairs -- one, two and three tiles a walk, blocks that nobody sees, walks over
several query heads -- and the forward with four waves a block, against the fp32 reference (bounds as in
test_attention_edges_gpu.py)."""
import pytest
import torch

from kubernetes_cloud_amd.ops import attention as A

from .test_attention_edges_gpu import _check, _close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Sq,Sk", [(1, 1), (31, 31), (33, 33), (64, 64), (65, 97), (96, 300), (128, 128), (129, 257), (260, 260)])
def test_walks(Sq, Sk, causal):
    _check(2, Sq, Sk, 3, 3, 256, causal)
    _check(2, Sq, Sk, 4, 2, 256, causal)


@pytest.mark.parametrize("causal", [True, False])
def test_masks(causal):
    _check(7, 290, 290, 2, 2, 256, causal, lens=[290, 0, 1, 127, 128, 129, 33])
    if causal:
        _check(2, 290, 290, 4, 1, 256, True, lens=[200, 31], alibi=True)
        for window in (1, 32, 33, 150):
            _check(2, 290, 290, 4, 2, 256, True, window=window)
        _check(2, 140, 330, 4, 1, 256, True, window=64, alibi=True)


@pytest.mark.parametrize("S", [40, 200])
def test_keys_past_the_length_are_not_read(S):
    """What lies behind a sequence's length may be anything, and gets no gradient: one tile a walk, and tiles requested ahead of the last."""
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v, do = (torch.randn(3, S, 2, 256, device="cuda", generator=g).bfloat16() for _ in range(4))
    ln = torch.tensor([S, S - 37, 1], device="cuda", dtype=torch.int32)
    gone = torch.arange(S, device="cuda")[None] >= ln[:, None]

    def grads():
        t = [x.clone().requires_grad_() for x in (q, k, v)]
        return torch.autograd.grad(A.flash_attention(*t, causal=True, kv_len=ln), t, do)
    want = grads()
    k[gone], v[gone] = float("nan"), float("inf")
    got = grads()
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    assert not got[1][gone].any() and not got[2][gone].any()


def test_rows_off_16_bytes():
    """Full tiles in rows that 16-byte loads do not fit keep the kernels of one wave a block."""
    g = torch.Generator(device="cuda").manual_seed(1)
    t = [torch.randn(1, 128, 2, 260, device="cuda", generator=g).bfloat16()[..., 2:258] for _ in range(3)]
    grads = []
    for off in (False, True):
        q, k, v = (x.requires_grad_() if off else x.detach().contiguous().requires_grad_() for x in (y.detach() for y in t))
        A.flash_attention(q, k, v, causal=True).float().square().sum().backward()
        grads.append((q.grad, k.grad, v.grad))
    for a, b in zip(*grads):
        assert (a.float() - b.float()).norm() <= 3 * 2.0 ** -9 * b.float().norm()


@pytest.mark.parametrize("H", [3, 40])
@pytest.mark.parametrize("S", [128, 129, 256, 330, 384, 600, 640])
def test_four_waves(S, H):
    """Forward in blocks of 128 rows, two workgroups a CU: odd and even counts of blocks, edges, masks; and whole blocks of 256."""
    _check(2, S, S, H, H, 256, True)
    _check(2, S, S + 31, H, 1, 256, True, window=100)
    _check(2, S, S, H, H, 256, True, alibi=True, lens=[S, S - 77])


@pytest.mark.parametrize("alibi", [False, True])
def test_four_waves_far_above_their_first_tile(alibi):
    """A late key far above a row's first tile: the rows are computed again in the same launch."""
    S, H, D = 640, 8, 256
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v = (torch.randn(3, S, H, D, device="cuda", generator=g) * 0.3 for _ in range(3))
    k[0, 200, 1] = q[0, 600, 1] * 40.0
    q, k, v = (x.bfloat16() for x in (q, k, v))
    sl = torch.full((H,), 0.25, device="cuda") if alibi else None
    o, lse = A._fwd(q, k, v, True, D ** -0.5, None, sl)
    r, want = A.attention_reference(*(t[:1, :, :2].float() for t in (q, k, v)), True, None, None, None if sl is None else sl[:2])
    _close(o[:1, :, :2], r)
    torch.testing.assert_close(lse[:1, :2], want, rtol=2.0 ** -18, atol=2.0 ** -16)  # (as in test_attention_split_gpu.py)


@pytest.mark.parametrize("H", [16, 40])
def test_a_window_divides_by_the_rounded_weights(H):
    """One key whose weight is 2^25 times all others' and no row's reference: a row is that key's value to the bit, for the rounding of
    its weight cancels, with the keys in two groups (16 heads) as in one."""
    S, D, at = 2048, 256, (500, 1600)
    q, k, v = (torch.zeros(1, S, H, D, device="cuda") for _ in range(3))
    q[..., 0] = 1
    v.copy_(1 + torch.rand(v.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(0)))
    for j in at:
        k[0, j, :, 0] = 16 * (18 + 0.25 * torch.arange(H, device="cuda"))  # (every head's weight rounds differently)
    q, k, v = (t.bfloat16() for t in (q, k, v))
    with torch.no_grad():
        o = A.flash_attention(q, k, v, causal=True, window=1024)
    for j in at:
        end = min(S, j + 1024)
        assert torch.equal(o[0, j:end], v[0, j].expand(end - j, H, D))


def test_variants_are_two_kernels():
    """``set_variant(0)`` takes the register-staged forward where the other one walks keys in two groups, whose sums are added in
    another order: not the same bits."""
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn(2, 1024, 3, 256, device="cuda", generator=g).bfloat16() for _ in range(3))
    outs = []
    for var in (1, 0):
        old = A.set_variant(var)
        try:
            with torch.no_grad():
                outs.append(A.flash_attention(q, k, v, causal=True))
        finally:
            A.set_variant(old)
    assert not torch.equal(*outs)
    _close(*outs)
