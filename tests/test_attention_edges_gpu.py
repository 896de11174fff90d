"""The general forms of the tiled attention kernels at the sizes where they can go wrong: edges of tiles and blocks, one
row, lengths of zero, windows narrower than a tile, more keys than queries, grouped heads, rows that are not 16-byte
aligned (which the generic kernels take) -- against the fp32 reference."""
import pytest
import torch

from kubernetes_cloud_amd.ops.attention import attention_reference, flash_attention

pytestmark = pytest.mark.gpu

# bf16 operands P and dS (relative error 2^-9 each, uncorrelated over a row's keys) and one rounding of the result:
# under 3 * 2^-9 in the 2-norm
TOL = 3 * 2.0 ** -9


def _buffer(B, S, H, D, g, pad=0, shift=0):
    """[B, S, H, D] inside a larger buffer of NaN: what lies past the last row must not be used."""
    big = torch.full((B * (S + 40) * H * (D + pad) + shift + 64,), float("nan"), device="cuda", dtype=torch.bfloat16)
    t = torch.as_strided(big, (B, S, H, D), ((S + 40) * H * (D + pad), H * (D + pad), D + pad, 1), shift)
    t.copy_(torch.randn(B, S, H, D, device="cuda", generator=g))
    return t


def _close(a, b):
    a, b = a.float(), b.float()
    assert torch.isfinite(a).all()
    floor = 2.0 ** -17 * b.numel() ** 0.5  # where a gradient cancels to nothing: fp32 sums of 256 products of order one
    assert (a - b).norm() <= TOL * b.norm() + floor, ((a - b).norm() / b.norm()).item()


def _check(B, Sq, Sk, H, Hkv, D, causal, lens=None, window=0, alibi=False, pad=0, shift=0):
    g = torch.Generator(device="cuda").manual_seed(Sq * 7 + Sk)
    q, do = _buffer(B, Sq, H, D, g, pad, shift), torch.randn(B, Sq, H, D, device="cuda", generator=g).bfloat16()
    k, v = _buffer(B, Sk, Hkv, D, g, pad, shift), _buffer(B, Sk, Hkv, D, g, pad, shift)
    ln = torch.tensor(lens, device="cuda", dtype=torch.int32) if lens else None
    sl = 2.0 ** (-torch.arange(1, H + 1, device="cuda").float()) if alibi else None
    x = [t.detach().requires_grad_() for t in (q, k, v)]
    o = flash_attention(*x, causal=causal, kv_len=ln, window=window, alibi=sl)
    gr = torch.autograd.grad(o, x, do)
    y = [t.detach().float().contiguous().requires_grad_() for t in (q, k, v)]
    r, lse = attention_reference(*y, causal, None, ln, sl, window)
    _close(o, r)
    # rows that see no key: their gradient is zero, which the reference's autograd does not give
    seen = torch.isfinite(lse).transpose(1, 2)[..., None]
    dm = do.float() * seen
    ref = _reference_grads(*y, dm, causal, ln, sl, window)
    for a, b in zip(gr, ref):
        _close(a, b)


def _reference_grads(q, k, v, do, causal, ln, sl, window):
    with torch.no_grad():
        B, Sq, H, D = q.shape
        Sk, rep = k.shape[1], H // k.shape[2]
        kk, vv = k.repeat_interleave(rep, 2), v.repeat_interleave(rep, 2)
        s = torch.einsum("bqhd,bkhd->bhqk", q, kk) * D ** -0.5
        qi, ki = torch.arange(Sq, device="cuda")[:, None] + Sk - Sq, torch.arange(Sk, device="cuda")[None]
        ok = torch.ones(B, 1, Sq, Sk, dtype=torch.bool, device="cuda")
        if causal:
            ok &= ki <= qi
        if window:
            ok &= ki > qi - window
        if ln is not None:
            ok &= ki < ln.view(B, 1, 1, 1)
        if sl is not None:
            s = s + sl.view(1, H, 1, 1) * (ki - qi)
        p = torch.softmax(s.masked_fill(~ok, -1e30), -1) * ok
        dv = torch.einsum("bhqk,bqhd->bkhd", p, do)
        dp = torch.einsum("bqhd,bkhd->bhqk", do, vv)
        ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * D ** -0.5
        dq, dk = torch.einsum("bhqk,bkhd->bqhd", ds, kk), torch.einsum("bhqk,bqhd->bkhd", ds, q)
        fold = lambda t: t.view(B, Sk, H // rep, rep, D).sum(3)  # noqa: E731
        return dq, fold(dk), fold(dv)


@pytest.mark.parametrize("D", [64, 96, 128, 160, 256])
@pytest.mark.parametrize("S", [1, 31, 33, 127, 129, 257, 300])
def test_causal_lengths(D, S):
    _check(2, S, S, 3, 3, D, True)


@pytest.mark.parametrize("D", [64, 96, 128, 160, 256])
def test_masks(D):
    _check(3, 200, 200, 2, 2, D, True, lens=[200, 33, 0])
    _check(2, 300, 300, 2, 2, D, True, window=40)
    _check(2, 300, 300, 2, 2, D, True, window=7, lens=[300, 64])
    _check(1, 261, 261, 4, 4, D, True, alibi=True)
    _check(2, 256, 256, 4, 4, D, True, alibi=True, lens=[129, 256])
    _check(1, 290, 290, 2, 2, D, True, alibi=True, window=100)


@pytest.mark.parametrize("D", [64, 96, 128, 160, 256])
def test_other_counts(D):
    _check(2, 70, 333, 2, 2, D, True)             # a chunk after a cached prefix
    _check(1, 128, 159, 2, 2, D, True)
    _check(2, 130, 77, 2, 2, D, False)            # cross attention, more queries than keys
    _check(2, 64, 200, 2, 2, D, False, lens=[200, 96])
    _check(1, 190, 190, 4, 2, D, True)            # grouped heads
    _check(1, 190, 190, 4, 2, D, True, alibi=True, lens=[150])


def test_rows_off_16_bytes():
    """Strides or bases that 16-byte loads do not fit keep the generic kernels."""
    _check(1, 140, 140, 2, 2, 64, True, pad=4)
    _check(1, 140, 140, 2, 2, 64, True, shift=4)


@pytest.mark.parametrize("early", [60.0, -60.0])
@pytest.mark.parametrize("D", [96, 128, 256])
@pytest.mark.parametrize("alibi", [False, True])
def test_late_score_far_above_the_reference(early, D, alibi):
    """A row whose first key of the walk scores 2^100 times lower than another one is recomputed by the generic kernel."""
    q = torch.zeros(1, 200, 1, D, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros_like(q)
    v = torch.randn(1, 200, 1, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(0)).bfloat16()
    q[..., 0], k[0, 3, 0, 0], k[0, 150, 0, 0] = 40.0, early, -early
    sl = torch.full((1,), 0.25, device="cuda") if alibi else None
    o = flash_attention(q, k, v, causal=True, alibi=sl)
    _close(o, attention_reference(q, k, v, True, None, None, sl)[0])


@pytest.mark.parametrize("D,window,tiles", [(64, 0, 1), (96, 0, 1), (256, 0, 1), (128, 256, 2), (256, 256, 2)])
def test_error_against_64_bits(D, window, tiles):
    """No further off than softmax weights in bf16 relative to the largest of a row's first tiles of 32 keys, as the generic
    kernels take them, a sum in 32 bits and one rounding of the result. (Over four million values the two errors' own spread is
    about 0.1 %; a reference out of 16 keys on average, a row's last tile, is 1 % above.)"""
    S, H = 1100, 16
    q, k, v = (torch.randn(4, S, 3, H, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(D))).bfloat16().unbind(2)
    i = torch.arange(S, device="cuda")
    seen = (i[None] <= i[:, None]) & ((i[None] > i[:, None] - window) if window else True)
    first = ((i - window + 1).clamp(min=0) if window else torch.zeros_like(i))[:, None] // 32
    near = seen & (i[None] // 32 < first + tiles)
    with torch.no_grad():
        o = flash_attention(q, k, v, causal=True, window=window).double()
    mine, other = 0.0, 0.0
    for b in range(4):
        z = torch.matmul(q[b].transpose(0, 1).double(), k[b].permute(1, 2, 0).double()) * D ** -0.5
        x = v[b].transpose(0, 1).double()
        want = torch.matmul(z.masked_fill(~seen, -torch.inf).softmax(-1), x)
        p = torch.exp(z - z.masked_fill(~near, -torch.inf).amax(-1, keepdim=True)).float() * seen
        ref = (torch.matmul(p.bfloat16().double(), x) / p.double().sum(-1, keepdim=True)).bfloat16().double()
        mine += float((o[b].transpose(0, 1) - want).square().sum())
        other += float((ref - want).square().sum())
    assert mine ** 0.5 <= 1.003 * other ** 0.5, (mine ** 0.5 / other ** 0.5)
