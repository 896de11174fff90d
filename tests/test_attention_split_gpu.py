"""Attention whose blocks split their keys over wave groups, and the same kernels with one group, which calls of many blocks
take: odd sizes around the tiles of 32, the blocks of 64 and 128 rows and the groups' strides, against the fp32 reference
(bounds as in test_attention_edges_gpu.py)."""
import pytest
import torch

from kubernetes_cloud_amd.ops.attention import _fwd, attention_reference, flash_attention

from .test_attention_edges_gpu import _check, _close

pytestmark = pytest.mark.gpu
FEW, MANY = (2, 3), (13, 48)  # batch, heads: of MANY every size here has more blocks than the split calls


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("S", [32, 65, 96, 130, 161])
def test_one_group(D, S):
    B, H = MANY
    _check(B, S, S, H, H, D, True)


@pytest.mark.parametrize("Sq,Sk", [(128, 128), (384, 384), (256, 512)])
def test_full_tiles_of_many_blocks(Sq, Sk):
    """64-wide heads: the plain forms of the backward, up to 384 keys and past 384 blocks, and the split ones beside them."""
    _check(10, Sq, Sk, 20, 10, 64, True)
    _check(20, Sq, Sk, 96 if Sq == 128 else 48, 48, 64, True)


@pytest.mark.parametrize("D", [64, 96, 128, 256])
def test_one_group_masks(D):
    B, H = MANY
    _check(B, 150, 150, H, H, D, True, lens=[150, 33, 0, 1, 64, 65, 31, 32, 150, 149, 128, 129, 96])
    _check(B, 170, 170, H, H, D, True, window=40)
    _check(B, 140, 140, H, H, D, True, alibi=True, window=70)
    _check(B, 40, 171, H, H, D, True)
    _check(B, 130, 130, H, H // 3, D, True, alibi=True)


@pytest.mark.parametrize("D", [64, 96, 128, 256])
@pytest.mark.parametrize("S", [63, 97, 193, 290, 417])
def test_two_groups(D, S):
    B, H = FEW
    _check(B, S, S, H, H, D, True, window=33)
    _check(B, S, S, H, H, D, True, alibi=True, lens=[S, S - 40])
    _check(B, S, S + 37, H, 1, D, True)


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("S", [127, 193, 225, 257, 290])
def test_tiles_in_turn(D, S):
    """Walks of 1 to 10 tiles over the places that they take in turn, one group and two."""
    for B, H in ((6, 48), (1, 2)):
        _check(B, S, S, H, H, D, True)
        _check(B, S, S, H, H, D, True, alibi=True)


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("B,H", [(2, 3), (13, 48)])
def test_rows_past_the_length_are_not_read(D, B, H):
    """What lies behind a sequence's length may be anything."""
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(B, 200, H, D, device="cuda", generator=g).bfloat16() for _ in range(3))
    ln = torch.tensor([200 - 17 * (b % 12) for b in range(B)], device="cuda", dtype=torch.int32)
    gone = torch.arange(200, device="cuda")[None] >= ln[:, None]
    want = flash_attention(q, k, v, causal=True, kv_len=ln)
    k[gone], v[gone] = float("nan"), float("inf")
    assert torch.equal(flash_attention(q, k, v, causal=True, kv_len=ln), want)


def test_eight_waves_dkdv():
    """128-wide heads between the two: dK/dV of 128 keys in two groups of four waves."""
    _check(5, 400, 400, 10, 10, 128, True)
    _check(5, 400, 400, 10, 10, 128, True, alibi=True, window=150)
    _check(5, 390, 520, 20, 10, 128, True, lens=[520, 0, 1, 129, 511])


@pytest.mark.parametrize("D", [64, 96, 128, 256])
@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("alibi", [False, True])
def test_rows_far_above_their_first_tile(D, many, alibi):
    """A late key that scores 2^900 times above a row's first tile: the rows are computed again with their true maximum, in the
    same launch, and the rows beside them keep their results."""
    S = 333
    B, H = (MANY if many else FEW)
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v = (torch.randn(B, S, H, D, device="cuda", generator=g) * 0.3 for _ in range(3))
    k[0, 200, 1] = q[0, 320, 1] * 40.0
    q, k, v = (t.bfloat16() for t in (q, k, v))
    sl = torch.full((H,), 0.25, device="cuda") if alibi else None
    o, lse = _fwd(q, k, v, True, D ** -0.5, None, sl)
    r, want = attention_reference(*(t[:1, :, :2].float() for t in (q, k, v)), True, None, None, None if sl is None else sl[:2])
    _close(o[:1, :, :2], r)
    # sums of up to 256 products in fp32, in another order: 16 roundings of 2^-24 on average, four times that
    torch.testing.assert_close(lse[:1, :2], want, rtol=2.0 ** -18, atol=2.0 ** -16)


@pytest.mark.parametrize("D", [64, 256])
def test_not_a_number_stays_in_its_rows(D):
    q, k, v = (torch.randn(1, 300, 2, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(i)).bfloat16()
               for i in range(3))
    want = flash_attention(q, k, v, causal=True)
    q[0, 70, 1] = float("nan")
    o = flash_attention(q, k, v, causal=True)
    assert torch.isnan(o[0, 70, 1]).all()
    o[0, 70, 1] = want[0, 70, 1]
    # (the row's block takes its true maxima: other rows of it are rounded relative to another weight)
    _close(o, want)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("scale", [0.0, -0.07, 1e-25, 0.2])
def test_scales(D, scale):
    """No scale, a negative one, hardly any (dK's sums start with lse over it) and a large one."""
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v, do = (torch.randn(13, 130, 48, D, device="cuda", generator=g).bfloat16() for _ in range(4))
    x = [t[:, :, :6].contiguous().requires_grad_() if D == 128 else t.requires_grad_() for t in (q, k, v)]
    do = do[:, :, :x[0].shape[2]].contiguous()
    o = flash_attention(*x, causal=True, scale=scale)
    gr = torch.autograd.grad(o, x, do)
    y = [t[:2, :, :3].detach().float().contiguous().requires_grad_() for t in x]
    r, _ = attention_reference(*y, True, scale)
    ref = torch.autograd.grad(r, y, do[:2, :, :3].float())
    for a, b in zip(gr, ref):
        _close(a[:2, :, :3], b)


@pytest.mark.parametrize("mask", ["ragged", "keys", "lens", "window", "alibi", "none"])
@pytest.mark.parametrize("D", [64, 96, 128, 160, 256])
def test_column_of_ones(D, mask):
    """A causal call that names V's column of ones has a result of its own whatever the mask and the size."""
    S = 200 if mask == "ragged" else 256
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v = (torch.randn(2, S + (40 if mask == "keys" and i else 0), 3, D, device="cuda", generator=g).bfloat16() for i in range(3))
    v[..., 40] = 1
    ln = torch.tensor([S, 77], device="cuda", dtype=torch.int32) if mask == "lens" else None
    sl = 2.0 ** -torch.arange(1, 4, device="cuda").float() if mask == "alibi" else None
    window = 50 if mask == "window" else 0
    # (what the allocator hands out next is zero: as overflow marks it leaves no row to the generic kernel)
    free = [torch.zeros(n, device="cuda", dtype=torch.uint8) for n in (*[512] * 64, *[65536] * 16, *[2 * S * 3 * D * 2] * 4)]
    del free
    with torch.no_grad():
        o = flash_attention(q, k, v, causal=True, kv_len=ln, alibi=sl, window=window, rowsum_col=40)
    _close(o, attention_reference(q.float(), k.float(), v.float(), True, None, ln, sl, window)[0])


@pytest.mark.parametrize("D,B,S,H,window,groups", [
    (64, 4, 320, 12, 69, 2), (64, 5, 228, 20, 49, 2), (128, 1, 360, 14, 92, 2), (128, 2, 320, 14, 91, 2), (96, 8, 251, 12, 96, 2),  # few blocks
    (64, 10, 320, 32, 69, 1), (128, 5, 832, 14, 159, 1), (96, 1, 2419, 20, 134, 1),                                                # many
    (64, 1, 1600, 32, 0, 2), (64, 1, 1280, 64, 0, 1), (64, 12, 97, 12, 0, 2), (64, 40, 97, 12, 0, 1), (96, 1, 2048, 20, 0, 2), (96, 16, 181, 12, 0, 1),
    (128, 1, 1280, 30, 0, 2), (128, 1, 1280, 40, 0, 1), (64, 12, 512, 8, 0, 2), (64, 6, 600, 13, 0, 1),
    (96, 7, 192, 12, 0, 2), (96, 11, 192, 8, 0, 1), (96, 11, 192, 12, 0, 2), (128, 11, 192, 8, 0, 1), (128, 5, 220, 25, 0, 1), (128, 8, 221, 12, 0, 2), (96, 11, 192, 8, 60, 2)])
def test_which_calls_are_split(D, B, S, H, window, groups):
    """A windowed call is split by the keys that its blocks see, not by the window alone; results in either form."""
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(B, S, H, D, device="cuda", generator=g).bfloat16() for _ in range(3))
    with torch.no_grad(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        o = flash_attention(q, k, v, causal=True, window=window)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages() if "attn_fwd_split_kernel" in e.key]
    assert len(names) == 1 and f"<{D}, 1, {4 // groups}, {groups}, " in names[0], names
    _close(o, attention_reference(q.float(), k.float(), v.float(), causal=True, window=window)[0])


@pytest.mark.parametrize("B,S,H,plain", [(10, 256, 20, True), (16, 256, 12, False), (11, 384, 12, True), (4, 384, 32, False), (10, 512, 20, False), (4, 1024, 20, False)])
def test_which_backwards_are_plain(B, S, H, plain):
    """64-wide heads, full tiles."""
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(B, S, H, 64, device="cuda", generator=g).bfloat16().requires_grad_() for _ in range(3))
    o = flash_attention(q, k, v, causal=True)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        o.backward(torch.ones_like(o))
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages() if "attn_bwd_dq" in e.key or "attn_bwd_dkdv" in e.key]
    assert len(names) == 2 and all(("_tiled_" if plain else "_split_") in n for n in names), names
