"""The forward of 256-wide heads in each of its forms, at calls that take it: 256 rows and eight waves a block (plain, with lengths, ALiBi or ragged
sizes, packed prompts), keys in two groups (lengths, windows, ALiBi), and rows that are computed again in each; 96-wide heads with a
window in two groups. Against the fp32 reference (bounds as in test_attention_edges_gpu.py). Which form a call takes hangs on its
blocks of 128 and 256 rows (attention_tiled.hip): few of either for two groups, from 512 of 128 rows on eight waves."""
import pytest
import torch

from kubernetes_cloud_amd import ops
from kubernetes_cloud_amd.ops import attention as A

from .test_attention_edges_gpu import _check, _close

pytestmark = pytest.mark.gpu
D = 256


def _forward(B, Sq, Sk, H, seed, Hkv=None, **kw):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(B, s, h, D, device="cuda", generator=g).bfloat16() for s, h in ((Sq, H), (Sk, Hkv or H), (Sk, Hkv or H)))
    return q, k, v, *A._fwd(q, k, v, True, D ** -0.5, kw.get("lens"), kw.get("slopes"), window=kw.get("window", 0))


def _compare(q, k, v, o, lse, rows=slice(None), heads=slice(None), **kw):
    sl = kw.get("slopes")
    ln = kw.get("lens")
    r, want = A.attention_reference(*(t[rows][:, :, heads].float() for t in (q, k, v)), True, None, None if ln is None else ln[rows],
                                    None if sl is None else sl[heads], kw.get("window", 0))
    _close(o[rows][:, :, heads], r)
    seen = torch.isfinite(want)
    # (as in test_attention_split_gpu.py)
    torch.testing.assert_close(lse[rows, heads][seen], want[seen], rtol=2.0 ** -18, atol=2.0 ** -16)


def _slopes(H):
    return 2.0 ** (-8.0 * torch.arange(1, H + 1, device="cuda").float() / H)


# ------------------------------------------------------------------- eight waves, 256 rows
@pytest.mark.parametrize("S,B,H", [(1024, 5, 13), (1024, 1, 70), (1536, 3, 15)])
def test_eight_waves_plain(S, B, H):
    _compare(*_forward(B, S, S, H, 1))


def test_eight_waves_more_keys_than_queries():
    _compare(*_forward(3, 1024, 1280, 24, 2))


@pytest.mark.parametrize("S", [897, 1000, 1279])
def test_eight_waves_ragged(S):
    _compare(*_forward(5, S, S, 15, S))


@pytest.mark.parametrize("S", [1152, 1920])
def test_eight_waves_half_a_last_block(S):
    """Full tiles whose last block of 256 rows is half empty."""
    _compare(*_forward(4, S, S, 20 if S < 1500 else 12, S))


@pytest.mark.parametrize("S", [1024, 1000])
def test_eight_waves_masks(S):
    B, H = 6, 12
    ln = torch.tensor([S, 0, 1, 255, 257, S - 300], device="cuda", dtype=torch.int32)
    _compare(*_forward(B, S, S, H, 3, lens=ln), lens=ln)
    _compare(*_forward(B, S, S, H, 4, slopes=_slopes(H), lens=ln), slopes=_slopes(H), lens=ln)
    _compare(*_forward(B, S, S + 70, H, 5, slopes=_slopes(H)), slopes=_slopes(H))
    _compare(*_forward(B, S, S, H, 6, window=500), window=500)


@pytest.mark.parametrize("kind", ["plain", "ragged", "lens", "alibi", "window"])
def test_eight_waves_compute_rows_again(kind):
    """A late key far above a row's first tile: the block's rows are taken once more with their true maxima."""
    S, B, H = 1000 if kind == "ragged" else 1024, 5, 13
    g = torch.Generator(device="cuda").manual_seed(7)
    q, k, v = (torch.randn(B, S, H, D, device="cuda", generator=g) * 0.3 for _ in range(3))
    k[1, 700, 2] = q[1, 950, 2] * 40.0
    q, k, v = (t.bfloat16() for t in (q, k, v))
    kw = {"lens": {"lens": torch.tensor([S, S - 1, 300, S, S], device="cuda", dtype=torch.int32)},
          "alibi": {"slopes": torch.full((H,), 0.25, device="cuda")},
          "window": {"window": 600}}.get(kind, {})
    o, lse = A._fwd(q, k, v, True, D ** -0.5, kw.get("lens"), kw.get("slopes"), window=kw.get("window", 0))
    _compare(q, k, v, o, lse, slice(0, 3), slice(0, 4), **kw)


@pytest.mark.parametrize("window", [0, 500])
@pytest.mark.parametrize("alibi", [False, True])
def test_eight_waves_packed(alibi, window):
    lens, H = [1000, 1, 257, 700, 31, 1000, 512], 11
    g = torch.Generator(device="cuda").manual_seed(8)
    q, k, v = torch.randn(sum(lens), 3, H, D, device="cuda", generator=g).bfloat16().unbind(1)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], device="cuda", dtype=torch.int32)
    sl = _slopes(H) if alibi else None
    o = ops.packed_attention(q, k, v, cu, max(lens), alibi=sl, window=window)
    for a, b in zip(cu.tolist(), cu.tolist()[1:]):
        _close(o[a:b], A.attention_reference(*(t[None, a:b].float() for t in (q, k, v)), True, None, None, sl, window)[0][0])


# ------------------------------------------------------------------- two groups of keys
@pytest.mark.parametrize("S", [901, 960, 1024, 1100, 1500])
def test_two_groups(S):
    _compare(*_forward(2, S, S, 4, S))
    _compare(*_forward(1, S, S + 45, 4, S, Hkv=2))


def test_two_groups_masks():
    B, S, H = 4, 1000, 4
    ln = torch.tensor([S, 33, 0, 990], device="cuda", dtype=torch.int32)
    _compare(*_forward(B, S, S, H, 1, lens=ln), lens=ln)
    _compare(*_forward(B, S, S, H, 2, slopes=_slopes(H), lens=ln), slopes=_slopes(H), lens=ln)
    for w in (901, 950, 1600):
        _compare(*_forward(2, 1800, 1800, H, 3, window=w), window=w)
    _compare(*_forward(2, 1300, 1700, H, 4, window=1000, slopes=_slopes(H)), window=1000, slopes=_slopes(H))


@pytest.mark.parametrize("kind", ["plain", "lens", "alibi", "window"])
def test_two_groups_compute_rows_again(kind):
    B, S, H = 2, 1100, 4
    g = torch.Generator(device="cuda").manual_seed(9)
    q, k, v = (torch.randn(B, S, H, D, device="cuda", generator=g) * 0.3 for _ in range(3))
    k[0, 700, 1] = q[0, 1050, 1] * 40.0
    q, k, v = (t.bfloat16() for t in (q, k, v))
    kw = {"lens": {"lens": torch.tensor([S - 1, 300], device="cuda", dtype=torch.int32)},
          "alibi": {"slopes": torch.full((H,), 0.25, device="cuda")},
          "window": {"window": 1000}}.get(kind, {})
    o, lse = A._fwd(q, k, v, True, D ** -0.5, kw.get("lens"), kw.get("slopes"), window=kw.get("window", 0))
    _compare(q, k, v, o, lse, **kw)


# ------------------------------------------------------------------- 96 wide, a window in two groups
@pytest.mark.parametrize("window", [66, 100, 129])
@pytest.mark.parametrize("S", [193, 290, 417])
def test_two_groups_of_a_window(S, window):
    _check(2, S, S, 3, 3, 96, True, window=window)
    _check(2, S, S + 37, 4, 2, 96, True, window=window, lens=[S, S - 40])
