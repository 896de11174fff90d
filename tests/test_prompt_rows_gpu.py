"""Prompts without padding: packed attention at edges of tiles and blocks, rotation with page writes against the separate
rotation and copies, and the runner's packed prompts against one prompt at a time."""
import pytest
import torch

from kubernetes_cloud_amd import ops
from kubernetes_cloud_amd.engine.runner import KVCache, ModelRunner
from kubernetes_cloud_amd.models.causal_lm import build_model
from kubernetes_cloud_amd.models.config import LMConfig
from kubernetes_cloud_amd.ops.attention import attention_reference
from kubernetes_cloud_amd.ops.rope import apply_rotary_, rope_tables

pytestmark = pytest.mark.gpu
TOL = 3 * 2.0 ** -9  # bf16 probabilities and results (tests/test_attention_edges_gpu.py)


@pytest.mark.parametrize("D,alibi,window", [(64, False, 0), (80, False, 0), (96, False, 0), (128, True, 0), (128, False, 40),
                                            (256, False, 0), (256, True, 33)])
def test_packed_attention(D, alibi, window):
    lens, H = [1, 129, 31, 300, 256, 64], 3
    g = torch.Generator(device="cuda").manual_seed(D)
    T = sum(lens)
    qkv = torch.randn(T, 3, H, D, device="cuda", generator=g).bfloat16()
    q, k, v = qkv.unbind(1)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], device="cuda", dtype=torch.int32)
    sl = 2.0 ** (-torch.arange(1, H + 1, device="cuda").float()) if alibi else None
    o = ops.packed_attention(q, k, v, cu, max(lens), alibi=sl, window=window)
    for a, b in zip(cu.tolist(), cu.tolist()[1:]):
        r = attention_reference(*(t[None, a:b] for t in (q, k, v)), True, None, None, sl, window)[0][0].float()
        assert (o[a:b].float() - r).norm() <= TOL * r.norm()


@pytest.mark.parametrize("early", [60.0, -60.0])
@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("alibi", [False, True])
def test_packed_attention_overflowing_rows(early, D, alibi):
    """Rows whose reference is 2^100 below a later score are recomputed in their own sequence."""
    lens = [40, 200]
    q = torch.zeros(240, 1, D, device="cuda", dtype=torch.bfloat16)
    k, v = torch.zeros_like(q), torch.randn(240, 1, D, device="cuda").bfloat16()
    q[..., 0], k[45, 0, 0], k[230, 0, 0] = 40.0, early, -early
    cu = torch.tensor([0, 40, 240], device="cuda", dtype=torch.int32)
    sl = torch.full((1,), 0.25, device="cuda") if alibi else None
    o = ops.packed_attention(q, k, v, cu, 200, alibi=sl)
    r = attention_reference(q[None, 40:], k[None, 40:], v[None, 40:], True, None, None, sl)[0][0].float()
    assert (o[40:].float() - r).norm() <= TOL * r.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,rot,inter", [(256, 64, True), (80, 20, False), (96, 24, False), (64, 64, False), (128, 0, False),
                                         (64, 18, True)])
@pytest.mark.parametrize("page_size", [0, 16])
def test_rope_append(dtype, D, rot, inter, page_size):
    H, lens, slots, start = 3, [5, 40, 1], [2, 0, 3], [0, 3, 17]
    c = KVCache(1, 4, H, 64, D, "cuda", dtype, page_size=page_size)
    ref = KVCache(1, 4, H, 64, D, "cuda", dtype, page_size=page_size)
    for s, n, p in zip(slots, lens, start):
        c.reserve(s, n + p)
        ref.reserve(s, n + p)
    page, off, pos = (torch.from_numpy(x).cuda() for x in c.rows(slots, lens, start))
    T = sum(lens)
    qkv = torch.randn(T, 3, H, D, device="cuda").to(dtype)
    page[4] = -1  # padding
    want = qkv.clone()
    q, k, v = want.unbind(1)
    cos, sin = rope_tables(rot, 64, 10000.0, "cuda") if rot else (None, None)
    if rot:  # in fp32 on one row of tokens, as the eager path does
        c_, s_ = cos[pos.long()], sin[pos.long()]
        from kubernetes_cloud_amd.ops.rope import _rotate_ref
        q.copy_(_rotate_ref(q, c_, s_, inter, 1.0))
        k.copy_(_rotate_ref(k, c_, s_, inter, 1.0))
    for i in range(T):
        if i != 4:
            ref.k[0][page[i], :, off[i]] = k[i]
            ref.v[0][page[i], :, off[i]] = v[i]
    assert ops.rope_append(*qkv.unbind(1), rot, inter, cos, sin, pos, page, off, c.k[0], c.v[0])
    # one rounding; a fused multiply-add may move a value to its neighbour
    tol = dict(rtol=2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10, atol=2.0 ** -9)
    torch.testing.assert_close(qkv, want, **tol)
    torch.testing.assert_close(c.k[0], ref.k[0], **tol)
    assert torch.equal(c.v[0], ref.v[0])


@pytest.mark.parametrize("D,rot,inter", [(256, 64, True), (128, 64, False), (64, 36, False), (64, 20, True)])
def test_rope_append_rounds_one_product_first(D, rot, inter):
    """Bit for bit a product in fp32 and a fused multiply-add of the other one (pairs side by side: w c first, then u s). Which of
    the two comes first shows in one of some 1e5 elements. (fp16 rounds some fused multiply-adds once, some twice.)"""
    T, H, half, dtype = 3001, 16, rot // 2, torch.bfloat16
    c = KVCache(1, 1, H, T, D, "cuda", dtype, page_size=0)
    page, off, pos = (torch.from_numpy(x).cuda() for x in c.rows([0], [T], [0]))
    qkv = torch.randn(T, 3, H, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).to(dtype)
    cos, sin = rope_tables(rot, T, 10000.0, "cuda")
    want = qkv.clone()
    x = want[:, :2, :, :rot]
    u, w = (x[..., 0::2], x[..., 1::2]) if inter else (x[..., :half], x[..., half:])
    cs, sn = (t[:, None, None].double() for t in (cos, sin))
    u, w = u.double(), w.double()
    first = lambda a, b: (a * b).float().double()  # noqa: E731
    if inter:
        a, b = u * cs - first(w, sn), u * sn + first(w, cs)
    else:
        a, b = u * cs + first(w, -sn), w * cs + first(u, sn)
    a, b = a.float().to(dtype), b.float().to(dtype)
    x.copy_(torch.stack([a, b], -1).flatten(-2) if inter else torch.cat([a, b], -1))
    assert ops.rope_append(*qkv.unbind(1), rot, inter, cos, sin, pos, page, off, c.k[0], c.v[0])
    assert torch.equal(qkv, want)
    assert torch.equal(c.k[0][0, :, :T], want[:, 1].transpose(0, 1)) and torch.equal(c.v[0][0, :, :T], want[:, 2].transpose(0, 1))


TINY = {
    "gptj": dict(model_type="gptj", vocab_size=512, n_embd=128, n_layer=2, n_head=2, n_positions=512, rotary_dim=32),
    "gpt2": dict(model_type="gpt2", vocab_size=512, n_embd=128, n_layer=2, n_head=2, n_positions=512),
    "bloom": dict(model_type="bloom", vocab_size=512, hidden_size=128, n_layer=2, n_head=2),
    "gpt_neox": dict(model_type="gpt_neox", vocab_size=512, hidden_size=160, num_hidden_layers=2, num_attention_heads=2,
                     intermediate_size=640, rotary_pct=0.25, max_position_embeddings=512, use_parallel_residual=True),
}


@pytest.mark.parametrize("name", TINY)
@pytest.mark.parametrize("on_gpu", [False, True])
def test_runner_packs_prompts(name, on_gpu):
    m = build_model(LMConfig.from_hf(TINY[name]), device="cuda", dtype=torch.bfloat16, seed=1)
    lens, slots = [70, 1, 200, 33], [3, 0, 2, 5]
    ids = torch.randint(0, 512, (4, 200), generator=torch.Generator().manual_seed(0))
    r, one = ModelRunner(m, max_slots=6, max_len=300), ModelRunner(m, max_slots=6, max_len=300)
    r.seen.fill_(1)
    got = r.prefill(ids.cuda() if on_gpu else ids, slots, lens)
    for i, (s, n) in enumerate(zip(slots, lens)):
        want = one.prefill(ids[i:i + 1, :n], [s])
        assert (got[i].float() - want[0].float()).norm() <= 2e-2 * want.float().norm()
        row = torch.zeros(512, dtype=torch.uint8, device="cuda")
        row[ids[i, :n].cuda()] = 1
        assert torch.equal(r.seen[s], row)
    rows = [{"token": 7, "pos": n, "slot": s, "temperature": 0.0, "top_k": 1, "top_p": 1.0, "rep": 1.0, "seed": 0}
            for s, n in zip(slots, lens)]
    a, b = r.decode(rows), one.decode(rows)
    assert max(abs(x - y) for x, y in zip(a[1], b[1])) < 0.05


def test_prompts_that_share_a_slot():
    """The later row's keys and values stay (without pages they are written one prompt after another)."""
    m = build_model(LMConfig.from_hf(TINY["gptj"]), device="cuda", dtype=torch.bfloat16, seed=1)
    ids = torch.randint(0, 512, (8, 64), generator=torch.Generator().manual_seed(0))
    r, one = (ModelRunner(m, max_slots=2, max_len=96, page_size=0) for _ in range(2))
    r.prefill(ids, [1] * 8)
    one.prefill(ids[7:], [1])
    for a, b in zip(r.cache.k + r.cache.v, one.cache.k + one.cache.v):
        assert (a[1, :, :64].float() - b[1, :, :64].float()).norm() <= 2e-2 * b[1, :, :64].float().norm()
