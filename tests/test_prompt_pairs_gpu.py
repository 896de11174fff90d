"""Two products of few rows in one launch (beside each other, or along K), a GELU on the fp32 sums, and LayerNorm of chosen rows,
against float64; and that a runner's short prompts take them for every layer kind."""
import pytest
import torch
import torch.nn.functional as F

from kubernetes_cloud_amd.engine import runner as R
from kubernetes_cloud_amd.models.causal_lm import build_model
from kubernetes_cloud_amd.models.config import LMConfig, PRESETS_HF
from kubernetes_cloud_amd.ops import linear as L
from kubernetes_cloud_amd.ops.norms import layer_norm, layer_norm_rows

pytestmark = pytest.mark.gpu


def _part(rows, n, k, dtype, bias, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.empty(rows, k, device="cuda", dtype=dtype).normal_(generator=g)
    w = torch.empty(n, k, device="cuda", dtype=dtype).normal_(std=k ** -0.5, generator=g)
    return x, w, torch.empty(n, device="cuda", dtype=dtype).normal_(generator=g) if bias else None


def _ref(x, w, b, act=None):
    y = x.double() @ w.double().t() + (0 if b is None else b.double())
    return y if act is None else F.gelu(y, approximate=act)


def _close(y, ref, terms=1):
    # one rounding to the type; 32-bit sums of terms of size k^-1/2 and a GELU of slope at most 1.13: well below 1e-4 a product
    eps = 2.0 ** -8 if y.dtype is torch.bfloat16 else 2.0 ** -11
    return ((y.double() - ref).abs() <= eps * ref.abs() + terms * 1e-4).all().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k,n2,k2,act", [(16, 64, 80, 64, "tanh"), (96, 512, 64, 1024, "none"), (1040, 2048, 1360, 1088, None),
                                           (3072, 1024, 4096, 1024, "tanh")])
def test_beside(dtype, rows, n, k, n2, k2, act):
    a, b = _part(rows, n, k, dtype, True, 1), _part(rows, n2, k2, dtype, n2 % 32 == 0, 2)
    with torch.no_grad():
        for _ in range(2):  # (the counters are left zeroed)
            y, y2 = L.few_rows_beside(a, b, act)
            assert _close(y, _ref(*a)) and _close(y2, _ref(*b, act))
            z = L.few_rows_gelu(*b, act or "tanh")
            assert _close(z, _ref(*b, act or "tanh"))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k,k2", [(16, 64, 64), (80, 64, 1984), (96, 4096, 1024), (2048, 64, 2112), (4096, 4096, 1024)])
def test_sum(dtype, rows, n, k, k2):
    a, b = _part(rows, n, k, dtype, True, 1), _part(rows, n, k2, dtype, n % 32 == 0, 2)
    with torch.no_grad():
        for _ in range(2):
            assert _close(L.few_rows_sum(a, b), _ref(*a) + _ref(*b), 2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 17, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k,k2", [(16, 64, 64), (80, 64, 1984), (2048, 64, 2112), (4096, 4096, 1024), (16400, 128, 64)])
@pytest.mark.parametrize("captured", [False, True])
def test_sum_and_residual_rows(dtype, rows, n, k, k2, captured):
    """The residual rows enter the 32-bit sums: one rounding, where the rounded sum of the products was added to them and rounded again."""
    if not L.few_rows(rows, n, k) or not L.few_rows(rows, n, k2):
        pytest.skip("the library's")
    a, b = _part(rows, n, k, dtype, True, 1), _part(rows, n, k2, dtype, n % 32 == 0, 2)
    res = torch.empty(1, rows, n, device="cuda", dtype=dtype).normal_(std=30, generator=torch.Generator(device="cuda").manual_seed(3))
    sc = L.few_rows_scratch(rows, torch.device("cuda", 0)) if captured else None  # (with a scratch: the launch from Python)
    with torch.no_grad():
        for _ in range(2):
            y = L.few_rows_sum(a, b, sc, res)
            assert _close(y, _ref(*a) + _ref(*b) + res[0].double(), 3)


def test_residual_rows_they_leave():
    a, b = _part(8, 96, 128, torch.bfloat16, True, 1), _part(8, 96, 192, torch.bfloat16, True, 2)
    r = torch.ones(8, 96, device="cuda", dtype=torch.bfloat16)
    for sc in (None, L.few_rows_scratch(8, torch.device("cuda", 0))):
        with torch.no_grad():
            for bad in (r.float(), r.half(), r[:7], torch.ones(8, 192, device="cuda", dtype=torch.bfloat16)[:, ::2], r.cpu(),
                        torch.ones(769, device="cuda", dtype=torch.bfloat16)[1:].view(8, 96)):
                assert L.few_rows_sum(a, b, sc, bad) is None
            assert L.few_rows_sum(a, b, sc, r) is not None


def test_what_they_leave():
    a, b = _part(8, 96, 128, torch.bfloat16, True, 1), _part(8, 96, 128, torch.bfloat16, True, 2)
    assert L.few_rows_beside(a, b) is not None if not torch.is_grad_enabled() else L.few_rows_beside(a, b) is None
    with torch.no_grad():
        assert L.few_rows_sum(a, (b[0], b[1][:80], None)) is None                       # other widths
        assert L.few_rows_beside((a[0], a[1][:90], None), b) is None                    # no multiple of 16
        assert L.few_rows_beside((a[0][:, :120], a[1][:, :120], None), b) is None       # strided
        assert L.few_rows_beside(_part(129, 96, 128, torch.bfloat16, True, 1), _part(129, 96, 128, torch.bfloat16, True, 1)) is None
        assert L.few_rows_beside(tuple(t.float() for t in a), b) is None
        assert L.few_rows_gelu(*a, "sigmoid") is None


@pytest.mark.parametrize("d", [8, 2040, 2048, 4096, 5120, 16384])
@pytest.mark.parametrize("residuals", [0, 1, 2])
def test_layer_norm_rows(d, residuals):
    g = torch.Generator(device="cuda").manual_seed(d)
    x, *r = (torch.randn(50, d, device="cuda", generator=g).bfloat16() for _ in range(1 + residuals))
    w, b = (torch.randn(d, device="cuda", generator=g).bfloat16() for _ in range(2))
    rows = torch.tensor([49, 0, 7, 7], device="cuda")
    with torch.no_grad():
        y = layer_norm_rows(x, w, b, 1e-5, tuple(r), rows)
        full = layer_norm(x, w, b, 1e-5, tuple(r))
    h = sum((t.double() for t in (x, *r)))
    ref = F.layer_norm(h, (d,), w.double(), b.double(), 1e-5)
    # the sum is not rounded on its way to a few rows
    assert ((y.double() - ref[rows]).abs() <= 2.0 ** -8 * ref[rows].abs() + 1e-4).all()
    full = full[0] if residuals else full
    assert ((full.double() - ref).abs() <= (2.0 ** -8 * ref.abs() + (2.0 ** -7 if residuals else 0) * (1 + w.double().abs()) * 4 + 1e-4)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name,kw", [("gpt-j-6b", dict(n_embd=512, n_head=2, rotary_dim=64, n_layer=2, vocab_size=1024)),
                                     ("gpt-neox-20b", dict(hidden_size=512, num_attention_heads=8, num_hidden_layers=2,
                                                           intermediate_size=2048, vocab_size=1024)),
                                     ("gpt2", dict(n_embd=512, n_head=8, n_layer=2, vocab_size=1024))])
def test_short_prompts_of_every_layer_kind(monkeypatch, dtype, name, kw):
    if name not in PRESETS_HF:
        pytest.skip("no such preset")
    m = build_model(LMConfig.from_hf(dict(PRESETS_HF[name], **kw)), device="cuda", dtype=dtype, seed=3).requires_grad_(False)
    ids, lens = torch.randint(0, 1024, (2, 40), generator=torch.Generator().manual_seed(0)), [40, 23]
    out, calls = [], []
    for off in (False, True):
        r = R.ModelRunner(m, max_slots=2, max_len=64)
        with monkeypatch.context() as mp:
            for f in ("few_rows_beside", "few_rows_sum", "few_rows_gelu"):
                if off:
                    mp.setattr(R, f, lambda *a, **k: None)
                else:
                    g = getattr(R, f)
                    mp.setattr(R, f, lambda *a, g=g, f=f, **k: calls.append(f) or g(*a, **k))
            out.append(r.prefill(ids, [0, 1], lens).double())
    assert set(calls) == ({"few_rows_beside", "few_rows_sum"} if m.cfg.parallel_residual else {"few_rows_gelu"})
    # two layers whose sums are rounded at other places: as tests/test_prompt_rows_gpu.py bounds packed prompts
    assert (out[0] - out[1]).norm() <= (2e-2 if dtype is torch.bfloat16 else 3e-3) * out[1].norm()


@pytest.mark.parametrize("how", ["global hook", "global pre-hook", "own forward", "own hook"])
@pytest.mark.parametrize("parallel", [True, False])
def test_hooks_see_short_prompts(how, parallel):
    """Whatever a caller has put around a layer's call runs for a short prompt as for a long one."""
    cfg = dict(PRESETS_HF["gpt-j-6b"], n_embd=512, n_head=2, rotary_dim=64) if parallel else dict(PRESETS_HF["gpt2"], n_embd=512, n_head=8)
    m = build_model(LMConfig.from_hf(dict(cfg, n_layer=2, vocab_size=1024)), device="cuda", dtype=torch.bfloat16, seed=3).requires_grad_(False)
    r, seen = R.ModelRunner(m, max_slots=1, max_len=256), []
    names = {x: n for n, x in m.named_modules()}
    inner = [x for x, n in names.items() if n.endswith(("qkv", "out", "mlp", "fc_in", "fc_out", "ln_f"))]
    if how.startswith("global"):
        reg = torch.nn.modules.module.register_module_forward_pre_hook if "pre" in how else torch.nn.modules.module.register_module_forward_hook
        handles = [reg(lambda x, *a: seen.append(names[x]) if x in inner else None)]
    elif how == "own hook":
        handles = [x.register_forward_hook(lambda x, *a: seen.append(names[x])) for x in inner]
    else:
        handles = []
        for x in inner:
            x.forward = lambda *a, x=x, f=x.forward, **k: seen.append(names[x]) or f(*a, **k)
    try:
        calls = []
        for n in (30, 200):
            seen.clear()
            r.prefill(torch.arange(n)[None], [0], [n])
            calls.append(sorted(seen))
    finally:
        for h in handles:
            h.remove()
    assert calls[0] == calls[1] == sorted(names[x] for x in inner)


def test_block_tables_go_up_in_order():
    """Edits while earlier uploads still wait for the GPU: each launch reads the table of its own time."""
    c = R.KVCache(1, 8, 1, 512, 64, "cuda", page_size=16)
    want, got = [], []
    torch.cuda._sleep(50_000_000)
    for i in range(40):
        c.release(i % 8)
        c.reserve((3 * i) % 8, 16 * (i % 32) + 1)
        c.sync()
        want.append(c.table_h.clone())
        got.append(c.table.clone())
    assert all(torch.equal(a, b.cpu()) for a, b in zip(want, got))
