"""What the speed of this framework is judged on: attention as the training and prompt paths call it, GPT-J-shaped
prompts and decode steps on the serving runner, and routed feed-forward sublayers.

Kinds of cases

* ``attention``  ``ops.flash_attention`` over [batch, tokens, heads, size], causal; forward alone (prompts) or forward
  and backward (finetuning: outputs and the three gradients). ``mask``: "none"; "length", right-padded batches;
  "alibi", BLOOM's bias by distance; "window", GPT-Neo's local layers.
* ``prompt``     ``LLMEngine``'s prompt call, ``ModelRunner.prefill``, of a few GPT-J layers: last-token logits and the
  key / value pages that decoding reads.
* ``decode``     one decode step of the same model, ``ModelRunner.decode_async``, every sequence ``cached`` tokens or
  more behind: sampled ids, their log-probabilities, and the pages.
* ``experts``    the routed feed-forward sublayer of the per-layer mixed decoders: router, grouping, expert products,
  residual and next norm. "sigmoid" is Megusun's, "softmax" Gibipel's (corrected choice in groups, identity experts).

Sizes are those of this repository's configurations and benchmarks: GPT-2 / GPT-Neo (heads of 64 and 128), GPT-NeoX (96),
BLOOM (128), GPT-J (256); ``bench/megusun_bench.py`` and ``bench/gibipel_bench.py`` for the experts.
"""
from __future__ import annotations

import math

import torch

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
VOCAB, ROT, BASE, EPS = 50400, 64, 10000.0, 1e-5
MEGUSUN, GIBIPEL = "sigmoid", "softmax"


def listed() -> list[dict]:
    return [
        # a GPT-J micro-batch of the finetuner at its full context, one layer's attention
        attention("train-gptj-2048", 2, 2048, 16, 256, "none", True),
        # GPT-2 finetuning on right-padded texts: no length is a multiple of a tile
        attention("train-gpt2-padded-1000", 8, 1000, 12, 64, "length", True),
        # a BLOOM tensor-parallel rank (112 heads over 8) finetuning a full context
        attention("train-bloom-alibi-2048", 1, 2048, 14, 128, "alibi", True),
        # the smallest finetuning call: one short text
        attention("train-gpt2-short-96", 1, 96, 12, 64, "none", True),
        # a GPT-NeoX prompt of any length
        attention("prompt-neox-1500", 1, 1500, 64, 96, "none", False),
        # a chat turn: one short prompt
        prompt("prompt-gptj-1x61", 4096, 4, 1, 61, 61, "bf16"),
        # a batch of prompts that the scheduler admitted together
        prompt("prompt-gptj-6x1100", 4096, 4, 6, 700, 1100, "bf16"),
        # interactive decoding, in the precision that FasterTransformer serves
        decode("decode-gptj-1", 4096, 4, 1, 512, "fp16"),
        # a loaded server
        decode("decode-gptj-32", 4096, 4, 32, 700, "bf16"),
        # prompts through routed experts
        experts("experts-prompt-4096", MEGUSUN, 4096, 4096, 16, 2, 4096),
        experts("experts-prompt-777", GIBIPEL, 777, 2048, 24, 5, 768),
        # a decode step of 32 sequences through routed experts
        experts("experts-decode-32", GIBIPEL, 32, 4096, 16, 3, 2048),
    ]


def draw(rng) -> dict:
    def spread(lo, hi):  # over the logarithm, odd sizes among them
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["attention", "attention", "attention", "prompt", "decode", "experts", "experts"])
    if kind == "attention":
        train = rng.random() < 0.6
        heads, dim = rng.choice([(12, 64), (16, 64), (20, 128), (14, 128), (32, 96), (16, 256)])
        mask = rng.choice(["none", "none", "length", "alibi", "window"])
        tokens = spread(64, 4096)
        if rng.random() < 0.3:
            tokens = max(128, tokens // 128 * 128)
        batch = max(1, min(spread(1, 16), 6144 // tokens))
        return attention("", batch, tokens, heads, dim, mask, train)
    if kind == "prompt":
        width = rng.choice([2048, 4096])
        n = rng.choice([1, 1, 2, 3, 4, 8])
        hi = min(2000, spread(24, 2000), 6600 // n)
        return prompt("", width, 4, n, max(8, int(hi * rng.uniform(0.4, 1.0))), hi, rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "decode":
        return decode("", rng.choice([2048, 4096]), 4, rng.choice([1, 2, 3, 5, 8, 13, 16, 24, 32]), spread(32, 900),
                      rng.choice(["bf16", "fp16"]))
    rule, width, n_exp, top, ff = rng.choice([(MEGUSUN, 4096, 16, 2, 4096), (MEGUSUN, 2048, 32, 4, 1024),
                                              (GIBIPEL, 4096, 16, 3, 2048), (GIBIPEL, 2048, 24, 5, 768)])
    return experts("", rule, spread(1, 4096), width, n_exp, top, ff)


def _named(name, c):
    return {"name": name, **c} if name else c


def attention(name, batch, tokens, heads, dim, mask, train):
    return _named(name, {"kind": "attention", "batch": batch, "tokens": tokens, "heads": heads, "dim": dim, "mask": mask,
                         "train": train})


def prompt(name, width, layers, prompts, shortest, longest, dtype):
    return _named(name, {"kind": "prompt", "width": width, "layers": layers, "prompts": prompts, "shortest": shortest,
                         "longest": longest, "dtype": dtype})


def decode(name, width, layers, batch, cached, dtype):
    return _named(name, {"kind": "decode", "width": width, "layers": layers, "batch": batch, "cached": cached, "dtype": dtype})


def experts(name, rule, tokens, width, n_experts, top, ff):
    return _named(name, {"kind": "experts", "rule": rule, "tokens": tokens, "width": width, "experts": n_experts, "top": top,
                         "ff": ff})


def _rng(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.empty(shape, device=DEV, dtype=dtype).normal_(0.0, std, generator=g)


def _lengths(n, lo, hi):
    """Between the two, spread evenly: the longest first."""
    return [hi - (hi - lo) * i // max(1, n - 1) for i in range(n)]


# ------------------------------------------------------------------------------------------------- attention
def _attention_inputs(c, seed):
    """q, k, v as a fused projection leaves them (one buffer), the output's gradient, key lengths, slopes."""
    B, S, H, D = c["batch"], c["tokens"], c["heads"], c["dim"]
    g = _rng(seed)
    qkv = _normal(g, B, S, 3, H, D)
    do = _normal(g, B, S, H, D)
    lens = slopes = None
    if c["mask"] == "length":
        lens = torch.tensor(_lengths(B, max(1, S // 3), S), device=DEV, dtype=torch.int32)
        do[torch.arange(S, device=DEV)[None] >= lens[:, None]] = 0  # padding has no loss
    if c["mask"] == "alibi":
        slopes = 2.0 ** (-8.0 * torch.arange(1, H + 1, device=DEV, dtype=torch.float32) / H)
    return qkv, do, lens, slopes


def _window(c):
    return 256 if c["mask"] == "window" else 0  # GPT-Neo's local layers


def _attention_prepare(c, seed):
    qkv, do, lens, slopes = _attention_inputs(c, seed)
    q, k, v = (qkv[:, :, i].requires_grad_(c["train"]) for i in range(3))
    return {"c": c, "q": q, "k": k, "v": v, "do": do, "lens": lens, "slopes": slopes}


def _attention_run(s):
    from kubernetes_cloud_amd import ops
    c = s["c"]
    if not c["train"]:
        with torch.no_grad():
            return [ops.flash_attention(s["q"], s["k"], s["v"], causal=True, kv_len=s["lens"], alibi=s["slopes"],
                                        window=_window(c))]
    o = ops.flash_attention(s["q"], s["k"], s["v"], causal=True, kv_len=s["lens"], alibi=s["slopes"], window=_window(c))
    return [o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])]


def _visible(S, window, length):
    i = torch.arange(S, device=DEV)
    m = i[None] <= i[:, None]
    if window:
        m &= i[None] > i[:, None] - window
    if length is not None:
        m &= (i < length)[None]
    return m


def _attend(q, k, v, scale, mask, slopes=None):
    """One sequence, [S, H, D]; queries that see nothing give zeros."""
    s = torch.einsum("qhd,khd->hqk", q, k) * scale
    if slopes is not None:
        i = torch.arange(q.shape[0], device=DEV, dtype=q.dtype)
        s = s + slopes.to(q.dtype)[:, None, None] * (i[None] - i[:, None])
    p = torch.softmax(s.masked_fill(~mask, -1e300), -1) * mask
    return torch.einsum("hqk,khd->qhd", p, v)


def _attention_exact(c, seed):
    qkv, do, lens, slopes = _attention_inputs(c, seed)
    B, S, H, D = do.shape
    outs = [torch.empty(B, S, H, D, device=DEV, dtype=torch.float64) for _ in range(4 if c["train"] else 1)]
    for b in range(B):
        mask = _visible(S, _window(c), None if lens is None else int(lens[b]))
        for h in range(0, H, 8):
            hs = slice(h, min(H, h + 8))
            x = [qkv[b, :, i, hs].double().requires_grad_(c["train"]) for i in range(3)]
            o = _attend(*x, D ** -0.5, mask, None if slopes is None else slopes[hs])
            res = [o, *torch.autograd.grad(o, x, do[b, :, hs].double())] if c["train"] else [o]
            for t, r in zip(outs, res):
                t[b, :, hs] = r.detach()
            del x, o, res
    return outs


def _pairs(c):
    """Query-key pairs that are computed, over the batch."""
    S, w = c["tokens"], _window(c) or c["tokens"]
    lens = _lengths(c["batch"], max(1, S // 3), S) if c["mask"] == "length" else [S] * c["batch"]
    return sum(sum(max(0, min(i + 1, n) - max(0, i + 1 - w)) for i in range(S)) for n in lens)


def _attention_work(c):
    n = c["batch"] * c["tokens"] * c["heads"] * c["dim"] * 2
    f = _pairs(c) * c["heads"] * c["dim"] * 2
    return {"bytes": n * (8 if c["train"] else 4), "flops": f * (7 if c["train"] else 2)}


# ---------------------------------------------------------------------------------------------------- GPT-J
def _gptj_weights(c, seed):
    """Weights under the module's names. The head's bias spreads as token frequencies do, with a newline that is likely
    everywhere: a decode step's likeliest token is hardly ever a tie."""
    g, d, dt = _rng(seed), c["width"], DTYPES[c["dtype"]]
    w = {"wte.weight": _normal(g, VOCAB, d, std=0.3, dtype=dt)}
    for i in range(c["layers"]):
        p = "h.%d." % i
        w[p + "ln_1.weight"] = 1 + _normal(g, d, std=0.1, dtype=dt)
        w[p + "ln_1.bias"] = _normal(g, d, std=0.02, dtype=dt)
        w[p + "attn.qkv.weight"] = _normal(g, 3 * d, d, std=0.02, dtype=dt)
        w[p + "attn.out.weight"] = _normal(g, d, d, std=0.02, dtype=dt)
        w[p + "mlp.fc_in.weight"], w[p + "mlp.fc_in.bias"] = _normal(g, 4 * d, d, std=0.02, dtype=dt), _normal(g, 4 * d, std=0.02, dtype=dt)
        w[p + "mlp.fc_out.weight"], w[p + "mlp.fc_out.bias"] = _normal(g, d, 4 * d, std=0.01, dtype=dt), _normal(g, d, std=0.02, dtype=dt)
    w["ln_f.weight"], w["ln_f.bias"] = 1 + _normal(g, d, std=0.1, dtype=dt), _normal(g, d, std=0.02, dtype=dt)
    w["lm_head.weight"], w["lm_head.bias"] = _normal(g, VOCAB, d, std=0.01, dtype=dt), _normal(g, VOCAB, dtype=dt)
    w["lm_head.bias"][198] = 7.0
    return w


def _gptj_prompts(c, seed):
    """Right-padded ids (on the host, as a tokenizer gives them) and their lengths."""
    g = torch.Generator().manual_seed(int(seed) + 1)
    if c["kind"] == "prompt":
        lens = _lengths(c["prompts"], c["shortest"], c["longest"])
    else:
        lens = [c["cached"] + 7 * i for i in range(c["batch"])]
    return torch.randint(0, VOCAB, (len(lens), max(lens)), generator=g), lens


def _gptj_runner(c, seed, slots, max_len):
    from kubernetes_cloud_amd.engine.runner import ModelRunner
    from kubernetes_cloud_amd.models.causal_lm import CausalLM
    from kubernetes_cloud_amd.models.config import LMConfig, PRESETS_HF
    cfg = LMConfig.from_hf(dict(PRESETS_HF["gpt-j-6b"], n_embd=c["width"], n_layer=c["layers"], n_head=c["width"] // 256,
                                vocab_size=VOCAB, rotary_dim=ROT))
    with torch.device("meta"):
        m = CausalLM(cfg)
    m.load_state_dict(_gptj_weights(c, seed), strict=True, assign=True)
    return ModelRunner(m.requires_grad_(False), max_slots=slots, max_len=max_len)


def _pools(r):
    return {"k": list(r.cache.k), "v": list(r.cache.v)}


def _prompt_prepare(c, seed):
    ids, lens = _gptj_prompts(c, seed)
    return {"c": c, "runner": _gptj_runner(c, seed, len(lens), max(lens) + 64), "ids": ids, "lens": lens}


def _prompt_run(s):
    r = s["runner"]
    for i in range(len(s["lens"])):  # the last requests have ended
        r.release(i)
    return {"logits": r.prefill(s["ids"], list(range(len(s["lens"]))), s["lens"]), **_pools(r)}


def _decode_prepare(c, seed):
    ids, lens = _gptj_prompts(c, seed)
    r = _gptj_runner(c, seed, len(lens), max(lens) + 64)
    slots = list(range(len(lens)))
    for i in range(0, len(lens), 8):
        r.prefill(ids[i:i + 8], slots[i:i + 8], lens[i:i + 8])
    rows = [{"token": int(ids[i, 0]), "pos": n, "slot": i, "temperature": 0.0, "top_k": 1, "top_p": 1.0, "rep": 1.0,
             "seed": i} for i, n in enumerate(lens)]
    r.decode(rows)  # a server has its step graphs
    return {"c": c, "runner": r, "rows": rows}


def _decode_run(s):
    r, n = s["runner"], len(s["rows"])
    h = r.decode_async(s["rows"])
    return {"ids": h.ids_dev[:n], "logprobs": h.lps_h[:n], **_pools(r)}


def _rotate(x, pos):
    """[T, H, D]: GPT-J's interleaved pairs of the first dims turn."""
    f = BASE ** (-torch.arange(0, ROT, 2, device=DEV, dtype=torch.float64) / ROT)
    a = pos.double()[:, None, None] * f
    y = x.clone()
    u, v = x[..., 0:ROT:2], x[..., 1:ROT:2]
    y[..., 0:ROT:2], y[..., 1:ROT:2] = u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()
    return y


def _gptj_last(w, c, ids):
    """Logits of a sequence's last token."""
    T, d = ids.shape[0], c["width"]
    H, pos = d // 256, torch.arange(ids.shape[0], device=DEV)
    ln = lambda x, p: torch.nn.functional.layer_norm(x, (d,), w[p + ".weight"].double(), w[p + ".bias"].double(), EPS)  # noqa: E731
    mm = lambda x, n: x @ w[n + ".weight"].double().T  # noqa: E731
    h, mask = w["wte.weight"][ids].double(), _visible(T, 0, None)
    for i in range(c["layers"]):
        p = "h.%d." % i
        x = ln(h, p + "ln_1")
        q, k, v = mm(x, p + "attn.qkv").view(T, 3, H, 256).unbind(1)
        a = _attend(_rotate(q, pos), _rotate(k, pos), v, 256 ** -0.5, mask)
        u = mm(x, p + "mlp.fc_in") + w[p + "mlp.fc_in.bias"].double()
        u = torch.nn.functional.gelu(u, approximate="tanh")
        h = h + mm(a.reshape(T, d), p + "attn.out") + mm(u, p + "mlp.fc_out") + w[p + "mlp.fc_out.bias"].double()
    return mm(ln(h[-1:], "ln_f"), "lm_head")[0] + w["lm_head.bias"].double()


def _gptj_exact(c, seed):
    w = _gptj_weights(c, seed)
    ids, lens = _gptj_prompts(c, seed)
    ids = ids.to(DEV)
    none = {"k": [None] * c["layers"], "v": [None] * c["layers"]}  # where a page lies is the allocator's choice
    if c["kind"] == "prompt":
        return {"logits": torch.stack([_gptj_last(w, c, row[:n]) for row, n in zip(ids, lens)]), **none}
    z = torch.stack([_gptj_last(w, c, torch.cat([row[:n], row[:1]])) for row, n in zip(ids, lens)])
    lp = torch.log_softmax(z, -1).max(-1)
    return {"ids": lp.indices, "logprobs": lp.values, **none}


def _gptj_work(c):
    d, L = c["width"], c["layers"]
    layer = 12 * d * d
    if c["kind"] == "prompt":
        lens = _lengths(c["prompts"], c["shortest"], c["longest"])
        T, n = sum(lens), len(lens)
        pairs, kv = sum(x * (x + 1) // 2 for x in lens), T * 2 * d * 2 * L
    else:
        lens = [c["cached"] + 7 * i + 1 for i in range(c["batch"])]
        T = n = len(lens)
        pairs, kv = sum(lens), sum(lens) * 2 * d * 2 * L
    return {"bytes": (layer * L + VOCAB * d + T * d) * 2 + kv + n * VOCAB * 2 * (c["kind"] == "prompt"),
            "flops": 2 * (T * layer * L + n * VOCAB * d) + 4 * pairs * d * L}


# -------------------------------------------------------------------------------------------------- experts
def _identity(c):
    return 0 if c["rule"] == MEGUSUN else c["experts"] // 4 if c["width"] == 4096 else c["experts"] // 3


def _choice_groups(c):
    return (4, 2) if c["width"] == 4096 else (8, 4)


def _experts_inputs(c, seed):
    g, T, d, E, F = _rng(seed), c["tokens"], c["width"], c["experts"], c["ff"]
    outs = E + _identity(c)
    x = _normal(g, T, d, dtype=torch.float32)
    w = {"h": x.to(torch.bfloat16), "x": x, "router": _normal(g, outs, d, std=d ** -0.5),
         "gate_up": _normal(g, E, 2 * F, d, std=d ** -0.5), "down": _normal(g, E, d, F, std=F ** -0.5),
         "gain": torch.ones((), device=DEV, dtype=torch.bfloat16)}
    if c["rule"] == MEGUSUN:
        w["a"] = _normal(g, T, d)  # what the mixer and the shared expert add
    else:
        w["fix"] = _normal(g, outs, std=0.02, dtype=torch.float32)
    return w


def _experts_prepare(c, seed):
    from kubernetes_cloud_amd.ops import moe
    s = {"c": c, **_experts_inputs(c, seed)}
    if c["rule"] == GIBIPEL:
        s["rule"] = moe.Router(True, s["fix"], *_choice_groups(c), _identity(c))
    return s


def _experts_run(s):
    from kubernetes_cloud_amd.ops import moe
    from kubernetes_cloud_amd.ops.norm_residual import NormedSum, postnorm
    from kubernetes_cloud_amd.ops.rms_shift import Branch, rms_shift
    c, h = s["c"], s["h"]
    outs = c["experts"] + _identity(c)
    mt = moe.tile_rows(c["tokens"], c["top"], outs, c["width"], c["ff"], h.dtype)
    rule = s.get("rule", moe.SIGMOID)
    ids, wts, _, g = moe.route_group(h, s["router"], c["top"], None, mt, rule)
    y = moe.experts(h, ids, wts, s["gate_up"], s["down"], g, c["rule"] == MEGUSUN)
    if c["rule"] == MEGUSUN:
        x, n, _ = rms_shift(s["x"], Branch(s["a"], y, g.inv), 0.5, s["gain"], EPS)
    else:
        # (the weights multiply the products' outputs; identity experts add the stream)
        x, n = postnorm(s["x"], NormedSum(s["gain"], None, y, g.inv, wts), EPS, h.dtype)
    return {"ids": ids, "weights": wts, "x": x, "h": n}


def _experts_exact(c, seed):
    s = _experts_inputs(c, seed)
    h, E, top = s["h"].double(), c["experts"], c["top"]
    z = h @ s["router"].double().T
    if c["rule"] == MEGUSUN:
        wts, ids = torch.sigmoid(z).topk(top, -1)
    else:
        sc = torch.softmax(z, -1)
        fixed = sc + s["fix"].double()
        n, keep = _choice_groups(c)
        best = fixed.view(h.shape[0], n, -1).amax(-1).topk(keep, -1).indices
        kept = torch.zeros(h.shape[0], n, device=DEV, dtype=torch.bool).scatter_(1, best, True)
        kept = kept.repeat_interleave(fixed.shape[1] // n, 1)
        ids = fixed.masked_fill(~kept, -1e300).topk(top, -1).indices
        wts = sc.gather(1, ids)
        wts = wts / wts.sum(-1, keepdim=True)
    y = torch.zeros_like(h)
    for e in range(E):
        at, k = torch.where(ids == e)
        if at.numel():
            a = wts[at, k, None]
            r = h[at] * a if c["rule"] == MEGUSUN else h[at]
            u = r @ s["gate_up"][e].double().T
            o = (torch.nn.functional.silu(u[:, :c["ff"]]) * u[:, c["ff"]:]) @ s["down"][e].double().T
            y.index_add_(0, at, o if c["rule"] == MEGUSUN else o * a)
    rms = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + EPS)  # noqa: E731
    x = s["x"].double()
    if c["rule"] == MEGUSUN:
        x = x + 0.5 * (s["a"].double() + y)
        return {"ids": ids.int(), "weights": wts, "x": x, "h": rms(x)}
    x = x + rms(y + (wts * (ids >= E)).sum(-1, keepdim=True) * x)
    return {"ids": ids.int(), "weights": wts, "x": x, "h": x}


def _experts_work(c):
    T, d, F, E, top = c["tokens"], c["width"], c["ff"], c["experts"], c["top"]
    outs = E + _identity(c)
    rows = T * top * E / outs  # identity experts have no products
    used = E * (1 - (1 - top / outs) ** T)
    return {"bytes": used * 3 * d * F * 2 + outs * d * 2 + T * d * (2 + 4 + 4 + 2 + (2 if c["rule"] == MEGUSUN else 0)),
            "flops": 2 * rows * 3 * d * F + 2 * T * outs * d}


# ------------------------------------------------------------------------------------------------- the cases
def prepare(case, seed):
    return {"attention": _attention_prepare, "prompt": _prompt_prepare, "decode": _decode_prepare,
            "experts": _experts_prepare}[case["kind"]](case, seed)


def run(state):
    return {"attention": _attention_run, "prompt": _prompt_run, "decode": _decode_run,
            "experts": _experts_run}[state["c"]["kind"]](state)


def exact(case, seed):
    with torch.set_grad_enabled(case["kind"] == "attention"):
        return {"attention": _attention_exact, "prompt": _gptj_exact, "decode": _gptj_exact,
                "experts": _experts_exact}[case["kind"]](case, seed)


def work(case):
    return {"attention": _attention_work, "prompt": _gptj_work, "decode": _gptj_work,
            "experts": _experts_work}[case["kind"]](case)


def tolerance(case):
    """About four times what the path is off from 64 bits (bf16 operands and results, fp32 sums)."""
    return {"attention": {"rel": 1e-2}, "prompt": {"rel": 1.2e-2}, "decode": {"rel": 1e-2, "differ": 0.01},
            "experts": {"rel": 8e-3, "differ": 0.005}}[case["kind"]]
