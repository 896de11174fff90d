"""Mixture of gated experts (``csrc/kernels/moe.hip``): top-k router (sigmoid scores, or softmax scores with a correction
of the choice, expert groups and identity experts), grouping by expert, expert products with the router weight on the
expert's input (or output), and the strided feed-forward activations (``csrc/kernels/act_rows.hip``).

Expert weights are stacked: gate-and-up [E, 2F, d] (gate rows first), down [E, d, F].
"""
from __future__ import annotations

import dataclasses
import math

import torch

from . import _lib
from .rms_shift import native_dt

GEMM_ROWS = 256
STREAM_ROWS = 32
SHARED_ROWS = 16  # tokens up to which a shared expert's weights stream beside the routed ones'


@dataclasses.dataclass(frozen=True)
class Router:
    """How scores become choices. sigmoid: the ``top`` largest scores, which are the weights. softmax: the largest
    scores + ``correction`` (fp32 [outputs]) within the ``keep`` of ``groups`` equal groups of neighbours whose best one is
    largest; the weights are the scores over their sum. The last ``identity`` router outputs have no expert: they
    pass the token on."""
    softmax: bool = False
    correction: torch.Tensor | None = None
    groups: int = 1
    keep: int = 1
    identity: int = 0


SIGMOID = Router()


def route(h: torch.Tensor, router: torch.Tensor, top: int, shared_gate: torch.Tensor | None = None,
          rule: Router = SIGMOID):
    """h [T, d] -> (ids int32 [T, top], weights fp32 [T, top], sigmoid of the shared expert's gate [T] | None)."""
    code = native_dt(h, router, shared_gate)
    T, d = h.shape
    E = router.shape[0]
    if code is None:
        z = h.float() @ router.float().t()
        sg = torch.sigmoid(h.float() @ shared_gate.float().reshape(-1)) if shared_gate is not None else None
        if rule.softmax:
            s = torch.softmax(z, -1)
            c = s if rule.correction is None else s + rule.correction
            best = c.view(T, rule.groups, -1).amax(-1)
            kept = torch.zeros_like(best, dtype=torch.bool).scatter_(1, best.topk(rule.keep, dim=-1).indices, True)
            ids = c.masked_fill(~kept.repeat_interleave(E // rule.groups, 1), -torch.inf).topk(top, dim=-1).indices
            w = s.gather(1, ids)
            w = w / (w.sum(-1, keepdim=True) + 1e-20)
        else:
            w, ids = torch.sigmoid(z).topk(top, dim=-1)
        return ids.to(torch.int32), w, sg
    assert h.is_contiguous() and router.is_contiguous() and router.shape[1] == d
    ids = torch.empty(T, top, device=h.device, dtype=torch.int32)
    w = torch.empty(T, top, device=h.device, dtype=torch.float32)
    sg = torch.empty(T, device=h.device, dtype=torch.float32) if shared_gate is not None else None
    space = _split_space(h, E, shared_gate, code)  # (held until the launch is on the stream)
    _lib.call("kca_moe_route", code, h.data_ptr(), router.data_ptr(), _lib.ptr(shared_gate), ids.data_ptr(),
              w.data_ptr(), _lib.ptr(sg), T, d, E, top, *_rule_args(rule, E), *_space_args(*space), _lib.stream())
    return ids, w, sg


def _split_space(h: torch.Tensor, E: int, shared_gate: torch.Tensor | None, code: int) -> tuple:
    """Workspace and counters of the router kernel whose cuts of K run in four workgroups, or none: the kernel of one
    workgroup a token block. That serves more than 64 outputs (a token's choice there takes a wave's whole time, and the
    last of four workgroups has four waves), more than 1024 tokens (blocks enough to fill the chip) and captures
    (whose counters would be cleared by a launch of their own)."""
    T, d = h.shape
    n = E + (shared_gate is not None)
    if (code != 1 or n > 64 or T > 1024 or d % 8 or h.data_ptr() % 16 or torch.cuda.is_current_stream_capturing()
            or h.get_device() != torch.cuda.current_device()):
        return None, None
    blocks = -(-T // 16)
    ws = torch.empty(blocks * 256 * (-(-n // 16) * 16), device=h.device, dtype=torch.float32)
    return ws, _lib.counters(h.device, blocks + 1)


def _space_args(ws: torch.Tensor | None, cnt: torch.Tensor | None) -> tuple:
    return (None, 0, None, 0) if ws is None else (ws.data_ptr(), ws.numel(), cnt.data_ptr(), cnt.numel())


def _rule_args(rule: Router, E: int) -> tuple:
    c = rule.correction
    assert c is None or (c.is_contiguous() and c.dtype == torch.float32 and c.numel() == E and rule.softmax)
    return int(rule.softmax), _lib.ptr(c), rule.groups, rule.keep


@dataclasses.dataclass
class Groups:
    """Assignments sorted by expert, in tiles of at most ``mt`` rows of one expert."""
    perm: torch.Tensor
    inv: torch.Tensor     # [T, top]; -1: an identity expert
    tiles: torch.Tensor
    ntiles: torch.Tensor
    mt: int


def tile_rows(T: int, top: int, E: int, d: int, F: int, dtype) -> int:
    """Row limit of an expert tile, by the rows ``r`` that an expert expects (``n`` over the experts): a streaming vector product (1
    .. 8), the weight stream on the matrix cores (32), the prompts' product in narrow blocks (128 or 192 rows x 128 weight rows)
    or wide ones (256 x 256). The lines, with both products of a layer in us on either side (width, experts, top, inner size:
    tokens; weights from memory, uneven routing):

    Vector product in tiles of 8 rows or of 4. Its block holds the tile's rows in LDS, and with 4 of them twice as many blocks
    run on a CU; an expert with more rows streams its weights again, which costs more where rows of weights are longer than the
    2048 that a block takes at one time. 4 up to 3 rows, and for weights of up to 2048 as far as it goes (8, 4):
        4096, 8, 4, 4096: 6: 145, 136; 8: 168, 171; 16: 257, 281     4096, 16, 6, 2048: 8: 151, 139; 16: 218, 219
        4096, 2, 2, 4096: 5: 57, 67; 16: 119, 130                    4096, 2, 1, 8192: 5: 72, 70; 16: 133, 143
        2048, 4, 4, 2048: 5: 37, 38; 16: 76, 72                      2048, 16, 8, 1024: 5: 50, 43; 16: 94, 79
        with a shared expert: 4096, 16, 3, 2048: 8: 112, 106; 16: 170, 155    4096, 8, 4, 4096: 16: 311, 337
    Vector, stream: from 1 row on, 2.25 where rows are longer than 2048 (the vector product's wave then has the longer walk over
    which to hide its reduction). Up to 16 tokens the vector product also carries the shared expert:
        4096, 16, 2, 4096: 17: 226, 240; 24: 270, 262      4096, 16, 3, 2048: 17: 158, 135
        2048, 32, 4, 1024: 17: 83, 73; 24: 97, 76          1024, 64, 2, 512: 17: 27, 26; 32: 39, 36
    Stream, narrow: a stream tile holds 32 rows, past which weights are read again, so it ends at 20 rows, as experts are uneven
    -- at 36 where narrow blocks (``blocks`` of 64 weight rows) are fewer than the 512 that run at one time, at 52 where they are less
    than half as many (stream tiles then have more of the chip):
        4096, 16, 2, 4096: 160: 283, 295; 260: 352, 301    2048, 32, 4, 1024: 128: 86, 94; 200: 96, 94; 240: 99, 94
        2048, 24, 5, 768: 153: 66, 71; 192: 73, 73         1536, 32, 4, 704: 256: 56, 58; 320: 65, 59
        5120, 8, 2, 2560: 100: 134, 149; 160: 170, 154     1024, 16, 2, 512: 384: 20, 22; 448: 25, 26; 2048, 16, 4, 512: 192: 33, 34; 224: 45, 40
    without it (widths that are no multiple of 64) vector, narrow: 4 rows:
        4104, 16, 2, 2056: r 3: 179, 154; 8: 335, 180      1032, 16, 2, 520: r 4: 34, 22      4104, 16, 2, 4104: r 3: 334, 337; 4: 376, 329
    Narrow, 128 rows or 192: the larger tile saves a second one a little over 128 rows and costs one over 192; uneven experts
    have more than 128 from some 100 on, and where rows are long it costs nothing from 56 on (4096, 16, 3, 2048 of 20 outputs, the largest
    expert at twice the mean: 400: 200, 191; 467: 218, 187; 600: 212, 194; five layers with other routing .99 to 1.02). Without so
    many blocks two thirds of the 512 places have to be taken, or a tile's length counts for more than their number, and r has to be
    past 130, as identity outputs count as experts here. Time of 192 rows over that of 128 at 115 to 175 rows (even, uneven
    and very uneven routing), 256 to 320 blocks .98 to 1.07 (8 layers; 2048, 28, 4, 640: 1.00, 1.03, 1.03), 352 (1536, 32, 4, 704) .97, .91, .91,
    384 (four layers) .92 to .97, .90 to .97, .91 to .99, 432 to 480 .85 to .90, .93 to 1.02, 1.0 to 1.06; with a quarter of identity outputs:
        2048, 24, 5, 768: r 104: 82, 83; 121: 84, 82; 136: 86, 84     2048, 30, 5, 704: 121: 93, 99; 136: 103, 102; 145: 105, 101
        2048, 24, 4, 896: 121: 86, 89; 136: 103, 92                   2048, 36, 5, 640: 121: 91, 99; 136: 95, 100; 145: 103, 101
    Narrow, wide: a wide block is alone on its CU. It wins where the matrix cores bound the products, from about 150 rows (64
    where a contraction is long), if its rounds are well filled (``fill``: the blocks' time over that of the rounds that they
    take; identity outputs count as experts here, so it is an estimate):
        4096, 16, 2, 4096: 300: 305, 306; 700: 338, 322; 2500: 610, 505    2048, 32, 4, 1024: 500: 93, 103; 1150: 115, 115; 3000: 211, 172
        4096, 16, 3, 2048: 900: 208, 209; 1500: 295, 227                   2048, 24, 5, 768: 777: 83, 85; 1300: 96, 86; 4096: 231, 189
    or with any rows where narrow blocks do not fill the chip and wide ones of both products are one round on more than half of
    the CUs. Wide over narrow at 40 to 100 rows, 5 layers: even routing .86 to .96, uneven .81 to 1.2, very uneven .87 to 1.3 (blocks of the
    products; r 40, 80, 110; narrow, wide):
        5120, 8, 2, 2560 (160, 160): 161, 138; 173, 161; 179, 187     5632, 6, 2, 2816 (132, 132): 166, 143; 173, 159; 187, 180
        4352, 8, 2, 2176 (136, 136): 135, 117; 131, 152; 141, 153     5120, 8, 2, 3840 (240, 160): 201, 180; 225, 210; 247, 218
        4096, 8, 2, 2560 (160, 128): 129, 130; 143, 154; 153, 161     5120, 6, 2, 5120 (240, 120): 184, 194
    (All with ordinary loads. Non-temporal weights, sublayer, narrow, wide: 4096, 16, 2, 4096: 300: 317, 333; 777: 380, 350; 2048, 32, 4, 1024:
    500: 118, 127; 900: 137, 138; 1200: 147, 141; 2048, 24, 5, 768: 500: 97, 104; 777: 110, 110; with four identity outputs, which the rule counts as
    experts, 4096, 16, 3, 2048: 500: 205, 221; 640: 240, 226; 777: 250, 227.)"""
    n = T * top
    used = min(E, n)
    # 32-bit offsets into an expert's weights and the rows of a tile (elsewhere only 128-row tiles have longer ones)
    near = 4 * F * d < 2 ** 32 and 2 * T * d < 2 ** 31 and 2 * GEMM_ROWS * F < 2 ** 31
    gemm = dtype == torch.bfloat16 and d % 8 == 0 and F % 8 == 0
    if gemm and not near and n > 16 * used:
        return 128
    if gemm and near:
        stream = d % 64 == 0 and F % 64 == 0
        r, short, blocks = n / used, min(d, F), used * (F // 64)
        full = blocks >= 512
        if r > ((20 if full else 36 if blocks >= 256 else 52) if stream else 4):
            if stream:
                tiles = used * -(-r // GEMM_ROWS)
                up, down = tiles * -(-F // 128), tiles * -(-d // 256)  # wide blocks of the two products; rounds of one a CU
                fill = (up * d + down * F) / (256 * (-(-up // 256) * d + -(-down // 256) * F))
                once = max(up, down) <= 256 and min(up, down) > 128
                if r > GEMM_ROWS:
                    wide = fill >= 0.8 or (fill >= 0.6 and r > 480 and short >= 2048)
                else:
                    wide = (r > 64 and short >= 4096 or once and not full and short >= 2048 or r > 150 and (once or fill >= 0.8)
                            or r > 175 and fill >= 0.6 and short >= 2048)
                if wide:
                    return GEMM_ROWS
            elif r > 96 and (short >= 4096 or (short >= 1024 and r > 512)):
                return GEMM_ROWS
            two = r > (56 if short >= 2048 else 100) if full else r > 130 and 3 * blocks >= 2 * 512  # a 128-row tile is often not enough
            return 192 if (two and r <= 175) or r > 240 else 128
        if stream and T > SHARED_ROWS and r > (2.25 if d > 2048 else 1):
            return STREAM_ROWS
    if dtype == torch.bfloat16 and T > 4 and (n <= 3 * used or (T <= SHARED_ROWS and max(d, F) <= 2048)):
        return 4
    return 1 if T == 1 else 2 if T == 2 else 4 if T <= 4 else 8


def _groups(T: int, top: int, E: int, mt: int, device) -> Groups:
    n = T * top
    z = dict(device=device, dtype=torch.int32)
    return Groups(torch.empty(n, **z), torch.empty(T, top, **z), torch.empty(min(E, n) + n // mt, 5, **z),
                  torch.empty(1, **z), mt)


def route_group(h: torch.Tensor, router: torch.Tensor, top: int, shared_gate: torch.Tensor | None, mt: int,
                rule: Router = SIGMOID):
    """``route`` and ``group`` -> (ids, weights, shared gate, groups); one launch for up to 16 bf16 tokens, and up to 1024
    where the router's split kernel runs (its own time and the grouping's, us, two launches against one: 32 tokens of 4096,
    20 outputs 13.9, 12.7; 300 14.7, 13.8; 777 of 2048 15.0, 14.3; the gap between them and a call's 9 us on the host come
    on top)."""
    T, d = h.shape
    E = router.shape[0]
    real = E - rule.identity
    one, space = False, (None, None)
    if native_dt(h, router, shared_gate) == 1 and T <= 1024 and top <= 64 and d % 8 == 0:
        if T <= 16:
            one = not rule.softmax or E <= 384
        if one or (E + (shared_gate is not None) <= 64 and router.data_ptr() % 16 == 0
                   and (shared_gate is None or shared_gate.data_ptr() % 16 == 0)):
            space = _split_space(h, E, shared_gate, 1)  # (held until the launch is on the stream)
            one = one or space[0] is not None
    if one:
        g = _groups(T, top, real, mt, h.device)
        ids = torch.empty(T, top, device=h.device, dtype=torch.int32)
        w = torch.empty(T, top, device=h.device, dtype=torch.float32)
        sg = torch.empty(T, device=h.device, dtype=torch.float32) if shared_gate is not None else None
        assert h.is_contiguous() and router.is_contiguous() and router.shape[1] == d
        _lib.call("kca_moe_route_group", h.data_ptr(), router.data_ptr(), _lib.ptr(shared_gate), ids.data_ptr(),
                  w.data_ptr(), _lib.ptr(sg), T, d, E, real, top, *_rule_args(rule, E), mt, g.perm.data_ptr(), g.inv.data_ptr(),
                  g.tiles.data_ptr(), g.tiles.shape[0], g.ntiles.data_ptr(), *_space_args(*space), _lib.stream())
        return ids, w, sg, g
    ids, w, sg = route(h, router, top, shared_gate, rule)
    return ids, w, sg, group(ids, real, mt)


def group(ids: torch.Tensor, E: int, mt: int) -> Groups:
    """Ids of ``E`` and beyond (identity experts) take no row."""
    T, top = ids.shape
    n = T * top
    g = _groups(T, top, E, mt, ids.device)
    mx = g.tiles.shape[0]
    if not ids.is_cuda:
        flat = ids.reshape(-1)
        real = int((flat < E).sum())
        order = torch.argsort(flat, stable=True)
        g.perm.copy_(order)
        g.inv.view(-1)[order] = torch.where(torch.arange(n) < real, torch.arange(n), -1).to(torch.int32)
        g.perm[real:] = -1
        return g
    _lib.call("kca_moe_group", ids.data_ptr(), n, E, mt, g.perm.data_ptr(), g.inv.data_ptr(), g.tiles.data_ptr(), mx,
              g.ntiles.data_ptr(), _lib.stream())
    return g


def shared_ok(T: int, mt: int) -> bool:
    """Whether a shared expert streams beside the routed ones' (``experts``): few tokens, streaming products."""
    return mt <= 8 and T <= SHARED_ROWS


def experts(h: torch.Tensor, ids: torch.Tensor, weights: torch.Tensor, gate_up: torch.Tensor, down: torch.Tensor,
            g: Groups, scale_in: bool = True, shared: tuple | None = None):
    """Output rows [n, d] of the routed experts in ``g``'s sorted order. ``shared`` (gate and up [2F', d], down [d, F']): an
    ungated expert for every token in the same launches (``shared_ok``) -> (rows, its output [T, d])."""
    E, F2, d = gate_up.shape
    F, top, n, T = F2 // 2, ids.shape[1], ids.numel(), h.shape[0]
    code = native_dt(h, gate_up, down, *(shared or ()))
    if code is None:
        flat, wt = ids.reshape(-1).long(), weights.reshape(-1)
        y = torch.empty(n, d, dtype=h.dtype)

        def ff(x, up, dn, s_in=1.0):
            u = up.float() @ (x * s_in)
            k = u.shape[0] // 2
            return dn.float() @ (torch.nn.functional.silu(u[:k]) * u[k:])

        for pos, a in enumerate(g.perm.tolist()):
            if a < 0:
                break
            e, w = int(flat[a]), float(wt[a])
            y[pos] = (ff(h[a // top].float(), gate_up[e], down[e], w if scale_in else 1.0) * (1.0 if scale_in else w)).to(h.dtype)
        return y if shared is None else (y, torch.stack([ff(r.float(), *shared).to(h.dtype) for r in h]))
    assert h.is_contiguous() and gate_up.is_contiguous() and down.is_contiguous() and down.shape == (E, d, F)
    if (g.mt == STREAM_ROWS and shared is None and n <= (3 if d > 2048 else 2) * E
            and (gate_up.data_ptr() % 16 or down.data_ptr() % 16)):
        # weights that the stream's loads do not fit, few rows of each: the vector product reads them where they are, in its own order
        own = group(ids, E, 8)
        y = experts(h, ids, weights, gate_up, down, own, scale_in)
        return y[own.inv.view(-1)[g.perm.clamp(0, n - 1).long()].clamp(min=0).long()]
    if g.mt > 8:  # (16-byte loads; the vector product has any address)
        h, gate_up, down = (t if t.data_ptr() % 16 == 0 else t.clone() for t in (h, gate_up, down))
    act = torch.empty(n, F, device=h.device, dtype=h.dtype)
    y = torch.empty(n, d, device=h.device, dtype=h.dtype)
    mx = g.tiles.shape[0]
    common = (g.perm.data_ptr(), weights.data_ptr(), g.tiles.data_ptr(), g.ntiles.data_ptr(), mx, g.mt, top)
    up_s = down_s = (None, None, None, 0, 0, 0)
    if shared is not None:
        w_up, w_down = shared
        Fs = w_down.shape[1]
        assert shared_ok(T, g.mt) and w_up.is_contiguous() and w_down.is_contiguous() and w_up.shape == (2 * Fs, d)
        act_s, y_s = torch.empty(T, Fs, device=h.device, dtype=h.dtype), torch.empty(T, d, device=h.device, dtype=h.dtype)
        up_s = (h.data_ptr(), w_up.data_ptr(), act_s.data_ptr(), T, Fs, d)
        down_s = (act_s.data_ptr(), w_down.data_ptr(), y_s.data_ptr(), T, d, Fs)
    _lib.call("kca_moe_expert", code, h.data_ptr(), gate_up.data_ptr(), act.data_ptr(), *common, F, d, 1,
              int(scale_in), *up_s, T, _lib.stream())
    _lib.call("kca_moe_expert", code, act.data_ptr(), down.data_ptr(), y.data_ptr(), *common, d, F, 0,
              int(not scale_in), *down_s, n, _lib.stream())
    return y if shared is None else (y, y_s)


ACT_ROWS = {"gelu": 0, "silu_gated": 1, "gelu_tanh_gated": 2, "tanh": 3, "relu2": 4, "softcap": 5}


def act_rows(x: torch.Tensor, out: torch.Tensor, gated: bool, row_scale: torch.Tensor | None = None, *,
             act: str | None = None, bias: torch.Tensor | None = None, cap: float = 0.0) -> torch.Tensor:
    """out = gelu(x) (exact), or silu(gate) * up * row_scale with x = [gate | up]; strided rows. ``act`` names
    another form (``ACT_ROWS``; "softcap": cap tanh(x / cap)); ``bias`` is added to x first. Without a gate, out
    may be x."""
    T, F = out.shape
    act = act or ("silu_gated" if gated else "gelu")
    gated = act.endswith("_gated")
    code = native_dt(x, out, bias)
    assert x.shape == (T, 2 * F if gated else F) and x.stride(1) == 1 and out.stride(1) == 1
    assert bias is None or (bias.is_contiguous() and bias.numel() == x.shape[1])
    if code is None:
        xf = x.float() if bias is None else x.float() + bias.float()
        if gated:
            g = xf[:, :F]
            y = (torch.nn.functional.silu(g) if act == "silu_gated" else
                 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))) * xf[:, F:]
            out.copy_(y if row_scale is None else y * row_scale[:, None])
        else:
            out.copy_(torch.tanh(xf) if act == "tanh" else torch.relu(xf) ** 2 if act == "relu2" else
                      cap * torch.tanh(xf / cap) if act == "softcap" else 0.5 * xf * (1 + torch.erf(xf / math.sqrt(2.0))))
        return out
    _lib.call("kca_act_rows", code, ACT_ROWS[act], x.data_ptr(), x.stride(0), _lib.ptr(row_scale), _lib.ptr(bias),
              out.data_ptr(), out.stride(0), T, F, float(cap), _lib.stream())
    return out


__all__ = ["Router", "SIGMOID", "route", "group", "route_group", "experts", "shared_ok", "act_rows", "tile_rows", "Groups"]
