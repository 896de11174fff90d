"""Linear layers whose backward runs both GEMMs in the K-contiguous ("TN") layout.

PyTorch's Linear backward issues dX = dY W as an NN GEMM and dW = dY^T X as an
NT GEMM; on MI355X (hipBLASLt, GPT-J shapes, profiles/gemm_layout_gptj_r1.jsonl)
those run at 1.21-1.31 and 1.10-1.15 PFLOP/s, against 1.43-1.54 for the same
math with both operands K-contiguous. ``TLinear`` keeps a transposed copy of
its weight (refreshed after every optimizer step: ~4.5 ms for GPT-J-6B) for
dX = F.linear(dY, W^T), and transposes dY and X with ``kca_transpose_bf16``
(HBM-speed, csrc/kernels/transpose.hip) so that dW = F.linear(dY^T, X^T).
CPU tensors and inference use plain ``F.linear``.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib


def transpose(x: torch.Tensor) -> torch.Tensor:
    """[R, C] -> contiguous [C, R]; native for bf16 GPU tensors with R, C % 8 == 0."""
    R, C = x.shape
    if (_lib.use_native(x) and R % 8 == 0 and C % 8 == 0 and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0):
        out = torch.empty(C, R, device=x.device, dtype=x.dtype)
        _lib.call("kca_transpose_bf16", x.data_ptr(), x.stride(0), out.data_ptr(), R, R, C, _lib.stream())
        return out
    return x.t().contiguous()


def _tn_ok(t: torch.Tensor) -> bool:
    return t.shape[0] % 8 == 0 and t.shape[1] % 8 == 0


class _LinearTN(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias, layer):
        y = F.linear(x, weight, bias)
        ctx.save_for_backward(x, weight)
        ctx.layer = layer
        ctx.has_bias = bias is not None
        return y

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        K, N = x.shape[-1], dy.shape[-1]
        x2 = x.reshape(-1, K)
        dy2 = dy.reshape(-1, N).contiguous()
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            wt = ctx.layer.weight_t
            dx = (F.linear(dy2, wt) if wt is not None else dy2 @ weight).view(x.shape)
        if ctx.needs_input_grad[1]:
            if _tn_ok(dy2) and _tn_ok(x2):
                dw = F.linear(transpose(dy2), transpose(x2))
            else:
                dw = dy2.t() @ x2
        if ctx.has_bias and ctx.needs_input_grad[2]:
            db = dy2.sum(0)
        return dx, dw, db, None


class _ParamLinear(torch.autograd.Function):
    """y = x W^T + b that saves the Parameter W itself for backward. F.linear
    saves ``W.t()`` -- a view that pins W's storage at forward time; ZeRO-3
    (train/engine.py) swaps a released parameter's storage out after forward
    and back in (re-gathered) before backward, which only works when the
    autograd graph refers to the Parameter."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        return F.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        K, N = x.shape[-1], dy.shape[-1]
        x2 = x.reshape(-1, K)
        dy2 = dy.reshape(-1, N)
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            dx = (dy2 @ weight).view(x.shape)
        if ctx.needs_input_grad[1]:
            dw = dy2.t() @ x2
        if ctx.has_bias and ctx.needs_input_grad[2]:
            db = dy2.sum(0)
        return dx, dw, db


def param_linear(x, weight, bias=None):
    if torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad):
        return _ParamLinear.apply(x, weight, bias)
    return F.linear(x, weight, bias)


class TLinear(nn.Linear):
    """nn.Linear (same parameters / state dict) with the TN backward above when
    ``enable_tn(True)`` was called and the input is a bf16 GPU tensor."""

    weight_t: torch.Tensor | None

    def __init__(self, *a, **kw):
        super().__init__(*a, **kw)
        self.weight_t = None
        self._tn = False

    def enable_tn(self, on: bool = True):
        # any 8-aligned shape: dX runs TN off weight_t, dW TN on transposed dY / X (edge tiles of
        # the transpose kernel cover GPT-J's 50400-row LM head: 12.2 ms NT per micro-batch before)
        self._tn = bool(on) and self.weight.is_cuda and self.weight.dtype == torch.bfloat16 \
            and self.weight.shape[0] % 8 == 0 and self.weight.shape[1] % 8 == 0
        self.weight_t = torch.empty(self.weight.shape[1], self.weight.shape[0], device=self.weight.device,
                                    dtype=self.weight.dtype) if self._tn else None
        self.refresh_transposed()

    @torch.no_grad()
    def refresh_transposed(self):
        if self.weight_t is not None:
            w = self.weight.detach()
            if not _tn_ok(w):
                self.weight_t.copy_(w.t())
                return
            _lib.call("kca_transpose_bf16", w.data_ptr(), w.stride(0), self.weight_t.data_ptr(), w.shape[0],
                      w.shape[0], w.shape[1], _lib.stream())

    def forward(self, x):
        if self._tn and torch.is_grad_enabled() and (x.requires_grad or self.weight.requires_grad) \
                and x.is_cuda and x.dtype == torch.bfloat16:
            return _LinearTN.apply(x, self.weight, self.bias, self)
        return linear_rows(x, self.weight, self.bias)


__all__ = ["TLinear", "transpose", "param_linear", "linear_rows"]


# ---------------------------------------------------------------- long prompts: whole waves, then the rest
_CUS, _TILE = 256, 256


def wave_rows(rows: int, n: int, k: int) -> int:
    """Rows of ``x[rows, k] W[n, k]^T`` for a first launch, the others go in a second; ``rows`` itself: one launch.

    hipBLASLt's output blocks are 256 x 256 at these sizes, one a CU. A product whose blocks fill whole waves of the 256
    CUs runs at 1500 to 1600 TFLOP/s; one with a last wave of a few blocks at 690 to 1200, for the chip waits on it, or
    on the smaller blocks that the library then takes for all rows. So the rows that fill whole waves are one launch.
    Measured, us, one launch against two: 5400 rows of 16384 x 4096 621 : 483, of 4096 x 16384 982 : 502, of
    12288 x 4096 419 : 387; 4209 rows 422 : 374, 844 : 382, 398 : 282; 7333 rows 694 : 652, 1172 : 709; 5762 rows of
    8192 x 2048 210 : 143. The worst: 6800 rows of 4096 x 4096 159 : 164, 3189 rows of 8192 x 2048 87 : 89.

    Left in one launch: up to 2048 rows (1700 of 16384 x 4096 165 : 172), k below 2048 (a second launch costs as
    much as the idle CUs), widths whose blocks fill a wave only at more rows (6144 and 2048 wide: 8192; there a
    first part of nearly whole waves loses, 7344 rows of 6144 x 2048 134 : 142), and rests of 1536 to 2048 rows where a
    wave is no more than that (they fill it nearly: 3948 rows of 8192 x 2048 95 : 98, 3588 of 8192 x 4096 170 : 179) or k is long
    (1600 to 1850 rows of 4096 x 16384 run at 560 TFLOP/s: 5888 rows 575 : 752, though 5636 883 : 723). Elsewhere such rests
    gain as others do: 5996 rows of 12288 x 4096 543 : 409, 5636 432 : 392, of 4096 x 4096 172 : 154."""
    across = -(-n // _TILE)
    wave = _TILE * (_CUS // math.gcd(across, _CUS))  # the fewest rows whose blocks fill whole waves
    first = rows // wave * wave
    if first < 2048 or first == rows or k < 2048 or (1536 < rows - first < 2048 and (wave <= 2048 or k > 8192)):
        return rows
    return first


FEW_ROWS = 128


def few_rows(rows: int, n: int, k: int, captured: bool = False) -> bool:
    """Whether a product of few rows goes to the weight-streaming kernel. On the GPU, us, hipBLASLt : the kernel, weights cold, in captures
    (where a product cut over K takes 1.6 to 2 us more, a fill of the graph's own counters, not counted here):

        12288 x 4096  16 rows 28.1 : 19.4    32: 22.5 : 19.6    64: 24.7 : 24.0    96: 29.5 : 31.6    128: 31.7 : 33.3
        16384 x 4096          33.1 : 23.2        31.5 : 22.1        32.5 : 25.6        34.7 : 33.7         36.6 : 35.1
        4096 x 4096           15.3 : 11.0        12.9 : 11.2        14.8 : 12.5        21.8 : 15.8         24.2 : 16.6
        4096 x 16384          30.1 : 25.0        33.9 : 25.9        41.5 : 29.3        68.0 : 39.2         80.8 : 41.4
        8192 x 2048           12.8 : 10.1        12.9 : 10.3        13.4 : 11.3        14.3 : 15.0         15.7 : 15.6
        5120 x 20480           114 : 38           121 : 39           129 : 46           139 : 62            146 : 64
        14336 x 14336         81.1 : 66.9        80.1 : 68.9        91.2 : 82.3       101.2 : 108.3       118.7 : 112.2
        50400 x 4096          80.7 : 67.8        77.2 : 71.0        82.2 : 76.4        85.1 : 91.1         88.1 : 95.5

    A call costs the host 6 to 12 us less, and a layer of a short prompt is issued in about the time that it runs in. So an eager
    call takes the kernel also where it is a little slower: four GPT-J layers of 4096, 100 tokens, 1030 us with the library from 65
    rows on for 12288 and 16384 outputs, 900 without it; of 2048, 980 and 735. Not past 2^27 weights and 64 rows, unless few
    blocks leave the library's products without CUs; and up to 24 rows where blocks of 64 weight rows are more than the CUs (24: 20480 x 5120
    43.1 : 42.4, 24576 x 6144 70.8 : 53.2; 64: 48.1 : 51.1, 73.9 : 59.8). More than 128 rows: the library (200 rows of 12288 x 4096 39.9 : 52.5).
    In a capture there is no host time to save: 16 rows of 1024 x 1024, cut over K, 7.2 : 6.7 and the fill."""
    if n > 64 * _CUS:
        return rows <= 24
    if captured:
        large = n * k >= 1 << 24
        return rows <= FEW_ROWS and (n <= 6144 and large if rows > 64 else _k_slices(n, k) == 1 or (rows > 24 and large))
    return rows <= 64 or (rows <= FEW_ROWS and (n <= 6144 or n * k <= 1 << 27))


def _k_slices(n: int, k: int) -> int:
    """Slices of K for the few-rows kernel's blocks of 64 weight rows: about one block a CU, of 512 or more of K each."""
    return max(1, min(_CUS // -(-n // 64), k // 512))


def _rows_mm(x2: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None) -> torch.Tensor | None:
    """The product of up to FEW_ROWS rows on the weight-streaming kernel; None: sizes or alignment it does not take. One row, and two
    where the vector kernel of the decode steps holds them in registers, go to that: no stage in LDS, no rows that are not there. us, rows'
    kernel : vector kernel, one row and two: 50400 x 4096 67.6 : 56.4, 59.3; 12288 x 4096 20.2 : 16.2, 17.9; 4096 x 16384 25.7 :
    21.8, 37.0; 2048 x 8192 11.2 : 7.6, 8.5; 14336 x 14336 67.8 : 59.5; 4096 x 1024 6.9 : 4.8, 5.9; short rows of wide
    weights stay: 32000 x 1024 13.3 : 16.4, 23.3; 50400 x 768 15.5 : 23.3. Errors against 64 bits are the same."""
    rows, k = x2.shape
    n = weight.shape[0]
    if (n % 16 or k % 64 or k == 0 or 2 * max(n, rows) * k >= 1 << 32 or not weight.is_contiguous() or x2.data_ptr() % 16
            or weight.data_ptr() % 16 or (bias is not None and not bias.is_contiguous()) or not _lib.has("kca_rows_mm")):
        return None
    bf16 = x2.dtype == torch.bfloat16
    if (rows == 1 or (rows == 2 and bf16 and k <= 8192)) and (k >= 2048 or n <= 4096):
        y = torch.empty(rows, n, device=x2.device, dtype=x2.dtype)
        _lib.call("kca_skinny_gemm" if bf16 else "kca_skinny_gemm_f16", x2.data_ptr(), k, weight.data_ptr(), _lib.ptr(bias), y.data_ptr(),
                  n, rows, n, k, 0, _lib.stream())
        return y
    ks, ws, cnt = _k_slices(n, k), None, None
    if ks > 1:
        blocks = -(-n // 64)
        ws = torch.empty(blocks * ks * 64 * (32 if rows <= 32 else 64 if rows <= 64 else 128), device=x2.device, dtype=torch.float32)
        cnt = _lib.counters(x2.device, blocks)
    y = torch.empty(rows, n, device=x2.device, dtype=x2.dtype)
    _lib.call("kca_rows_mm", 1 if bf16 else 2, x2.data_ptr(), weight.data_ptr(), _lib.ptr(bias),
              y.data_ptr(), _lib.ptr(ws), _lib.ptr(cnt), 0 if ws is None else ws.numel(), 0 if cnt is None else cnt.numel(),
              rows, n, k, ks, _lib.stream())
    return y


def linear_rows(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """``F.linear`` without gradients: few rows on the weight-streaming kernel (``few_rows``), many in one product or two
    (``wave_rows``). ``F.linear`` itself for all else (a gradient or a tangent recorded, a transform or autocast at work,
    tensor subclasses, strided rows, other types)."""
    n, k = weight.shape
    if (torch.is_grad_enabled() or not x.is_cuda or x.dtype not in (torch.bfloat16, torch.float16) or x.numel() == 0
            or x.shape[-1] != k):
        return F.linear(x, weight, bias)
    rows = x.numel() // k
    few = rows <= FEW_ROWS and few_rows(rows, n, k, torch.cuda.is_current_stream_capturing())
    first = rows if few else wave_rows(rows, n, k)
    if ((first == rows and not few) or not x.is_contiguous() or weight.dtype != x.dtype
            or (bias is not None and (bias.shape != (n,) or bias.dtype != x.dtype)) or not _lib.inference(x, weight, bias)):
        return F.linear(x, weight, bias)
    x2 = x.view(rows, k)
    if few:
        y = _rows_mm(x2, weight, bias)
        return F.linear(x, weight, bias) if y is None else y.view(*x.shape[:-1], n)
    wt = weight.t()
    y = torch.empty(rows, n, device=x.device, dtype=x.dtype)
    for part in (slice(0, first), slice(first, rows)):
        if bias is None:
            torch.mm(x2[part], wt, out=y[part])
        else:
            torch.addmm(bias, x2[part], wt, out=y[part])
    return y.view(*x.shape[:-1], n)


ACTS = {None: 0, "tanh": 1, "none": 2}  # none, GELU (tanh form, erf form)


def _few_weight(weight: torch.Tensor, bias: torch.Tensor | None, rows: int) -> bool:
    n, k = weight.shape
    return (few_rows(rows, n, k) and weight.dtype in (torch.bfloat16, torch.float16) and weight.is_contiguous() and n % 16 == 0
            and n > 0 < k and k % 64 == 0 and 2 * max(n, rows) * k < 1 << 32 and weight.data_ptr() % 16 == 0
            and (bias is None or (bias.shape == (n,) and bias.dtype == weight.dtype and bias.is_contiguous())))


def _few_part(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, rows: int) -> bool:
    return (_few_weight(weight, bias, rows) and x.dtype == weight.dtype and x.numel() == rows * weight.shape[1] and x.is_contiguous()
            and x.data_ptr() % 16 == 0)


def few_rows_serve(rows: int, products, approx: str | None = None) -> bool:
    """Whether these (weight, bias) go to the weight-streaming kernel for ``rows`` fresh rows, with this GELU, before anything is launched."""
    return (0 < rows <= FEW_ROWS and approx in ACTS and all(_few_weight(w, b, rows) for w, b in products)
            and _lib.inference(*(t for p in products for t in p)) and _lib.has("kca_rows_mm_two"))


def few_rows_scratch(rows: int, device: torch.device) -> tuple[torch.Tensor, torch.Tensor]:
    """What the products of up to ``rows`` rows need for their slices of K (some 256 blocks' partial sums and arrival counters, left
    zeroed), for launches that follow one another on one stream."""
    return (torch.empty(_CUS * 64 * (32 if rows <= 32 else 64 if rows <= 64 else 128), device=device, dtype=torch.float32),
            torch.zeros(_CUS, device=device, dtype=torch.int32))


def _few_launch(parts, act: int, act2: int, beside: bool, rows: int, scratch=None, res=None):
    """One launch of ``kca_rows_mm_two`` over one or two (x, weight, bias); None: sizes, types or a mode of torch (gradients,
    transforms, captures without ``few_rows_scratch``, ...) that it does not serve."""
    x = parts[0][0]
    ext = _lib.plain_ext() if scratch is None and x.is_cuda else None
    if ext is not None and 0 < rows <= FEW_ROWS and all(few_rows(rows, *p[1].shape) for p in parts):
        y = ext.few_rows(*parts[0], *(parts[1] if len(parts) > 1 else (None, None, None)), act, act2, beside, rows, res)
        if y is not None:
            _lib.LAUNCHES[0] += 1
            return y
    if (not 0 < rows <= FEW_ROWS or not x.is_cuda or (scratch is None and torch.cuda.is_current_stream_capturing())
            or not all(p[0].dtype == x.dtype and _few_part(*p, rows) for p in parts)
            or (res is not None and (res.dtype != x.dtype or res.numel() != rows * parts[0][1].shape[0] or not res.is_contiguous()
                                     or res.data_ptr() % 8))
            or not _lib.inference(*(t for p in parts for t in p), res) or not _lib.has("kca_rows_mm_two")):
        return None
    outs = [torch.empty(rows, p[1].shape[0], device=x.device, dtype=x.dtype) for p in (parts if beside else parts[:1])]
    blocks = sum(-(-y.shape[1] // 64) for y in outs)
    k = min(p[1].shape[1] for p in parts) if beside else sum(p[1].shape[1] for p in parts)
    ks, ws, cnt = max(1, min(_CUS // blocks, k // 512)), None, None  # (about one block a CU, as _k_slices)
    if ks > 1 and scratch is not None:
        ws, cnt = scratch
    elif ks > 1:
        ws = torch.empty(blocks * ks * 64 * (32 if rows <= 32 else 64 if rows <= 64 else 128), device=x.device, dtype=torch.float32)
        cnt = _lib.counters(x.device, blocks)
    a = []
    for i in range(2):
        if i < len(parts):
            px, w, b = parts[i]
            a += [px.data_ptr(), w.data_ptr(), _lib.ptr(b), outs[i].data_ptr() if i < len(outs) else None, *w.shape, (act, act2)[i]]
        else:
            a += [None, None, None, None, 0, 0, 0]
    _lib.call("kca_rows_mm_two", 1 if x.dtype == torch.bfloat16 else 2, int(beside), *a, _lib.ptr(res), _lib.ptr(ws), _lib.ptr(cnt),
              0 if ws is None else ws.numel(), 0 if cnt is None else cnt.numel(), rows, ks, _lib.stream())
    return outs


def few_rows_gelu(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, approx: str) -> torch.Tensor | None:
    """gelu(x W^T + bias) of few rows in one launch, the GELU on the fp32 sums; None: a call that ``linear_rows`` and
    ``ops.gelu`` serve."""
    rows = x.numel() // x.shape[-1]
    y = _few_launch([(x, weight, bias)], ACTS[approx], 0, False, rows) if approx in ACTS else None
    return None if y is None else y[0].view(*x.shape[:-1], -1)


def few_rows_beside(first: tuple, second: tuple, approx2: str | None = None, scratch=None):
    """Two products (x, weight, bias) of the same few rows in one launch, a GELU on the second's fp32 sums -> (y, y2) or None.
    On the GPU, us, apart and together, 61 rows: 12288 and 16384 x 4096 24.0 + 25.6, 40.5; 6144 and 8192 x 2048 11.0 + 11.3, 16.5;
    128 rows 33.3 + 35.1, 54.9; and a launch and the GELU's less."""
    x = first[0]
    rows = x.numel() // x.shape[-1]
    y = _few_launch([first, second], 0, ACTS[approx2], True, rows, scratch) if approx2 in ACTS else None
    return None if y is None else tuple(t.view(*x.shape[:-1], -1) for t in y)


def few_rows_sum(first: tuple, second: tuple, scratch=None, res: torch.Tensor | None = None) -> torch.Tensor | None:
    """The sum of two products (x, weight, bias) of the same few rows, and of rows ``res``, in one launch, rounded once; or None. On the GPU, us, apart and
    together, 61 rows: 4096 x 16384 and x 4096 29.3 + 12.5, 35.3; 2048 x 8192 and x 2048 13.2 + 8.8, 15.2;
    128 rows 41.4 + 16.6, 49.9."""
    x = first[0]
    rows = x.numel() // x.shape[-1]
    if first[1].shape[0] != second[1].shape[0]:
        return None
    y = _few_launch([first, second], 0, 0, False, rows, scratch, res)
    return None if y is None else y[0].view(*x.shape[:-1], -1)


# ---------------------------------------------------------------- split-K weight gradients
def _wgrad_splits(tokens: int, n: int, k: int) -> int:
    """Token chunks for dW = dY^T X: one hipBLASLt GEMM leaves most CUs idle when the output is
    small and the token (reduction) dimension long (SD UNet linears: 320x320 over 65536 tokens ran
    at ~90 TFLOP/s). Split into a batched GEMM over token chunks + an fp32 sum: 320x320 / 65536
    0.131 -> 0.065 ms, 640x640 / 16384 0.076 -> 0.052 ms, 320x1280 / 65536 0.179 -> 0.103 ms
    (bench/wgrad_splitk_bench.py, profiles/wgrad_splitk_r2.jsonl); 5120x640 is faster unsplit."""
    if tokens < 16384 or n * k > 1_700_000:
        return 1
    s = min(16, tokens // 2048)
    while s > 1 and tokens % s:
        s //= 2
    return s


_COLSUM = __import__("os").environ.get("KCA_COLSUM", "1") not in ("0", "false")  # A/B knob


def column_sum(x2: torch.Tensor, out_dtype: torch.dtype | None = None) -> torch.Tensor:
    """Sum over the rows of a [M, N] tensor (a bias gradient), in ``out_dtype`` (default x2's):
    ``kca_colsum_bf16`` (row-chunk partials, then a small fp32 sum) for contiguous bf16 on the GPU."""
    M, N = x2.shape
    out_dtype = out_dtype or x2.dtype
    if not (_COLSUM and _lib.use_native(x2) and x2.dtype == torch.bfloat16 and x2.is_contiguous() and N % 8 == 0
            and x2.data_ptr() % 16 == 0 and _lib.has("kca_colsum_bf16")):
        return x2.sum(0) if out_dtype == x2.dtype else x2.sum(0, dtype=torch.float32).to(out_dtype)
    rb = max(64, -(-M // 256) // 8 * 8)  # ~256 row chunks
    nb = -(-M // rb)
    part = torch.empty(nb, N, device=x2.device, dtype=torch.float32)
    _lib.call("kca_colsum_bf16", x2.data_ptr(), part.data_ptr(), M, N, rb, _lib.stream())
    return sum_parts(part, out_dtype)


def sum_parts(part: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """[S, *shape] fp32 partials -> their sum over S in ``out_dtype`` (bf16 / fp32): one native pass
    (``kca_col_reduce_f32``) instead of torch's sum + cast."""
    S = part.shape[0]
    C = part[0].numel()
    if (part.is_cuda and part.dtype == torch.float32 and part.is_contiguous() and C % 64 == 0
            and out_dtype in (torch.bfloat16, torch.float32) and _lib.has("kca_col_reduce_f32")):
        out = torch.empty(part.shape[1:], device=part.device, dtype=out_dtype)
        bf = out_dtype == torch.bfloat16
        _lib.call("kca_col_reduce_f32", part.data_ptr(), S, C, out.data_ptr() if bf else None,
                  None if bf else out.data_ptr(), _lib.stream())
        return out
    return part.sum(0).to(out_dtype)


_BMM_F32 = [None]  # aten::bmm.dtype (bf16 in, fp32 out): probed on first use


def _bmm_f32(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    if _BMM_F32[0] is not False and a.is_cuda and a.dtype == torch.bfloat16:
        try:
            r = torch.bmm(a, b, out_dtype=torch.float32)
            _BMM_F32[0] = True
            return r
        except (TypeError, RuntimeError, NotImplementedError):
            _BMM_F32[0] = False
    return torch.bmm(a, b).float()


class _LinearSplitKW(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        return F.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, gy):
        x, w = ctx.saved_tensors
        n, k = w.shape
        gy2 = gy.reshape(-1, n)
        x2 = x.reshape(-1, k)
        gx = gw = gb = None
        if ctx.needs_input_grad[0]:
            gx = (gy2 @ w).view(x.shape)
        if ctx.needs_input_grad[1]:
            t = gy2.shape[0]
            s = _wgrad_splits(t, n, k)
            if s > 1:
                gy2c = gy2 if gy2.is_contiguous() else gy2.contiguous()
                x2c = x2 if x2.is_contiguous() else x2.contiguous()
                # per-chunk products in fp32 straight from the GEMM, one native reduction to w's dtype
                gw = sum_parts(_bmm_f32(gy2c.view(s, t // s, n).transpose(1, 2), x2c.view(s, t // s, k)), w.dtype)
            else:
                gw = gy2.t() @ x2
        if ctx.has_bias and ctx.needs_input_grad[2]:
            gb = column_sum(gy2 if gy2.is_contiguous() else gy2.contiguous())
        return gx, gw, gb


def linear_splitk_wgrad(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """F.linear whose weight gradient splits long token reductions (see _wgrad_splits); plain
    F.linear when no gradient is recorded or off the GPU."""
    if not (torch.is_grad_enabled() and x.is_cuda and weight.requires_grad):
        return F.linear(x, weight, bias)
    return _LinearSplitKW.apply(x, weight, bias)


class SplitKLinear(nn.Linear):
    """nn.Linear (same parameters / state-dict keys) training through linear_splitk_wgrad."""

    def forward(self, x):
        return linear_splitk_wgrad(x, self.weight, self.bias)


_WS: dict[int, torch.Tensor] = {}
_WS_BYTES = 32 << 20


def _workspace(dev: torch.device) -> torch.Tensor | None:
    """hipBLASLt workspace, allocated once per device outside any graph capture."""
    ws = _WS.get(dev.index)
    if ws is None and not torch.cuda.is_current_stream_capturing():
        ws = _WS[dev.index] = torch.empty(_WS_BYTES, device=dev, dtype=torch.uint8)
    return ws


class _LinearResidualFn(torch.autograd.Function):
    """Training ``res + F.linear(x, W, b)``: the forward is the one-GEMM epilogue form; the backward
    passes dY through to ``res`` (no copy), dX = dY W, dW by the split-K weight gradient, db by the
    column-sum kernel -- the residual add's separate read-read-write pass is gone."""

    @staticmethod
    def forward(ctx, x, weight, bias, res):
        with torch.no_grad():
            y = linear_residual(x, weight, bias, res)
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        return y

    @staticmethod
    def backward(ctx, gy):
        x, w = ctx.saved_tensors
        gb = None
        gx, gw, gb0 = _LinearSplitKW.backward(_Saved(x, w, ctx.has_bias, ctx.needs_input_grad[:3]), gy)
        if ctx.has_bias and ctx.needs_input_grad[2]:
            gb = gb0
        return gx, gw, gb, (gy if ctx.needs_input_grad[3] else None)


class _Saved:
    """ctx stand-in for reusing _LinearSplitKW.backward."""

    def __init__(self, x, w, has_bias, needs):
        self.saved_tensors = (x, w)
        self.has_bias = has_bias
        self.needs_input_grad = tuple(needs)


def linear_residual_train(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None,
                          res: torch.Tensor) -> torch.Tensor:
    """``res + F.linear(x, weight, bias)`` with autograd, fused on the GPU (see _LinearResidualFn)."""
    if torch.is_grad_enabled() and _lib.use_native(x, weight, res) and res.stride(-1) == 1 and x.stride(-1) == 1:
        return _LinearResidualFn.apply(x, weight, bias, res)
    return linear_residual(x, weight, bias, res)


def linear_residual(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None,
                    res: torch.Tensor) -> torch.Tensor:
    """``res + F.linear(x, weight, bias)`` in ONE hipBLASLt GEMM (bias and residual in its epilogue,
    csrc/kernels/gemm_lt.hip) at inference on the GPU; the two-pass form otherwise (autograd,
    CPU). ``res`` is any view whose rows are the output rows ([..., N], unit last stride); the
    result has ``res``'s shape."""
    N, K = weight.shape
    if not (not torch.is_grad_enabled() and _lib.use_native(x, weight, res) and (bias is None or bias.is_cuda)
            and x.shape[-1] == K and res.shape[-1] == N and x.stride(-1) == 1 and res.stride(-1) == 1
            and weight.stride(1) == 1 and (bias is None or bias.is_contiguous())):
        return res + F.linear(x, weight, bias).reshape(res.shape)
    x2 = x.reshape(-1, K)
    r2 = res.reshape(-1, N)
    M = x2.shape[0]
    if r2.shape[0] != M or x2.stride(1) != 1 or r2.stride(1) != 1:
        return res + F.linear(x, weight, bias).reshape(res.shape)
    out = torch.empty(M, N, device=x.device, dtype=x.dtype)
    ws = _workspace(x.device)
    _lib.call("kca_gemm_lt", x2.data_ptr(), x2.stride(0), weight.data_ptr(), weight.stride(0), _lib.ptr(bias),
              r2.data_ptr(), r2.stride(0), out.data_ptr(), N, M, N, K, 1.0, _lib.ptr(ws),
              _WS_BYTES if ws is not None else 0, _lib.stream())
    return out.view(res.shape)


def few_rows_head(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None) -> torch.Tensor:
    """Logits [rows, n] of a decode step's rows: past ``few_rows``' 24 rows of more blocks of 64 weight rows than CUs too, where blocks of 128
    are on most CUs (table of ``few_rows``; 48 rows of 43008 x 4096 79.0 : 65.7, of 20480 x 5120, 160 blocks, 47.0 : 48.4)."""
    (rows, k), n = x.shape, weight.shape[0]
    if (n > 64 * _CUS and rows <= (64 if n >= 96 * _CUS else 32) and k >= 1024 and x.dtype in (torch.bfloat16, torch.float16)
            and x.dtype == weight.dtype and x.is_contiguous() and (bias is None or (bias.shape == (n,) and bias.dtype == x.dtype))
            and _lib.inference(x, weight, bias)):
        y = _rows_mm(x, weight, bias)
        if y is not None:
            return y
    return linear_rows(x, weight, bias)
