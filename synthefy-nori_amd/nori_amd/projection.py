"""Projections of the attention sublayers: ``F.linear`` under fp16 autocast on the HIP kernel.

``linear(x, weight)`` is ``torch.nn.functional.linear(x, weight)`` for fp16 operands (what the
reference's projections compute under the GPU's fp16 autocast, layer.py:651-683, 1114-1160):
fp32 sums of fp16 products, rounded once to fp16. ``nori_linear_f16`` (csrc/linear.hip) reads
x and writes the output through strides -- a token subset of each row, a slice of a stacked
output buffer (``out``), the transposed [table, group, row] view of a cell buffer -- without
copies. ``linear`` routes to it the shapes where it is the faster of the two (same-box A/B against the
library GEMM at inner width 128: 139,264 rows x 128 -> 128 in 20 against 26 us, -> 256 in 25.5
against 28, -> 384 in 32 against 59.5; 655,360 rows 67 against 101, 114 against 126, 157 against 261.
At inner width 256 neither is ahead throughout: 65,536 rows 256 -> 256 in 21.4 against 18.8 us, 163,840 in
40.9 against 43.1); everything else (other dtypes, widths or shapes, short operands, CPU
tensors) is ``F.linear``. The two differ only in the order of the fp32 sums.
"""

from __future__ import annotations

import ctypes

import torch

from . import _native as nat

__all__ = ["linear", "linear_head_norm", "linear_param", "linear_residual", "linear_residual_norm", "param_weight",
           "takes_kernel"]

_WIDTHS = (128,)  # inner widths routed to the kernel (it also takes 256, where neither is ahead throughout)
_MAX_N = 384      # output widths up to this
_MIN_ROWS = 4096  # below this the library GEMM's launch is as cheap


def _row_levels(t: torch.Tensor) -> list[tuple[int, int]] | None:
    """The rows of ``t`` [..., C] as at most three (count, stride) levels, outer first (adjacent
    leading dims merged where their strides chain), or None when they need more levels."""
    merged: list[tuple[int, int]] = []
    for size, stride in zip(t.shape[:-1], t.stride()[:-1]):
        size, stride = int(size), int(stride)
        if size == 1:
            continue
        if merged and merged[-1][1] == stride * size:
            merged[-1] = (merged[-1][0] * size, stride)
        else:
            merged.append((size, stride))
    return merged if len(merged) <= 3 else None


def _common_grid(*tensors: torch.Tensor) -> tuple | None:
    """((n_outer, n_mid, n_inner), strides of each tensor ...): one three-level row grid
    addressing the rows of every tensor (same leading shape) in the same order, or None. The
    grid's levels are the union of the tensors' level boundaries; a tensor level that spans
    several grid levels gives each of them its stride times the rows inside it."""
    per = [_row_levels(t) for t in tensors]
    if any(levels is None for levels in per):
        return None
    bounds = set()
    for levels in per:
        prod = 1
        for count, _ in reversed(levels):
            prod *= count
            bounds.add(prod)
    counts, prev = [], 1  # inner first
    for b in sorted(bounds):
        if b % prev:
            return None
        counts.append(b // prev)
        prev = b
    if len(counts) > 3:
        return None
    strides = []
    for levels in per:
        st, gi = [], 0
        for count, stride in reversed(levels):
            inside, mult = 1, 1
            while gi < len(counts) and inside * counts[gi] <= count:
                st.append(stride * mult)
                mult *= counts[gi]
                inside *= counts[gi]
                gi += 1
            if inside != count:
                return None
        strides.append(st)
    pad = 3 - len(counts)
    grid = tuple([1] * pad + counts[::-1])
    return (grid,) + tuple(tuple([0] * pad + st[::-1]) for st in strides)


def takes_kernel(x: torch.Tensor, weight: torch.Tensor, *, any_width: bool = False, min_rows: int = _MIN_ROWS,
                 weight_dtype: torch.dtype = torch.float16) -> bool:
    """Whether ``linear(x, weight)`` runs on the HIP kernel (``any_width``: whether the kernel
    can take the operands at all, whatever the routing rule says; ``weight_dtype`` float32: the one
    that rounds its weights)."""
    if not (x.is_cuda and x.dtype == torch.float16 and weight.dtype == weight_dtype and weight.dim() == 2
            and weight.get_device() == x.get_device()):  # (F.linear refuses a weight on another device)
        return False
    k = int(x.shape[-1])
    widths = (128, 256) if any_width else _WIDTHS
    if k not in widths or int(weight.shape[1]) != k or int(weight.shape[0]) % 4:
        return False
    if not any_width and int(weight.shape[0]) > _MAX_N:
        return False
    if x.stride(-1) != 1:
        return False
    if weight.stride(-1) != 1 or weight.stride(0) * weight.element_size() % 16 or weight.data_ptr() % 16 \
            or x.data_ptr() % 16:
        return False
    if x.numel() // k < min_rows:
        return False
    levels = _row_levels(x)
    return levels is not None and all(st % 8 == 0 for _, st in levels)


def linear(x: torch.Tensor, weight: torch.Tensor, out: torch.Tensor | None = None, *,
           any_width: bool = False) -> torch.Tensor:
    """``F.linear(x, weight)`` (no bias) -> [..., N]; with ``out`` (a view of that shape, any
    row strides) the result is written there and ``out`` returned. ``any_width`` takes the
    kernel for every shape it can (a caller whose strided ``out`` would otherwise cost a copy)."""
    if not takes_kernel(x, weight, any_width=any_width):
        y = torch.nn.functional.linear(x, weight)
        if out is None:
            return y
        out.copy_(y)
        return out
    n = int(weight.shape[0])
    if out is None:
        out = torch.empty(tuple(x.shape[:-1]) + (n,), dtype=torch.float16, device=x.device)
    elif tuple(out.shape) != tuple(x.shape[:-1]) + (n,) or out.dtype != torch.float16 or out.device != x.device:
        raise ValueError(f"out {tuple(out.shape)} {out.dtype} is not the [..., {n}] fp16 result of x {tuple(x.shape)}")
    common = _common_grid(x, out)
    if common is None or out.stride(-1) != 1 or out.data_ptr() % 8 or any(st % 4 for st in common[2]):
        out.copy_(linear(x, weight))
        return out
    (no, nm, ni), (xo, xm, xr), (yo, ym, yr) = common
    nat.check(
        nat.lib().nori_linear_f16(
            ctypes.c_void_p(x.data_ptr()), no, nm, ni, int(x.shape[-1]), xo, xm, xr,
            ctypes.c_void_p(weight.data_ptr()), int(weight.stride(0)), n,
            ctypes.c_void_p(out.data_ptr()), yo, ym, yr, nat.stream_of(x.device),
        ),
        "linear_f16",
    )
    return out


def param_weight(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``weight``, a parameter or rows of one, as ``linear_param`` takes it for operands like x: itself
    where the kernel rounds fp32 weights as it stages them (``nori_linear_f16_w32``), else the cast
    autocast makes, formed by this call. Nothing is kept, so an edit through ``.data``, which moves
    neither address nor version, reaches the next call, and each call is ordered on its own stream."""
    if not torch.is_autocast_enabled("cuda") or weight.dtype not in (torch.float32, torch.float16, torch.bfloat16):
        return weight
    dtype = torch.get_autocast_dtype("cuda")
    if dtype == torch.float16 and takes_kernel(x, weight, weight_dtype=torch.float32):
        return weight
    return weight.to(dtype)


def linear_param(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``linear(x, weight)`` as autocast computes it, of a parameter as it is on this call
    (``param_weight``)."""
    weight = param_weight(x, weight)
    if weight.dtype != torch.float32 or x.dtype != torch.float16:
        return linear(x, weight)
    n = int(weight.shape[0])
    out = torch.empty(tuple(x.shape[:-1]) + (n,), dtype=torch.float16, device=x.device)
    common = _common_grid(x, out)
    if not torch.is_autocast_enabled("cuda") or common is None:
        return linear(x, weight)
    (no, nm, ni), sx, sy = common
    nat.check(
        nat.lib().nori_linear_f16_w32(
            x.data_ptr(), no, nm, ni, int(x.shape[-1]), *sx, weight.data_ptr(), int(weight.stride(0)), n, out.data_ptr(),
            *sy, nat.stream_of(x.device),
        ),
        "linear_f16_w32",
    )
    return out


def linear_head_norm(x: torch.Tensor, weight: torch.Tensor, gain: torch.Tensor, eps: float,
                     norm_cols: int) -> torch.Tensor | None:
    """``linear(x, weight)`` with the first ``norm_cols`` columns taken as heads of 64 and each head
    row RMS-normed with ``gain`` [64], in one kernel (``nori_linear_f16_head_norm``): the
    projection and the per-head q/k norm of ``MultiheadAttention``, each rounded to fp16. Any row
    count; None where the kernel does not take the operands."""
    if gain.shape != (64,) or gain.device != x.device or gain.dtype not in (torch.float32, torch.float16, torch.bfloat16):
        return None
    if norm_cols % 64 or not takes_kernel(x, weight, any_width=True, min_rows=1):
        return None
    n = int(weight.shape[0])
    out = torch.empty(tuple(x.shape[:-1]) + (n,), dtype=torch.float16, device=x.device)
    common = _common_grid(x, out)
    if common is None:
        return None
    (no, nm, ni), sx, sy = common
    gain = gain.contiguous()
    nat.check(
        nat.lib().nori_linear_f16_head_norm(
            x.data_ptr(), no, nm, ni, int(x.shape[-1]), *sx, weight.data_ptr(), int(weight.stride(0)), n, out.data_ptr(),
            *sy, gain.data_ptr(), nat.dtype_code(gain.dtype), float(eps), int(norm_cols), nat.stream_of(x.device),
        ),
        "linear_f16_head_norm",
    )
    return out


def linear_residual_norm(a: torch.Tensor, weight: torch.Tensor, stream: torch.Tensor, alpha: float, eps: float,
                         out: torch.Tensor | None = None, dest: torch.Tensor | None = None) -> torch.Tensor | None:
    """``stream += alpha * F.linear(a, weight)`` in place, then the RMSNorm (no weight, ``eps``)
    of the updated stream rows in fp16, in one kernel (``nori_linear_f16_residual_rms_norm``):
    bit for bit ``linear`` followed by the fused residual + norm pass. ``a`` [..., K] fp16,
    ``weight`` [K, K] fp16, or fp32 rounded to fp16 as it is read (K 128 or 256), ``stream`` [..., K] fp32 with ``a``'s leading shape
    (any row strides: e.g. the [table, row, group] cells beside an attention output in
    [table, group, row] order), ``out`` the same shape in fp16 (new and laid out like
    ``stream`` when None). ``dest`` (``stream``'s shape and strides) takes the sum in ``stream``'s
    place. Returns the normalized rows, or None where the kernel does not take the operands
    (nothing is then written)."""
    if out is None:
        if a.shape != stream.shape:
            return None
        out = torch.empty_like(stream, dtype=torch.float16)
    elif tuple(out.shape) != tuple(a.shape) or out.dtype != torch.float16 or out.stride(-1) != 1:
        return None
    return out if _linear_residual(a, weight, stream, alpha, eps, out, dest) else None


def linear_residual(a: torch.Tensor, weight: torch.Tensor, stream: torch.Tensor, alpha: float,
                    dest: torch.Tensor | None = None) -> bool:
    """``linear_residual_norm`` without the norm; whether the kernel took the operands."""
    return _linear_residual(a, weight, stream, alpha, 0.0, None, dest)


def _linear_residual(a, weight, stream, alpha, eps, out, dest) -> bool:
    k = int(a.shape[-1])
    if not (a.is_cuda and a.dtype == torch.float16 and weight.dtype in (torch.float16, torch.float32) and stream.dtype == torch.float32
            and k in (128, 256) and tuple(weight.shape) == (k, k) and tuple(stream.shape) == tuple(a.shape)
            and stream.device == a.device and weight.device == a.device):
        return False
    if a.stride(-1) != 1 or stream.stride(-1) != 1 or weight.stride(-1) != 1:
        return False
    if dest is None:
        dest = stream
    elif dest.shape != stream.shape or dest.stride() != stream.stride() or dest.dtype != stream.dtype \
            or dest.device != stream.device:
        return False
    common = _common_grid(a, stream) if out is None else _common_grid(a, stream, out)
    if common is None:
        return False
    (no, nm, ni), sa, sx = common[:3]
    sy = (0, 0, 0) if out is None else common[3]
    if (a.data_ptr() % 16 or any(st % 8 for st in sa) or weight.data_ptr() % 16
            or weight.stride(0) * weight.element_size() % 16 or stream.data_ptr() % 16 or dest.data_ptr() % 16 or any(st % 4 for st in sx)
            or (out is not None and (out.data_ptr() % 8 or any(st % 4 for st in sy)))):
        return False
    head = (a.data_ptr(), no, nm, ni, k, *sa, weight.data_ptr(), int(weight.stride(0)))
    update = (float(alpha), stream.data_ptr(), *sx)
    tail = (float(eps), nat.ptr(out), *sy, nat.stream_of(a.device))
    if out is not None and dest is stream and weight.dtype == torch.float16:
        nat.check(nat.lib().nori_linear_f16_residual_rms_norm(*head, *update, *tail), "linear_f16_residual_rms_norm")
    else:
        nat.check(nat.lib().nori_linear_f16_residual(*head, nat.dtype_code(weight.dtype), *update, dest.data_ptr(), *tail),
                  "linear_f16_residual")
    return True
