"""Dense-layer helpers: residual add + RMSNorm, SiLU-gated product, few-row linear.

``add_rms_norm(x, delta, weight, eps)`` stands for ``x = x + delta`` followed
by ``F.rms_norm(x, (H,), weight, eps)`` (DecoderLayer.forward,
model.py:324-344; RMSNorm, model.py:115-122); ``silu_mul(gate_up)`` for
``F.silu(gate) * up`` over the fused gate/up projection (MLP,
model.py:301-311).  Both run one HIP kernel (``mi_add_rms_norm`` /
``mi_silu_mul``); there is no torch fallback.  ``linear(x, weight, bias)`` is
``F.linear`` with a decode step's few rows on ``mi_linear``, and
``linear_silu(x, gate_up)`` is ``silu_mul(linear(x, gate_up))`` with those rows
in one launch (``mi_linear_silu``).
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch._C import _len_torch_dispatch_stack
from torch._C._functorch import peek_interpreter_stack
from torch.autograd import forward_ad
from torch.overrides import has_torch_function

from . import _lib
from ._util import require_dtype, require_gpu, stream_of


def _rows(name: str, t: torch.Tensor, width: int | None = None) -> None:
    require_gpu(name, t)
    require_dtype(name, t, torch.bfloat16)
    if t.dim() != 2 or t.stride(1) != 1:
        raise ValueError(f"{name} must be [rows, width] with a contiguous last axis; got {tuple(t.shape)}")
    if width is not None and t.shape[1] != width:
        raise ValueError(f"{name} must have {width} columns; got {t.shape[1]}")


def add_rms_norm(x: torch.Tensor, delta: torch.Tensor | None, weight: torch.Tensor, eps: float, *,
                 write_x: bool = True, norm: bool = True,
                 h_out: torch.Tensor | None = None) -> torch.Tensor | None:
    """In place: ``x += delta`` (bf16, when ``delta`` is given and ``write_x``);
    returns ``rms_norm(x + delta) * weight`` (or None when ``norm`` is false)."""
    rows, hidden = x.shape
    _rows("x", x)
    if delta is not None:
        _rows("delta", delta, hidden)
        if delta.shape[0] != rows:
            raise ValueError("delta rows differ from x")
    if norm:
        require_gpu("weight", weight)
        require_dtype("weight", weight, torch.bfloat16)
        if weight.dim() != 1 or weight.numel() != hidden or not weight.is_contiguous():
            raise ValueError(f"weight must be a contiguous [{hidden}] tensor")
        if h_out is None:
            h_out = torch.empty(rows, hidden, dtype=x.dtype, device=x.device)
        _rows("h_out", h_out, hidden)
    elif not (write_x and delta is not None):
        raise ValueError("nothing to do: neither the sum nor the norm is requested")
    xo = x if (write_x and delta is not None) else None
    _lib.call("mi_add_rms_norm", x.data_ptr(), x.stride(0),
              delta.data_ptr() if delta is not None else None, delta.stride(0) if delta is not None else 0,
              weight.data_ptr() if norm else None, xo.data_ptr() if xo is not None else None,
              xo.stride(0) if xo is not None else 0, h_out.data_ptr() if norm else None,
              h_out.stride(0) if norm else 0, rows, hidden, float(eps), stream_of(x))
    return h_out if norm else None


def silu_mul(gate_up: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """``silu(gate_up[:, :I]) * gate_up[:, I:]`` as one kernel; returns [rows, I]."""
    _rows("gate_up", gate_up)
    rows, width = gate_up.shape
    if width % 2:
        raise ValueError("gate_up must have an even number of columns")
    inter = width // 2
    if out is None:
        out = torch.empty(rows, inter, dtype=gate_up.dtype, device=gate_up.device)
    _rows("out", out, inter)
    _lib.call("mi_silu_mul", gate_up.data_ptr(), gate_up.stride(0), out.data_ptr(), out.stride(0), rows, inter,
              stream_of(gate_up))
    return out


# What the few-row kernel takes at most: rows, elements that x's rows span, k.
LINEAR_MAX_ROWS = 32
LINEAR_MAX_SPAN = 1 << 29
LINEAR_MAX_K = 1 << 23


def _few_rows(rows: int, n: int, k: int) -> bool:
    """Whether the few-row kernel is the faster one (us, kernel and library).  Up to 16
    rows everywhere but on the largest weights of long rows (59,136 x 8,192, 16 rows:
    181, 170) and those of a few more tiles than it has workgroups at once (10,240 x
    8,192, 16 rows: 38.2, 34.5; 8 rows 35.9, 34.3); up to 32 while k is short (4,096 x
    14,336: 34, 31; 28,672 x 4,096: 46, 55), from 5,120 on without the weights of a
    little over one round of four tiles each (18,432 x 5,120: 46, 43)."""
    if rows <= 16:
        return k < 8192 or n <= 8192 or 16384 <= n <= 32768
    return rows <= LINEAR_MAX_ROWS and (k < 5120 or (k < 8192 and not 16384 < n <= 32768))


def _plain(*tensors: torch.Tensor | None) -> bool:
    """Whether nothing of torch's stands between a call of F.linear and its kernel:
    no function mode or tensor subclass, dispatch mode, function transform,
    forward-mode level or autocast (a call of the library passes all of them by)."""
    return not (has_torch_function(tensors) or _len_torch_dispatch_stack() or peek_interpreter_stack() is not None
                or forward_ad._current_level >= 0 or torch.is_autocast_enabled())


def _takes(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None) -> bool:
    """Whether ``linear`` runs on the few-row kernel."""
    rows, k = x.shape
    n = weight.shape[0]
    return not (weight.dim() != 2 or rows == 0 or n == 0 or not 0 < k <= LINEAR_MAX_K
                or not _few_rows(rows, n, k) or n % 16 or k % 64 or not x.is_cuda
                or not _plain(x, weight, bias)
                or x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or weight.device != x.device
                or weight.shape[1] != k or not weight.is_contiguous() or x.stride(1) != 1 or x.stride(0) % 8
                or x.stride(0) < k or rows * x.stride(0) > LINEAR_MAX_SPAN or x.data_ptr() % 16 or weight.data_ptr() % 16
                or (torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad))
                or (bias is not None and (bias.dtype != torch.bfloat16 or bias.shape != (n,)
                                          or not bias.is_contiguous() or bias.device != x.device
                                          or bias.data_ptr() % 8
                                          or (torch.is_grad_enabled() and bias.requires_grad))))


def linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """``F.linear`` of [rows, k]; a decode step's few rows of bf16 go to the kernel
    that streams the weight once (fp32 accumulation, one rounding), everything else
    to torch."""
    if not _takes(x, weight, bias):
        return F.linear(x, weight, bias)
    rows, k = x.shape
    n = weight.shape[0]
    out = torch.empty(rows, n, dtype=x.dtype, device=x.device)
    _lib.call("mi_linear", x.data_ptr(), x.stride(0), weight.data_ptr(), bias.data_ptr() if bias is not None else None,
              out.data_ptr(), n, rows, n, k, stream_of(x))
    return out


def linear_silu(x: torch.Tensor, gate_up: torch.Tensor) -> torch.Tensor:
    """``silu_mul(linear(x, gate_up))``, the same bits, in one launch where ``linear``
    runs on the few-row kernel."""
    rows, k = x.shape
    n = gate_up.shape[0] // 2
    # (over 16 long rows the pairs of tiles hold too many registers: 51,200 x 5,120, 32
    # rows, 113 us, library and SiLU kernel 96)
    if n % 16 or gate_up.shape[0] % 2 or (rows > 16 and k >= 5120) or not _takes(x, gate_up, None):
        return silu_mul(linear(x, gate_up))
    out = torch.empty(rows, n, dtype=x.dtype, device=x.device)
    _lib.call("mi_linear_silu", x.data_ptr(), x.stride(0), gate_up.data_ptr(), out.data_ptr(), n, rows, n, k,
              stream_of(x))
    return out
