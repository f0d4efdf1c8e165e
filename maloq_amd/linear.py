"""Linear layers over many rows: the library's products forward and for the
input gradient, this package's kernels for the weight and bias gradients.

A weight gradient ``dy^T x`` reduces over every row into a small matrix.  The
library runs that on a few dozen workgroups (640 x 128 over 40 000 rows: 243 us,
here 94);
``maloq_rows_dw`` splits the rows over the whole chip and sums the parts in a
fixed order, on the bf16 matrix cores at fp32 exactness.
"""
from __future__ import annotations

import torch
import torch.nn.functional as F

from . import _lib

# From this many rows on the split kernel is the faster one.  640 x 128 and 128 x 128,
# library -> here: 4096 rows 25 -> 31 and 25 -> 27 us (two launches), 8192 50 -> 34 and
# 45 -> 29, 16 384 96 -> 49 and 91 -> 34.
MIN_ROWS = 8192


def _row_strided(t: torch.Tensor):
    """``t``, or a copy where the kernel cannot step through its rows, and the row
    stride (of a single row, whose own may be anything: its length)."""
    n = t.shape[1]
    ld = t.stride(0) if t.shape[0] > 1 else n
    return (t, ld) if t.stride(1) == 1 and n <= ld < 1 << 24 else (t.contiguous(), n)


def rows_weight_grad(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """``dy^T x`` [n, k] of fp32 GPU matrices dy [rows, n] and x [rows, k]."""
    (dy, ld_dy), (x, ld_x) = _row_strided(dy), _row_strided(x)
    rows, n, k = dy.shape[0], dy.shape[1], x.shape[1]
    parts = torch.empty(_lib.load().maloq_rows_dw_partials_floats(rows, n, k), device=dy.device, dtype=torch.float32)
    dw = torch.empty(n, k, device=dy.device, dtype=torch.float32)
    _lib.call("maloq_rows_dw", dy, ld_dy, n, x, ld_x, k, rows, parts, dw, _lib.stream_of(dy.device))
    return dw


def rows_sum(dy: torch.Tensor) -> torch.Tensor:
    """Column sums [n] of an fp32 GPU matrix [rows, n] (maloq_message_colsum)."""
    rows, n = dy.shape
    if n % 4:
        return dy.sum(0)
    dy = dy.contiguous()
    parts = torch.empty(max(1, _lib.load().maloq_message_colsum_partials_floats(1, n, rows)), device=dy.device,
                        dtype=torch.float32)
    out = torch.empty(n, device=dy.device, dtype=torch.float32)
    _lib.call("maloq_message_colsum", 0, dy, 1, 0, 1, n, rows, parts, out, _lib.stream_of(dy.device))
    return out


class _RowsLinear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w)
        return F.linear(x, w, b)

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        need_x, need_w, need_b = ctx.needs_input_grad
        # torch's products for a gradient that can be differentiated again
        # (create_graph) or that is batched
        kernels = not torch.is_grad_enabled() and _lib.eager(g, x, w)
        gx = g @ w if need_x else None
        gw = (rows_weight_grad(g, x) if kernels else g.t() @ x) if need_w else None
        gb = (rows_sum(g) if kernels else g.sum(0)) if need_b else None
        return gx, gw, gb


def linear(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """``F.linear`` on [rows, k], with the gradients above for many fp32 rows."""
    fast = (x.is_cuda and x.dtype == w.dtype == torch.float32 and (b is None or b.dtype == torch.float32)
            and x.dim() == 2 and x.shape[0] >= MIN_ROWS and torch.is_grad_enabled() and w.requires_grad
            and not torch.is_autocast_enabled() and _lib.eager(x, w, b))
    return _RowsLinear.apply(x, w, b) if fast else F.linear(x, w, b)
