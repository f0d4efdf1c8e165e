"""Linear layers over many rows: the library's products forward and for the
input gradient, this package's kernels for the weight and bias gradients.

A weight gradient ``dy^T x`` reduces over every row into a small matrix.  The
library runs that on a few dozen workgroups (640 x 128 over 40 000 rows: 243 us,
here 94);
``maloq_rows_dw`` splits the rows over the whole chip and sums the parts in a
fixed order, on the bf16 matrix cores at fp32 exactness.  The layer itself is in C++
(torch_ops.cpp), so that it takes no more of the host than torch's: forward and
backward 112 us against 121 (a Python autograd function: 164).
"""
from __future__ import annotations

import torch
import torch.nn.functional as F

from . import _lib

# From this many rows on the split kernel is the faster one.  640 x 128 and 128 x 128,
# library -> here: 4096 rows 25 -> 31 and 25 -> 27 us (two launches), 8192 50 -> 34 and
# 45 -> 29, 16 384 96 -> 49 and 91 -> 34.
MIN_ROWS = 8192


def rows_weight_grad(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """``dy^T x`` [n, k] of fp32 GPU matrices dy [rows, n] and x [rows, k]."""
    from . import ops
    return ops.rows_weight_grad(dy, x)


def rows_sum(dy: torch.Tensor) -> torch.Tensor:
    """Column sums [n] of an fp32 GPU matrix [rows, n] (maloq_message_colsum)."""
    from . import ops
    return ops.rows_sum(dy)


def linear(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """``F.linear`` on [rows, k], with the gradients above for many fp32 rows."""
    fast = (x.is_cuda and x.dtype == w.dtype == torch.float32 and (b is None or b.dtype == torch.float32)
            and x.dim() == 2 and x.shape[0] >= MIN_ROWS and torch.is_grad_enabled() and w.requires_grad
            and not torch.is_autocast_enabled() and _lib.eager(x, w, b))
    if not fast:
        return F.linear(x, w, b)
    from . import ops
    return ops.rows_linear(x, w, b)
