"""Weight and bias gradients of linear layers over many rows (maloq_amd.linear)
at the edges of the kernel's 256 x 256 tiles and of its row splits, against 64
bits, and the layer itself against torch's.

Tolerance: as for the other fp32 products on the bf16 matrix cores (below 2^-23 of a
product rms, and n products added in fp32, 16 at a time, six times over), four times
over, relative 2-norm.
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _tol(n):
    return 4 * (2.0 ** -23 + math.sqrt(3 * n / 8) * 2.0 ** -25)


def _rel(got, ref):
    return ((got.double().cpu() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("rows", [1, 16, 127, 129, 2049, 33000])
@pytest.mark.parametrize("n,k,pad", [(1, 1, 0), (31, 33, 5), (256, 257, 1), (300, 128, 0)])
def test_rows_weight_grad(rows, n, k, pad, device):
    from maloq_amd.linear import rows_weight_grad
    gen = torch.Generator().manual_seed(rows + n)
    # the last columns of wider rows: what lies past a row's end must not count
    dy = torch.randn(rows, n + pad, generator=gen)
    x = torch.randn(rows, k + pad, generator=gen)
    got = rows_weight_grad(dy.to(device)[:, pad:], x.to(device)[:, pad:])
    assert _rel(got, dy[:, pad:].double().T @ x[:, pad:].double()) < _tol(rows)


@pytest.mark.parametrize("rows", [8191, 8192])  # torch's layer, the kernels
def test_linear_gradients(rows, device):
    from maloq_amd.linear import linear
    gen = torch.Generator().manual_seed(rows)
    x, w, b, g, h = (torch.randn(*s, generator=gen) for s in ((rows, 24), (36, 24), (36,), (rows, 36), (36, 24)))
    leaves = [t.to(device).requires_grad_() for t in (x, w, b)]
    y = linear(*leaves)
    gx, gw, gb = torch.autograd.grad(y, leaves, g.to(device), retain_graph=True)
    assert torch.equal(y, torch.nn.functional.linear(*leaves))
    g64, x64 = g.double(), x.double()
    assert _rel(gx, g64 @ w.double()) < _tol(36)
    assert _rel(gw, g64.T @ x64) < _tol(rows)
    assert _rel(gb, g64.sum(0)) < _tol(rows)
    # a gradient of a gradient: of <w's gradient, h> with respect to x
    gw2, = torch.autograd.grad(y, leaves[1:2], g.to(device), create_graph=True)
    gxx, = torch.autograd.grad((gw2 * h.to(device)).sum(), leaves[0])
    assert _rel(gxx, g64 @ h.double()) < _tol(36)
