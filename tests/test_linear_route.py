"""Which gradients of maloq_amd.linear go to this package's kernels, with these replaced
by recorders: plain ones do; batched and twice differentiable ones are torch's.  And the
row strides that the weight gradient's kernel is given."""
import types

import pytest
import torch

from maloq_amd import _lib
from maloq_amd import linear as lin


@pytest.fixture
def layer(monkeypatch):
    calls = []

    def weight_grad(dy, x):
        calls.append("weight")
        return dy.t() @ x

    def total(dy):
        calls.append("bias")
        return dy.sum(0)

    monkeypatch.setattr(lin, "rows_weight_grad", weight_grad)
    monkeypatch.setattr(lin, "rows_sum", total)
    gen = torch.Generator().manual_seed(0)
    leaves = [torch.randn(*s, generator=gen).requires_grad_() for s in ((9, 5), (3, 5), (3,))]
    return calls, leaves, lin._RowsLinear.apply(*leaves), torch.nn.functional.linear(*leaves)


def test_plain_gradients_use_the_kernels(layer):
    calls, leaves, y, ref = layer
    g = torch.randn(y.shape)
    for a, b in zip(torch.autograd.grad(y, leaves, g), torch.autograd.grad(ref, leaves, g)):
        torch.testing.assert_close(a, b)
    assert calls == ["weight", "bias"]


def test_batched_gradients(layer):
    calls, leaves, y, ref = layer
    g = torch.randn(4, *y.shape)
    got = torch.autograd.grad(y, leaves, g, is_grads_batched=True, retain_graph=True)
    mapped = torch.func.vmap(lambda v: torch.autograd.grad(y, leaves, v, retain_graph=True))(g)
    want = torch.autograd.grad(ref, leaves, g, is_grads_batched=True)
    for a, b, c in zip(got, mapped, want):
        torch.testing.assert_close(a, c)
        torch.testing.assert_close(b, c)
    assert calls == []


def test_gradients_of_gradients(layer):
    calls, leaves, y, ref = layer
    g = torch.randn(y.shape)
    twice = lambda out: torch.autograd.grad(
        sum(t.square().sum() for t in torch.autograd.grad(out, leaves[:2], g, create_graph=True)), leaves[:2])
    for a, b in zip(twice(y), twice(ref)):
        torch.testing.assert_close(a, b)
    assert calls == []


@pytest.mark.parametrize("make,ld", [
    (lambda n: torch.randn(5, n), "n"),
    (lambda n: torch.randn(5, n + 3)[:, 2:2 + n], "n + 3"),
    (lambda n: torch.randn(n, 5).t(), "n"),                # a copy
    (lambda n: torch.randn(1, n).expand(5, n), "n"),       # a copy
    (lambda n: torch.randn(n, 1).t(), "n"),                # one row, of stride 1
    (lambda n: torch.randn(4, n)[::4], "n"),               # one row, of stride 4 n
    (lambda n: torch.randn(0, n), "n"),
])
@pytest.mark.parametrize("n", [1, 7])
def test_row_strides(monkeypatch, make, ld, n):
    seen = []
    monkeypatch.setattr(_lib, "call", lambda name, *args: seen.append(args))
    monkeypatch.setattr(_lib, "load", lambda: types.SimpleNamespace(maloq_rows_dw_partials_floats=lambda *a: 4))
    monkeypatch.setattr(_lib, "stream_of", lambda device: 0)
    dy = make(n)
    lin.rows_weight_grad(dy, torch.randn(dy.shape[0], 3))
    (got, stride, cols, _, ld_x, k, rows, *_), = seen
    assert (stride, cols, ld_x, k, rows) == (eval(ld), n, 3, 3, dy.shape[0])
    flat = torch.as_strided(got, (rows, n), (stride, 1))  # as the kernel steps through it
    assert torch.equal(flat, dy)
