"""Which gradients of maloq_amd.linear go to this package's kernels, with these replaced
by recorders: plain ones do; batched and twice differentiable ones are torch's."""
import pytest
import torch

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
