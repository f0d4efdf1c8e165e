"""The linear layer of maloq_amd.linear beside torch's, for every kind of gradient that
a caller may ask of it: plain, batched and twice differentiable ones; and the row
strides that the weight gradient's kernel meets."""
import pytest
import torch

from maloq_amd import ops


def _layers(device, rows, needs=(True, True, True), bias=True):
    gen = torch.Generator().manual_seed(0)
    leaves = [torch.randn(*s, generator=gen).to(device).requires_grad_(n)
              for s, n in zip(((rows, 8), (4, 8), (4,)), needs)]
    args = leaves if bias else [*leaves[:2], None]
    wanted = [t for t in args if t is not None and t.requires_grad]
    return wanted, ops.rows_linear(*args), torch.nn.functional.linear(*args)


def _close(got, want, rows):
    # sums of `rows` products in fp32, in other orders
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=2.0 ** -22 * rows ** 0.5 * 8)


DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("needs", [(True, True, True), (False, True, True), (True, False, True), (True, True, False)])
def test_plain_gradients(device, needs, bias):
    wanted, y, ref = _layers(device, 300, needs, bias)
    g = torch.randn_like(y)
    assert torch.equal(y, ref)
    _close(torch.autograd.grad(y, wanted, g), torch.autograd.grad(ref, wanted, g), 300)


@pytest.mark.parametrize("device", DEVICES)
def test_batched_gradients(device):
    wanted, y, ref = _layers(device, 300)
    g = torch.randn(3, *y.shape, device=device)
    got = torch.autograd.grad(y, wanted, g, is_grads_batched=True, retain_graph=True)
    mapped = torch.func.vmap(lambda v: torch.autograd.grad(y, wanted, v, retain_graph=True))(g)
    want = torch.autograd.grad(ref, wanted, g, is_grads_batched=True)
    _close(got, want, 300)
    _close(mapped, want, 300)


@pytest.mark.parametrize("device", DEVICES)
def test_gradients_of_gradients(device):
    wanted, y, ref = _layers(device, 300)
    g = torch.randn_like(y)
    twice = lambda out: torch.autograd.grad(
        sum((t * t.detach().sign()).sum() for t in torch.autograd.grad(out, wanted[:2], g, create_graph=True)),
        wanted[:2])
    _close(twice(y), twice(ref), 300)


@pytest.mark.gpu
@pytest.mark.parametrize("make", [
    lambda n: torch.randn(5, n, device="cuda"),
    lambda n: torch.randn(5, n + 3, device="cuda")[:, 2:2 + n],
    lambda n: torch.randn(n, 5, device="cuda").t(),              # a copy
    lambda n: torch.randn(1, n, device="cuda").expand(5, n),     # a copy
    lambda n: torch.randn(n, 1, device="cuda").t(),              # one row, of stride 1
    lambda n: torch.randn(4, n, device="cuda")[::4],             # one row, of stride 4 n
    lambda n: torch.randn(0, n, device="cuda"),
])
@pytest.mark.parametrize("n", [1, 7])
def test_row_strides(make, n, device):
    from maloq_amd.linear import rows_weight_grad
    dy = make(n)
    x = torch.randn(dy.shape[0], 3, device=device)
    torch.testing.assert_close(rows_weight_grad(dy, x).cpu(), (dy.cpu().double().t() @ x.cpu().double()).float())
