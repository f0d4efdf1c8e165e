"""fp32 kernels on the bf16 matrix cores (three bf16 planes per float, six
products), at the edges of their tiles, against 64 bits.

Tolerance: each product's error is below 2^-23 of it (the dropped planes and
the roundings inside a matrix instruction), and a sum of n products, added 16 at
a time, six times over, in fp32, rounds about n 6 / 16 times at 2^-25 (rms) of a
partial sum: sqrt(3 n / 8) 2^-25 of the result for random signs.  The bound is
four times the two together, as a relative 2-norm.
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _tol(n):
    return 4 * (2.0 ** -23 + math.sqrt(3 * n / 8) * 2.0 ** -25)


def _rel(got, ref):
    return ((got.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("E", [1, 15, 16, 17, 33, 700])
@pytest.mark.parametrize("lmax,mmax,c_in,c_out,gate,splits", [
    (2, 2, 32, 32, False, 1),     # one partly filled tile per group
    (4, 2, 128, 96, True, 2),     # remainders of 256 columns in both operands, gate group
    (4, 4, 96, 128, False, 3),    # last split empty or short
])
def test_weight_gradient(lmax, mmax, c_in, c_out, gate, splits, E, device):
    from maloq_amd import message as M
    gen = torch.Generator().manual_seed(E + lmax)
    kept = M.kept_rows(lmax, mmax)
    rows = kept + (lmax if gate else 0)
    # values over several binades; rows past E must not count
    dz = torch.randn(E + 3, rows, c_out, generator=gen) * torch.exp2(torch.randint(-6, 6, (E + 3, 1, 1), generator=gen))
    y = torch.randn(E + 3, kept, c_in, generator=gen)
    dw0, dwm, _ = M.message_weight_grad(dz.to(device), y.to(device), lmax, mmax, c_out, c_in, splits=splits,
                                        num_edges=E, gate=gate)
    z, x = dz[:E].double(), y[:E].double()
    n0 = lmax + 1
    ref0 = z[:, :n0].reshape(E, -1).T @ x[:, :n0].reshape(E, -1)
    if gate:
        ref0 = torch.cat([z[:, kept:].reshape(E, -1).T @ x[:, :n0].reshape(E, -1), ref0])
    assert _rel(dw0.cpu(), ref0) < _tol(E)
    at = n0
    for m in range(1, mmax + 1):
        k = lmax - m + 1
        zp, zm = (z[:, at + s * k:at + (s + 1) * k].reshape(E, -1) for s in (0, 1))
        xp, xm = (x[:, at + s * k:at + (s + 1) * k].reshape(E, -1) for s in (0, 1))
        ref = torch.cat([zp.T @ xp + zm.T @ xm, zm.T @ xp - zp.T @ xm])
        assert _rel(dwm[m - 1].cpu(), ref) < _tol(2 * E)
        at += 2 * k
