"""fp32 kernels on the bf16 matrix cores (three bf16 planes per float, six
products), at the edges of their tiles, against 64 bits.

Tolerance of a sum of n products: the planes left out are 2^-25.5 of a product
(rms; 2^-22 at most), which with the roundings inside a matrix instruction stays
below 2^-23; n products, added 16 at a time, six times over, in fp32, round about
n 6 / 16 times at 2^-25 (rms) of a partial sum: sqrt(3 n / 8) 2^-25 of the result for
random signs.  The bound is four times the two together, as a relative 2-norm.

Of a whole block (BLOCK): its longest sums here, 2 (lmax + 1) 128 products, give
6.5e-7 at lmax 4 and 7.7e-7 at lmax 6, the two rotations (sums of up to 13 products
with fp32 matrices) 2e-7 each, the gate's factors as much: 9e-7 together, and twice
that.  A third plane left out of one operand gives 6.9e-6 whatever the sizes.
"""
import math

import pytest
import torch

from oracle import message as omsg
from oracle import rotation as orot

pytestmark = pytest.mark.gpu


BLOCK = 2e-6


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


# Edge counts around the tiles (32 and 64 edges) of one group of waves, and large
# enough for two groups per workgroup (256 workgroups and more) with a last group
# that is empty or cut.
@pytest.mark.parametrize("lmax,mmax,gate,E", [
    (2, 2, False, 1), (4, 2, False, 63), (4, 2, False, 65), (4, 2, True, 33), (4, 4, False, 31), (4, 4, True, 33),
    (6, 2, True, 33), (6, 6, False, 33),
    (4, 2, False, 8192 + 1), (4, 2, False, 8192 + 65), (4, 4, True, 4096 + 1), (6, 2, True, 4096 + 40),
])
def test_block_forward_and_gradients(lmax, mmax, gate, E, device):
    from maloq_amd import message as M
    from maloq_amd.wigner import extract_euler_angles
    C = 128 if E > 4000 else 32
    N = max(2, E // 20)
    gen = torch.Generator().manual_seed(E + lmax + mmax)
    ei = torch.stack([torch.randint(0, N, (E,), generator=gen), torch.randint(0, N, (E,), generator=gen)])
    k0 = (lmax + 1) * C
    n0 = k0 + (lmax * C if gate else 0)
    w = [torch.randn(n0, k0, generator=gen) / math.sqrt(k0), torch.randn(n0, generator=gen) * 0.1]
    for m in range(1, mmax + 1):
        k = (lmax - m + 1) * C
        w.append(torch.randn(2 * k, k, generator=gen) / math.sqrt(2 * k))
    x = torch.randn(N, (lmax + 1) ** 2, C, generator=gen)
    rad = torch.rand(E, M.rad_width(lmax, mmax, C), generator=gen) + 0.5
    gout = torch.randn(N, (lmax + 1) ** 2, C, generator=gen)
    eul = extract_euler_angles(torch.randn(E, 3, generator=gen).to(device), seed=E)
    plan = M.MessagePlan(ei.to(device), N)
    dev = [t.to(device).requires_grad_() for t in (x, rad, *w)]
    out = M.message_block(dev[0], plan, plan.sort_edges(eul), plan.sort_edges(dev[1]), dev[2], dev[3], dev[4:], lmax,
                          mmax, gate=gate)
    grads = torch.autograd.grad(out, dev, gout.to(device))
    ref_in = [t.double().requires_grad_() for t in (x, rad, *w)]
    e64 = eul.cpu().double()
    ref = omsg.message_block(ref_in[0], ei, (e64[:, 0], e64[:, 1], e64[:, 2]), orot.load_jd(), lmax, mmax,
                             {"w0": ref_in[2], "b0": ref_in[3], "wm": ref_in[4:], "c_out": C}, rad=ref_in[1], gate=gate)
    ref_grads = torch.autograd.grad(ref, ref_in, gout.double())
    assert _rel(out.cpu(), ref.detach()) < BLOCK
    for got, want in zip(grads, ref_grads):
        assert _rel(got.cpu(), want) < BLOCK


# The two-convolution layer on a grid of two tiles a workgroup, three and two channel
# blocks: 32-edge tiles (the gated first convolution) and 64-edge ones (its own and the
# second's gradients), an odd number of each, the last of five edges.
@pytest.mark.parametrize("lmax,mmax", [(4, 2), (4, 4), (6, 2)])
@pytest.mark.parametrize("mode", ["node", "edge"])
def test_two_convolutions_many_edges(lmax, mmax, mode, device):
    from maloq_amd import message as M
    from maloq_amd.wigner import extract_euler_angles
    from test_message_hip import _conv
    E, N, C, H = 86 * 64 + 5, 270, 32, 96
    gen = torch.Generator().manual_seed(lmax + mmax)
    ei = torch.randint(0, N, (2, E), generator=gen)
    f = lambda conv: [conv["w0"].float(), conv["b0"].float(), *(w.float() for w in conv["wm"])]
    ts = [torch.randn(N, (lmax + 1) ** 2, C, generator=gen),
          torch.rand(E, M.rad_width(lmax, mmax, 2 * C), generator=gen) + 0.5,
          *f(_conv(lmax, mmax, 2 * C, H, gen, True)), *f(_conv(lmax, mmax, H, C, gen, False))]
    k = 2 + 2 + mmax  # where the second convolution's begin
    gout = torch.randn(N if mode == "node" else E, (lmax + 1) ** 2, C, generator=gen)
    eul = extract_euler_angles(torch.randn(E, 3, generator=gen).to(device), seed=E)
    plan = M.MessagePlan(ei.to(device), N)
    dev = [t.to(device).requires_grad_() for t in ts]
    out = M.edgewise_block(dev[0], plan, plan.sort_edges(eul), plan.sort_edges(dev[1]), (dev[2], dev[3], dev[4:k]),
                           (dev[k], dev[k + 1], dev[k + 2:]), lmax, mmax, node_or_edge=mode)
    grads = torch.autograd.grad(out, dev, gout.to(device))
    ref_in = [t.double().requires_grad_() for t in ts]
    e64 = eul.cpu().double()
    conv = lambda a, b, c_out: {"w0": ref_in[a], "b0": ref_in[a + 1], "wm": ref_in[a + 2:b], "c_out": c_out}
    ref = omsg.message_block(ref_in[0], ei, (e64[:, 0], e64[:, 1], e64[:, 2]), orot.load_jd(), lmax, mmax,
                             conv(2, k, H), rad=ref_in[1], conv2=conv(k, len(ts), C), gate=True,
                             concat="source-target", reduce=(mode == "node"))
    ref_grads = torch.autograd.grad(ref, ref_in, gout.double())
    for got, want in zip((out, *grads), (ref, *ref_grads)):  # two blocks' errors
        assert _rel(got.detach().cpu(), want.detach()) < 2 * BLOCK


# K loops whose last step is half (channels an odd number of 8s) or that the two
# groups of one tile cannot halve evenly; few edges and many (two tiles a workgroup).
@pytest.mark.parametrize("c_in", [8, 24, 40, 96, 104])
@pytest.mark.parametrize("lmax,mmax,E", [(2, 2, 50), (4, 2, 70), (4, 4, 70), (6, 2, 70), (4, 4, 8200)])
def test_block_input_channels(lmax, mmax, E, c_in, device):
    from test_message_hip import _run
    _, got, ref = _run(lmax, mmax, torch.float32, lmax == 4, True, N=max(8, E // 20), E=E, c_in=c_in, c_out=32,
                       seed=c_in, device=device)
    assert _rel(got, ref) < BLOCK


# An infinity in the node features, the output gradient or a weight: what it reaches is
# infinite, with the sign that a large number in its place gives, and the rest is finite.
# (A permutation graph: no sum meets two infinities.)
@pytest.mark.parametrize("where", ["x", "w0", "gout"])
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("lmax,mmax,E,C", [(4, 2, 70, 32), (6, 2, 70, 32), (6, 6, 70, 32), (4, 4, 2100, 128)])
def test_infinite_inputs(lmax, mmax, E, C, sign, where, device):
    from maloq_amd import message as M
    from maloq_amd.wigner import extract_euler_angles
    gen = torch.Generator().manual_seed(E + lmax)
    ei = torch.stack([torch.randperm(E, generator=gen), torch.arange(E)])
    k0 = (lmax + 1) * C
    ts = {"x": torch.randn(E, (lmax + 1) ** 2, C, generator=gen),
          "rad": torch.rand(E, M.rad_width(lmax, mmax, C), generator=gen) + 0.5,
          "w0": torch.randn(k0, k0, generator=gen) / math.sqrt(k0), "b0": torch.randn(k0, generator=gen) * 0.1}
    for m in range(1, mmax + 1):
        k = (lmax - m + 1) * C
        ts[f"w{m}"] = torch.randn(2 * k, k, generator=gen) / math.sqrt(2 * k)
    gout = torch.randn(E, (lmax + 1) ** 2, C, generator=gen)
    at = (5, 3) if where == "w0" else (7, 0, 3)
    eul = extract_euler_angles(torch.randn(E, 3, generator=gen).to(device), seed=E)
    plan = M.MessagePlan(ei.to(device), E)

    def leaves(value, cast):
        mine = {k: v.clone() for k, v in {**ts, "gout": gout}.items()}
        mine[where][at] = value
        g = cast(mine.pop("gout"))
        return [cast(t).requires_grad_() for t in mine.values()], g

    def results(out, ins, g):
        return out.detach(), *torch.autograd.grad(out, ins, g)

    dev, g = leaves(sign * math.inf, lambda t: t.to(device))
    got = results(M.message_block(dev[0], plan, plan.sort_edges(eul), plan.sort_edges(dev[1]), dev[2], dev[3], dev[4:],
                                  lmax, mmax), dev, g)
    ref_in, g = leaves(sign * 2.0 ** 100, torch.Tensor.double)
    e64 = eul.cpu().double()
    want = results(omsg.message_block(ref_in[0], ei, (e64[:, 0], e64[:, 1], e64[:, 2]), orot.load_jd(), lmax, mmax,
                                      {"w0": ref_in[2], "b0": ref_in[3], "wm": ref_in[4:], "c_out": C}, rad=ref_in[1]),
                   ref_in, g)
    for a, b in zip(got, want):
        a, large = a.cpu(), b.abs() > 2.0 ** 60
        assert torch.equal(a.isinf(), large) and torch.equal(a[large].sign(), b[large].sign().float())
        assert a[~large].isfinite().all()
    assert got[0].isinf().any() or where == "gout"


def test_infinite_rows_of_a_weight_gradient(device):
    from maloq_amd.linear import rows_weight_grad
    gen = torch.Generator().manual_seed(0)
    dy, x = torch.randn(300, 40, generator=gen), torch.randn(300, 33, generator=gen)
    dy[17, 3], x[201, 8], x[202, 9] = -math.inf, math.inf, math.nan
    dy[44, 5], x[44, 6] = math.inf, -math.inf
    dy[50, 0] = x[50, 0] = 1.1 * 2.0 ** 66  # finite; their product is not
    got = rows_weight_grad(dy.to(device), x.to(device)).cpu()
    want = (dy.double().T @ x.double()).float()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
