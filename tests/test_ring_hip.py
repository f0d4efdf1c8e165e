"""The bf16 message GEMM that shares its weights through LDS (gated mmax = lmax = 4
forwards whose grid is more than one round), against 64 bits and beside the direct
kernel at the same shapes; and bit for bit against the direct kernel, which takes the
same edges in grids of less than one round.

Tolerance: the rows are rounded to bf16 once (2^-9 of each at most, half of that
rms); products and sums are fp32.  Twice the larger figure, relative 2-norm.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


# K loops of 1, 2, 3, 5, 8 and 16 steps: phases of up to 4 steps, cut and whole; edge
# counts with a last pair of tiles that is whole, half empty or cut, and one round less.
@pytest.mark.parametrize("c_in", [16, 32, 48, 80, 128, 256])
@pytest.mark.parametrize("E", [1000, 8192 + 1, 8192 + 32 + 5, 8192 + 64])
def test_gated_forward(E, c_in, device):
    from test_message_hip import _run
    _, got, ref = _run(4, 4, torch.bfloat16, True, True, N=E // 20, E=E, c_in=c_in, c_out=32, seed=c_in + E,
                       device=device)
    assert ((got - ref).norm() / ref.norm()).item() < 2.0 ** -8


# Three channel blocks; 97 tiles (a grid of 312 workgroups) with a last pair that is half
# empty and a last tile of 5 edges, against 32 tiles at a time (96 workgroups).  Nodes
# own 8 consecutive edges, so that no node's sum crosses a tile.
@pytest.mark.parametrize("c", [32, 96])
@pytest.mark.parametrize("two_convolutions", [False, True])
def test_bits_of_the_direct_kernel(two_convolutions, c, device):
    from maloq_amd import message as M
    from maloq_amd.wigner import extract_euler_angles
    from test_message_hip import _conv
    L, H, E, chunk = 4, 96, 97 * 32 - 27, 32 * 32
    gen = torch.Generator().manual_seed(c + two_convolutions)
    N = -(-E // 8)
    ei = torch.stack([torch.randint(0, N, (E,), generator=gen), torch.arange(E) // 8]).to(device)
    x = torch.randn(N, (L + 1) ** 2, c, generator=gen).to(device, torch.bfloat16)
    eul = extract_euler_angles(torch.randn(E, 3, generator=gen).to(device), seed=1)
    parts = 2 if two_convolutions else 1
    rad = (torch.rand(E, M.rad_width(L, L, parts * c), generator=gen) + 0.5).to(device)
    convs = [_conv(L, L, parts * c, H, gen, True), _conv(L, L, H, c, gen, False)]
    convs = [(k["w0"].to(device).float(), k["b0"].to(device).float(), [w.to(device).float() for w in k["wm"]])
             for k in convs]

    def forward(a, b):
        plan = M.MessagePlan(ei[:, a:b], N)
        args = (x, plan, plan.sort_edges(eul[a:b]), plan.sort_edges(rad[a:b]))
        if two_convolutions:
            return M.edgewise_forward(*args, *convs, L, L)
        return M.message_forward(*args, *convs[0], L, L, gate=True)

    whole = forward(0, E)
    for a in range(0, E, chunk):
        b = min(E, a + chunk)
        nodes = slice(a // 8, -(-b // 8))
        assert torch.equal(whole[nodes], forward(a, b)[nodes])
