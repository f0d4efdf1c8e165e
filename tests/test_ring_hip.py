"""The bf16 message GEMM that shares its weights through LDS (gated mmax = lmax = 4
forwards whose grid is more than one round), against 64 bits and beside the direct
kernel at the same shapes.

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
