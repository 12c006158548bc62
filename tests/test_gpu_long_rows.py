"""Decode products of rows longer than a workgroup's registers hold (over 5120 elements), whose activations pass the weights' ring
(csrc/rows_ring.h), and the line to the form that cuts K over workgroups (csrc/linear.hip).  fp32 sums in another order than float64's:
2e-5 of the largest value; bf16 outputs one rounding."""
import pytest
import torch

from msa_amd import ops, seq_ops
from seq_helpers import BF16, F32, Rand, close

pytestmark = pytest.mark.gpu


# K: one vector over 5 x 1024, no whole units with an odd and an even number of rounds, whole ones; N: workgroups of 4 rows, of 17 (two
# blocks that take turns in the plane of sums) and of 50 in equal and unequal shares; all counts of activations at the edges of the loads
@pytest.mark.parametrize("M,N,K", [(1, 1030, 5128), (8, 1030, 5128), (9, 4300, 5128), (16, 4300, 7176), (15, 12801, 5640), (2, 2560, 10248), (16, 8192, 6144), (7, 255, 9728)])
def test_products(M, N, K):
    r = Rand(N + K)
    (x, x_), (y, y_), (w, w_) = r(M, K, dtype=BF16), r(M, K, dtype=BF16), r(N, K, dtype=BF16, scale=K ** -0.5)
    got = seq_ops.rows_linear_f32(x, w)
    close(got, x_ @ w_.T, F32)
    assert torch.equal(got, seq_ops.rows_linear_f32(x, w))
    wide = torch.full((M, K + 24), float("nan"), device="cuda", dtype=BF16)      # rows apart: what lies between them is not read
    wide[:, 8:8 + K] = x
    assert torch.equal(seq_ops.rows_linear_f32(wide[:, 8:8 + K], w), got)
    n = N // 2 // 32 * 32
    close(seq_ops.rows_linear(x, w, x_b=y, n_b=n), torch.cat([x_ @ w_[:n].T, y_ @ w_[n:].T], 1), BF16, 4e-3)


# either side of the line: few rows of weights, 14 and 15 rows of activations, matrices above and below the ring's line
@pytest.mark.parametrize("N,K", [(1024, 7168), (1024, 7296), (768, 5376), (2048, 6144), (2560, 9728), (2064, 5376)])
@pytest.mark.parametrize("M", [8, 9, 14, 15, 16])
def test_residual_beside_the_cut_form(M, N, K):
    r = Rand(M + N)
    (x, x_), (w, w_), (res, res_) = r(M, K, dtype=BF16), r(N, K, dtype=BF16, scale=K ** -0.5), r(M, N, dtype=BF16)
    close(ops.skinny_linear(x, w, residual=res), (x_ @ w_.T) + res_, BF16, 1e-2)
    close(ops.skinny_linear(x, w), x_ @ w_.T, BF16, 4e-3)
