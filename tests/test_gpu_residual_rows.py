"""The gated residual with norm and token shift of the hybrid decoder's prompts at the sizes where its launch changes: one, two and four rows
a thread, four and eight columns, sequences that begin anywhere in a workgroup's rows.  Tolerances as in the tests of the step itself."""
import pytest
import torch

from msa_amd import seq_ops
from oracle import recurrent_layers as R
from seq_helpers import BF16, F32, Rand, batch, close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,counts", [(1024, [700, 1, 835]), (1024, [1, 2, 1534]), (1024, [1000, 5, 2066]), (1024, [3, 1, 2500, 569]), (1028, [1500, 1552]),
                                      (2570, [2, 700, 900]), (1031, [3060, 3]), (136, [23000, 6, 100])])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_shift(dtype, W, counts):
    r = Rand(W)
    slots = list(range(len(counts)))[::-1]
    T = sum(counts)
    (x, x_), (y, y_), (g, g_) = r(T, W), r(T, W, dtype=dtype), r(T, W + 8, dtype=dtype)
    (gb, gb_), (w, w_), (b, b_), (sh, sh_) = r(W), r(W), r(W), r(W)
    prev, prev_ = r(len(counts) + 1, W)
    norm = seq_ops.DynTanhNorm(w, b, 0.7)
    xo, h, hs = seq_ops.residual_norm(x, batch(counts, slots), dtype, y, g[:, 8:], gb, norm, sh, prev)
    want_x = x_ + R.sigmoid(g_[:, 8:] + gb_) * y_
    want_h = R.dyn_tanh(want_x, 0.7, w_, b_)
    close(xo, want_x, F32)
    close(h, want_h, dtype)
    at = 0
    for c, s in zip(counts, slots):
        close(hs[at:at + c], R.token_shift(want_h[at:at + c], sh_, prev_[s]), dtype)
        prev_[s] = want_h[at + c - 1]
        at += c
    close(prev, prev_, F32)
    x1, h1, none = seq_ops.residual_norm(x, batch(counts, slots), dtype, y, g[:, 8:], gb, norm)      # without the shift: one row a thread
    assert none is None and torch.equal(x1, xo) and torch.equal(h1, h)
