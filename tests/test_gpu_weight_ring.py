"""The ring form of the decode products (csrc/rows_ring.h) where its shares, units and ring can go wrong: rows that are no whole
units, more units than stay in registers, workgroups of a few rows and of many, both operands.  Sums are fp32 over K bf16 products
in another order than float64's: 2e-5 of the largest value, as for every fp32 product of these tests."""
import pytest
import torch

from msa_amd import ops, seq_ops
from oracle import delta_attention_layers as O
from oracle import recurrent_layers as R
from seq_helpers import BF16, F32, Rand, batch, close

pytestmark = pytest.mark.gpu
# rows: 3 and 4 a workgroup, 16 and 17, several rounds; K: one unit over a multiple of the wavefronts' 1024, one short, 5 x 1024 (the
# most that stays in registers), above it with an odd and an even number of rounds (some of the smaller matrices lie below the ring's
# line and cover the form beside it)
SHAPES = [(1, 1021, 2056), (16, 1100, 1528), (7, 4097, 1024), (16, 4360, 520), (2, 777, 5120), (3, 2600, 5128), (16, 300, 6152), (5, 4500, 7168), (1, 9000, 1016),
          (2, 2049, 2056), (16, 3000, 1528), (9, 14300, 520)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_plain_and_two_operands(M, N, K):
    assert N * K >= 3 << 19
    r = Rand(M + N)
    (x, x_), (y, y_), (w, w_), (add, add_) = r(M, K, dtype=BF16), r(M, K, dtype=BF16), r(N, K, dtype=BF16, scale=K ** -0.5), r(N)
    close(seq_ops.rows_linear_f32(x, w, add=add), x_ @ w_.T + add_, F32)
    n = N // 2 // 32 * 32
    got = seq_ops.rows_linear(x, w, x_b=y, n_b=n)
    close(got, torch.cat([x_ @ w_[:n].T, y_ @ w_[n:].T], 1), BF16, 4e-3)
    assert torch.equal(got, seq_ops.rows_linear(x, w, x_b=y, n_b=n))
    wide = torch.cat([x, y, y], 1)                       # a column range of wider rows
    close(seq_ops.rows_linear(wide[:, :K], w), x_ @ w_.T, BF16, 4e-3)


@pytest.mark.parametrize("N,K", [(1001, 1640), (1001, 3368), (3001, 1640)])
def test_not_finite_weights_stay_in_their_rows(N, K):
    """A row of infinities or NaN changes its own column only, also where a workgroup's last rows and a row's last units are empty."""
    r = Rand(3)
    (x, x_), (w, w_) = r(5, K, dtype=BF16), r(N, K, dtype=BF16, scale=K ** -0.5)
    for n, v in ((0, float("nan")), (499, float("inf")), (1000, float("nan"))):
        w[n, K - 8:] = v
    got = seq_ops.rows_linear_f32(x, w)
    bad = torch.tensor([0, 499, 1000])
    assert not torch.isfinite(got[:, bad.cuda()]).any()
    keep = torch.ones(N, dtype=torch.bool)
    keep[bad] = False
    close(got[:, keep.cuda()], (x_ @ w_.T)[:, keep], F32)


@pytest.mark.parametrize("M,ff,K", [(16, 901, 1032), (1, 4100, 1024), (9, 130, 6152), (16, 3101, 1032)])
def test_gated_units(M, ff, K):
    r = Rand(ff)
    (x, x_), (g, g_), (u, u_) = r(M, K, dtype=BF16), r(ff, K, dtype=BF16, scale=1.5 * K ** -0.5), r(ff, K, dtype=BF16, scale=1.5 * K ** -0.5)
    close(seq_ops.rows_glu(x, seq_ops.interleave_pairs(g, u), 1.5), O.clamped_glu(x_ @ g_.T, x_ @ u_.T, 1.5), BF16)


@pytest.mark.parametrize("M,N,K", [(16, 1100, 1536), (4, 600, 6144), (16, 2900, 1536)])
def test_residual(M, N, K):
    r = Rand(N)
    (x, x_), (w, w_), (g, g_) = r(M, K, dtype=BF16), r(N, K, dtype=BF16, scale=K ** -0.5), r(M, N + 16, dtype=BF16)
    (s, s_), (gb, gb_), (nw, nw_), (nb, nb_), (sh, sh_), (prev, prev_) = r(M, N), r(N), r(N), r(N), r(N), r(20, N)
    slot = torch.arange(19, 19 - M, -1, dtype=torch.int32, device="cuda")
    h, hs = seq_ops.rows_residual(x, w, s, g[:, 5:5 + N], gb, slot, seq_ops.DynTanhNorm(nw, nb, 0.9), sh, prev)
    want = s_ + R.sigmoid(g_[:, 5:5 + N] + gb_) * (x_ @ w_.T)
    wh = R.dyn_tanh(want, 0.9, nw_, nb_)
    at = slot.cpu().long()
    close(s, want, F32)
    close(h, wh, BF16, 4e-3)
    close(hs, wh + (prev_[at] - wh) * sh_, BF16, 4e-3)
    prev_[at] = wh
    close(prev, prev_, F32)


@pytest.mark.parametrize("W", [1104, 2064])
@pytest.mark.parametrize("taps_n", [1, 4, 5])
def test_convolution(taps_n, W):
    r = Rand(taps_n)
    lo, C, n_b, rows = 40, 1500, 1600, 333
    (w, _), (taps, _), (b, _) = r(n_b + rows, W, dtype=BF16, scale=1.6 * W ** -0.5), r(C, taps_n), r(C)
    s1, s2 = torch.zeros(4, taps_n - 1, C, device="cuda"), torch.zeros(4, taps_n - 1, C, device="cuda")
    for step in range(6):
        (x, _), (y, _) = r(3, W, dtype=BF16), r(3, W, dtype=BF16)
        slot = torch.tensor([2, 0, 3], dtype=torch.int32, device="cuda")
        out = seq_ops.rows_conv(x, w, y, n_b, lo, taps, b, s1, slot)
        plain = seq_ops.rows_linear(x, w, x_b=y, n_b=n_b)
        conv = seq_ops.conv_silu(plain[:, lo:lo + C], taps, b, s2, batch([1, 1, 1], [2, 0, 3]))
        assert torch.equal(out[:, :lo], plain[:, :lo]) and torch.equal(out[:, lo + C:], plain[:, lo + C:])
        close(out[:, lo:lo + C], conv, BF16)
    if taps_n > 1:
        close(s1, s2, BF16, 4e-3)
        assert torch.all(s1[1] == 0)


@pytest.mark.parametrize("n,W,more", [(1401, 1544, 1500), (4500, 640, 7)])
def test_recurrence(n, W, more):
    assert (3 * n + more) * W >= 8 << 20
    r = Rand(n)
    (wz, _), (wu, _), (wg, _), (wr, _) = (r(m, W, dtype=BF16, scale=2 * W ** -0.5) for m in (n, n, n, more))
    w = torch.cat([seq_ops.interleave_gru(wz, wu, wg), wr]).contiguous()
    n_b = w.shape[0] - more
    (zb, _), (ub, _) = r(n), r(n)
    s1, s2 = torch.zeros(3, n, device="cuda"), torch.zeros(3, n, device="cuda")
    for step in range(3):
        (x, _), (y, _) = r(2, W, dtype=BF16), r(2, W, dtype=BF16)
        slot = torch.tensor([2, 0], dtype=torch.int32, device="cuda")
        act, out = seq_ops.rows_gru(x, w, y, n, zb, ub, s1, slot)
        plain = seq_ops.rows_linear(x, w, x_b=y, n_b=n_b)
        close(act, seq_ops.min_gru(plain[:, :n_b], zb, ub, n, s2, batch([1, 1], [2, 0])), BF16, 2e-2)
        close(out[:, n_b:], plain[:, n_b:], BF16)
    close(s1, s2, BF16)
    assert torch.all(s1[1] == 0)


@pytest.mark.parametrize("M,N,K", [(16, 1600, 5120), (3, 336, 5120), (8, 2560, 9728), (1, 6160, 640), (16, 2576, 1152), (1, 1040, 7296), (8, 176, 14336),
                                   (5, 512, 8192), (3, 1040, 5120), (1, 14000, 640), (16, 9600, 1152),
                                   (12, 6144, 5248), (11, 8176, 5248), (16, 8192, 5248)])
def test_skinny_linear(M, N, K):
    """Folded norm, silu-mul of whole 16-row groups, residual; (1, 1040, 7296) to (5, 512, 8192) cut
    K over workgroups."""
    r = Rand(N + K)
    (x, x_), (w, w_), (nw, nw_), (res, res_) = r(M, K, dtype=BF16, scale=3.0), r(N, K, dtype=BF16, scale=K ** -0.5), r(K, dtype=BF16, scale=0.1, add=1.0), r(M, N, dtype=BF16)
    close(ops.skinny_linear(x, w, residual=res), (x_ @ w_.T) + res_, BF16, 1e-2)
    normed = R.rms(x_, 1e-6) * nw_
    if K <= 5120:
        close(ops.skinny_linear(x, w, norm_weight=nw), normed @ w_.T, BF16, 1e-2)
    gate, up = w[:N // 2], w[N // 2:]
    wi = ops.interleave_gate_up(gate, up)
    a, b = (x_ @ w_[:N // 2].T), (x_ @ w_[N // 2:].T)
    close(ops.skinny_linear(x, wi, silu_mul=True), R.silu(a) * b, BF16, 1.5e-2)
