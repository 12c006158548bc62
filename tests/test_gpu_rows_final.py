"""Products of decode rows that form their operand on the way: the head's, behind the last residual step and the norm behind that, and
the first layer's, the rows of an embedding table."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(1, 1024, 151936), (8, 1024, 6000), (9, 1024, 6000), (1, 520, 40000), (7, 1032, 20011), (3, 2048, 6200), (4, 2048, 6200),
                                   (2, 3072, 4100), (1, 3080, 4100), (2, 2560, 64), (16, 512, 6000)])
def test_final_operand(M, K, N):
    """Against 64-bit sums.  The operand is the bf16 rounding of values that carry the fp32 rounding of two sums of K squares (1e-6 of
    a value): one bf16 step of the few values that lie so near the middle of two, and 2^-24 K sum |w h| bounds the fp32 sums.  (9, 1024), (7, 1032), (4, 2048), (1, 3080), (2, 2560, 64) and (16, 512) take the separate launch."""
    from msa_amd import seq_ops
    g = torch.Generator().manual_seed(K + N)
    x, wide = (3 * torch.randn((M, K), generator=g)).cuda(), torch.randn((M, K + 8), generator=g).bfloat16().cuda()
    y, w, nw = wide[:, :K], (1 + 0.1 * torch.randn(K, generator=g)).cuda(), (1 + 0.1 * torch.randn(K, generator=g)).cuda()
    head, add = (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16().cuda(), torch.randn(N, generator=g).cuda()
    x0, flush = x.clone(), torch.empty(1 << 26, device="cuda")
    norm = lambda v: v / torch.sqrt((v ** 2).mean(1, keepdim=True) + 1e-5)
    h = norm(x.double() + norm(y.double()) * w.double()) * nw.double()
    hb, hd = h.bfloat16().double(), head.double()
    half = torch.ldexp(torch.ones_like(h), torch.frexp(h).exponent - 9)                     # of a bf16 step
    parts = 2 * half * ((h - hb).abs() >= half - 2e-6 * h.abs())                             # (may round to either neighbour)
    bound = (2 ** -24 * K * hb.abs() + parts) @ hd.abs().t() + 1e-6
    for i in range(3):
        flush.fill_(float(i))
        final = seq_ops.FinalRows(x, y, w, 1e-5, nw)
        got = seq_ops.rows_linear_f32(final, head, add=add).double() - add.double()
        assert ((got - hb @ hd.t()).abs() <= bound + 2 ** -23 * add.double().abs()).all()
        rows = final.rows()
        assert ((rows.double() - hb).abs() <= parts + 1e-9).all()
        assert torch.equal(x, x0)


@pytest.mark.parametrize("form", ["plain", "conv"])
@pytest.mark.parametrize("M,K,N", [(1, 1024, 3104), (16, 1024, 6000), (3, 520, 12000), (7, 2568, 2000), (15, 5120, 1000), (2, 5128, 1000), (4, 512, 6000),
                                   (2, 1024, 40)])
def test_embedded_operand(form, M, K, N):
    """The product is the one of the table's rows, bit for bit, and the rows in fp32 are exact; tokens from the table's end, its first and
    its last row.  (2, 5128), (4, 512) and (2, 1024, 40) take the separate launch."""
    from msa_amd import seq_ops
    g = torch.Generator().manual_seed(K + N)
    vocab = 1009
    table, m = torch.randn((vocab, K), generator=g).bfloat16().cuda(), (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16().cuda()
    table[5, 0] = float("inf")
    tokens = torch.randint(-vocab, vocab, (M,), generator=g)
    tokens[0], tokens[M // 2], tokens[-1] = 0, vocab - 1, -vocab if M % 2 else -1
    tokens = tokens.cuda()
    taps, state = torch.randn((N, 4), generator=g).cuda(), torch.randn((M + 2, 3, N), generator=g).cuda()
    slot = torch.arange(M, dtype=torch.int32).flip(0).cuda()
    s1, s2 = state.clone(), state.clone()
    product = lambda h, st: seq_ops.rows_linear(h, m) if form == "plain" else seq_ops.rows_conv(h, m, None, None, 0, taps, None, st, slot)
    rows = seq_ops.EmbedRows(table, tokens)
    got = product(rows, s1)
    assert torch.equal(rows.out, table[tokens].float())
    assert torch.equal(got, product(table[tokens], s2)) and torch.equal(s1, s2)


def test_final_operand_refuses_what_the_residual_step_refuses():
    from msa_amd import seq_ops
    x, y, w = torch.zeros((2, 1024), device="cuda"), torch.zeros((2, 1024), dtype=torch.bfloat16, device="cuda"), torch.ones(1024, device="cuda")
    for bad in ((x, y, w, 1e-5, w[:8]), (x, y.float(), w, 1e-5, w), (x.bfloat16(), y, w, 1e-5, w)):
        with pytest.raises(ValueError):
            seq_ops.FinalRows(*bad)
    head = torch.zeros((4096, 1024), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(Exception):
        seq_ops.rows_linear_f32(seq_ops.FinalRows(x.repeat(9, 1), y.repeat(9, 1), w, 1e-5, w), head)
    with pytest.raises(Exception):
        seq_ops.rows_linear(seq_ops.FinalRows(x, y, w, 1e-5, w), head)
