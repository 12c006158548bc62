"""Products of decode rows that form their operand x + rms_norm(y) * w on the way, against the launches of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(M, K, seed):
    g = torch.Generator().manual_seed(seed)
    x = (3 * torch.randn((M, K), generator=g)).cuda()
    wide = torch.randn((M, K + 8), generator=g).bfloat16().cuda()
    return x, wide[:, :K], (1 + 0.1 * torch.randn(K, generator=g)).cuda(), g


@pytest.mark.parametrize("form", ["plain", "glu", "conv"])
@pytest.mark.parametrize("M,K,N", [(1, 520, 4096), (15, 520, 4096), (3, 1024, 2000), (7, 1032, 1600), (4, 2048, 800), (2, 2560, 6144), (2, 3072, 4100),
                                   (16, 2560, 4096), (4, 3080, 1024), (5, 512, 4096), (1, 1024, 64), (1, 520, 11000), (15, 520, 11000), (3, 1024, 3100),
                                   (5, 1032, 12200), (7, 1032, 12200), (3, 2048, 6200), (2, 2560, 4900)])
def test_post_operand(form, M, K, N):
    """The sum to the rounding of fp32 sums of K squares (1e-6 of the largest value); the product is the one of that sum's bf16 rows,
    bit for bit.  The first five, (16, 2560, 4096) to (1, 1024, 64) and (7, 1032, 12200) take the separate launch: too few weights, too
    many elements, too long, too short."""
    from msa_amd import seq_ops
    x, y, w, g = operands(M, K, K + N)
    m = (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16().cuda()
    taps, state = torch.randn((N, 4), generator=g).cuda(), torch.randn((M + 2, 3, N), generator=g).cuda()
    slot = torch.arange(M, dtype=torch.int32).flip(0).cuda()

    def product(h, st):
        if form == "plain":
            return seq_ops.rows_linear(h, m)
        if form == "glu":
            return seq_ops.rows_glu(h, m, 7.0)
        return seq_ops.rows_conv(h, m, None, None, 0, taps, None, st, slot)
    x0, s1, s2 = x.clone(), state.clone(), state.clone()
    post = seq_ops.PostRows(x, y, w, 1e-5)
    got = product(post, s1)
    yd = y.double()
    want = x.double() + yd / torch.sqrt((yd ** 2).mean(1, keepdim=True) + 1e-5) * w.double()
    assert torch.equal(x, x0)
    assert (post.out.double() - want).abs().max() <= 1e-6 * want.abs().max()
    assert torch.equal(got, product(post.out.bfloat16(), s2)) and torch.equal(s1, s2)


@pytest.mark.parametrize("form", ["plain", "glu", "conv"])
@pytest.mark.parametrize("M,K,N", [(1, 1024, 4096), (3, 2048, 6200), (1, 3072, 6144)])
def test_post_operand_with_cold_weights(form, M, K, N):
    """The norm's weights come from memory (a gigabyte has been written since they were), the sublayer's output from a near cache:
    the product is again the one of the sum's bf16 rows, bit for bit, from every workgroup."""
    from msa_amd import seq_ops
    x, y, w, g = operands(M, K, K + N)
    m = (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16().cuda()
    taps, state = torch.randn((N, 4), generator=g).cuda(), torch.zeros((M, 3, N), device="cuda")
    slot = torch.arange(M, dtype=torch.int32).cuda()
    product = {"plain": lambda h: seq_ops.rows_linear(h, m), "glu": lambda h: seq_ops.rows_glu(h, m, 7.0),
               "conv": lambda h: seq_ops.rows_conv(h, m, None, None, 0, taps, None, state.clone(), slot)}[form]
    flush = torch.empty(1 << 28, device="cuda")
    for i in range(4):
        flush.fill_(float(i))
        x.mul_(1.0), y.mul_(1.0)
        post = seq_ops.PostRows(x, y, w, 1e-5)
        got = product(post)
        assert torch.equal(got, product(post.out.bfloat16())), i


def test_post_operand_refuses_what_the_residual_step_refuses():
    from msa_amd import seq_ops
    x, y, w, _ = operands(2, 1024, 1)
    for bad in ((x.bfloat16(), y, w), (x, y.float(), w), (x, y[:1], w), (x, y, w[:8])):
        with pytest.raises(ValueError):
            seq_ops.PostRows(*bad, 1e-5)
    with pytest.raises(Exception):
        seq_ops.rows_linear(seq_ops.PostRows(x.repeat(9, 1), y.repeat(9, 1), w, 1e-5), torch.zeros((2048, 1024), dtype=torch.bfloat16, device="cuda"))
