"""Single products of the fp32 routing on the bf16 matrix cores (values in three parts), where no sum over many of them hides an error."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def scores(kr, q, scale):
    """``q [B, 8, 128]`` as queries of one token whose group sums are exact: one head of each group is not zero."""
    from msa_amd import ops
    C, B = kr.shape[0], q.shape[0]
    bank = ops.Bank(1, list(range(C + 1)), list(range(C)), 8, 128, torch.float32)
    bank.set_layer(0, kr.cuda(), None, None)
    full = torch.zeros((B, 1, 8, 4, 128))
    full[:, 0, :, 1] = q
    return ops.chunk_scores(bank, 0, full.view(B, 1, 32, 128).cuda(), None, "scaled_dot", scale).cpu().double()


@pytest.mark.parametrize("C,B,size", [(2000, 4, 1.0), (8000, 2, 1.0), (8191, 1, -1.0), (300, 1, 2.0**60), (3300, 6, 2.0**-40)])
def test_keys_of_one_component(C, B, size):
    """What is left out is below 2^-24 of a product, and its sum is rounded once (2^-24): among the values are those furthest from bf16 ones,
    halfway between them and just beside that."""
    g = torch.Generator().manual_seed(C)
    hard = torch.tensor([0x3f80ff7f, 0x3f807fff, 0x3f808000, 0x3f808001, 0x3f817f80, 0x3f80ffff, 0x3f800001, 0x3fffffff, 0x3f818181], dtype=torch.int32).view(torch.float32)
    pick = lambda *s: torch.where(torch.rand(s, generator=g) < 0.5, hard[torch.randint(0, len(hard), s, generator=g)], 1 + torch.rand(s, generator=g))
    at, val = torch.randint(0, 1024, (C,), generator=g), pick(C) * size
    kr = torch.zeros((C, 1024))
    kr[torch.arange(C), at] = val
    q = pick(B, 1024)
    got = scores(kr.view(C, 8, 128), q.view(B, 8, 128), 32.0)              # (scores are a 32nd of the sum over heads)
    want = q.double()[:, at] * val.double()
    assert ((got - want) / want).abs().max().item() <= 2.0**-23


def test_values_that_round_to_infinity():
    """The largest floats are above the largest bf16 value: queries are cut off there, and keys formed again value by value."""
    big = torch.finfo(torch.float32).max
    kr, q = torch.zeros((64, 8, 128)), torch.zeros((2, 8, 128))
    kr[5, 1, 7], kr[6, 1, 7], kr[7, 0, 0], q[0, 1, 7], q[1, 0, 0] = big, -big, 0.25, 0.5, big
    got = scores(kr, q, 32.0)
    want = torch.zeros((2, 64), dtype=torch.float64)
    want[0, 5], want[0, 6], want[1, 7] = 0.5 * big, -0.5 * big, 0.25 * big
    assert ((got - want).abs() <= 2.0**-23 * want.abs()).all()


def test_keys_that_are_not_gaussian():
    """A few large components among small ones, of either sign, as trained keys have them: 1e-6 of the largest score, as for Gaussian ones."""
    g = torch.Generator().manual_seed(3)
    kr, q = (torch.randn(s, generator=g).sign() * torch.exp(3 * torch.randn(s, generator=g)) for s in ((2000, 8, 128), (3, 8, 128)))
    got, want = scores(kr, q, 32.0), q.double().view(3, -1) @ kr.double().view(2000, -1).t()
    assert (got - want).abs().max() <= 1e-6 * want.abs().max()
