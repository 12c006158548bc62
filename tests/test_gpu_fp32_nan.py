"""fp32 routing sums that are formed again value by value: NaN and infinities in chunks and query rows of every wavefront, both of its halves and
several blocks, against float64 with a maximum that ignores NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,B,S,share", [(300, 3, 70, 0.02), (33, 1, 64, 0.3), (2000, 2, 128, 0.001), (64, 2, 32, 1.0), (8191, 1, 256, 0.0005)])
def test_scores(C, B, S, share):
    from msa_amd import ops
    g = torch.Generator().manual_seed(C + S)
    kr, q = torch.randn((C, 1024), generator=g), torch.randn((B * S, 1024), generator=g)
    for t in (kr, q):
        for value in (float("nan"), float("inf"), -float("inf")):
            rows = torch.nonzero(torch.rand(t.shape[0], generator=g) < share).flatten()
            t[rows, torch.randint(0, 1024, (len(rows),), generator=g)] = value
    full = torch.zeros((B, S, 8, 4, 128))
    full[..., 2, :] = q.view(B, S, 8, 128)
    bank = ops.Bank(1, list(range(C + 1)), list(range(C)), 8, 128, torch.float32)
    bank.set_layer(0, kr.view(C, 8, 128).cuda(), None, None)
    got = ops.chunk_scores(bank, 0, full.view(B, S, 32, 128).cuda(), None, "scaled_dot", 32.0).cpu().double()
    want = (q.double() @ kr.double().t()).view(B, S, C)
    want = torch.where(want.isnan(), torch.full_like(want, -float("inf")), want).amax(1)
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got.sign()[want.isinf()], want.sign()[want.isinf()])
    seen = want.isfinite()
    # fp32 sums of 1024 products (the largest score is some 40 of them)
    assert not seen.any() or (got - want)[seen].abs().max() <= 1e-6 * want[seen].abs().max()
