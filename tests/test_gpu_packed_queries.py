"""Batches of short queries that share row blocks in the routing scan: units of 8 and 4 rows in the streaming forms, of 8 in the large tiles."""
import numpy as np
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu
# fp32 sums of 1024 products of bf16 operands in another order: 2 * 1024 * 2^-24 of the sum of the products' magnitudes, which is at most
# one (the mean over heads of unit vectors' products)
SUMS = 2 * 1024 * 2.0 ** -24


def _case(B, S, Hkv, chunks, seed):
    from msa_amd import ops
    g = torch.Generator(device="cuda").manual_seed(seed)
    dco = np.concatenate([[0], np.cumsum(chunks)])
    kr = torch.randn((int(dco[-1]), Hkv, 128), generator=g, device="cuda")
    kr = kr.div_(kr.norm(dim=-1, keepdim=True)).to(torch.bfloat16)
    bank = ops.Bank(1, dco.tolist(), list(range(len(chunks))), Hkv, 128, torch.bfloat16)
    bank.set_layer(0, kr)
    q = torch.randn((B, S, 4 * Hkv, 128), generator=g, device="cuda").to(torch.bfloat16)
    mask = torch.rand((B, S), generator=g, device="cuda") > 0.25
    mask[:, S // 2] = True
    mask[B - 1] = False                        # nothing scored
    return ops, bank, kr, dco, q, mask


@pytest.mark.parametrize("B,S,Hkv", [(28, 2, 8), (10, 3, 8), (16, 4, 8), (32, 1, 8), (32, 4, 4), (7, 5, 8), (16, 8, 8), (3, 37, 8), (5, 24, 8), (2, 57, 2),
                                     (13, 9, 8), (32, 5, 8), (9, 100, 8), (5, 33, 8), (40, 17, 4), (300, 2, 2), (33, 7, 1), (4, 260, 8)])
def test_packed_queries(B, S, Hkv):
    print(f"[case] packed B={B} S={S} Hkv={Hkv}", flush=True)
    ops, bank, kr, dco, q, mask = _case(B, S, Hkv, [5, 1, 8, 2, 11, 3, 1, 40] * 31, 70 + B + S)
    bank.workspace(B, S, 4 * Hkv, 64, "cuda").fill_(0xFF)
    s, d, _ = ops.route_topk(bank, 0, q, mask, "cosine", 1.0, 64)
    ds = cf.doc_scores(cf.chunk_scores(q.cpu(), mask.cpu(), kr.cpu(), "cosine"), dco)
    live = mask.any(dim=1).cpu()
    s, d = s.cpu(), d.cpu().long()
    assert not cf.topk_acceptable(ds[live], d[live], 64)
    assert cf.rel_err(s[live], torch.gather(ds, 1, d)[live]) < 1e-2
    assert torch.isinf(s[~live]).all()
    for b in range(0, B - 1, max(1, B // 6)):  # a query by itself has row blocks of its own
        alone, _, _ = ops.route_topk(bank, 0, q[b:b + 1], mask[b:b + 1], "cosine", 1.0, 64)
        assert (alone.cpu()[0] - s[b]).abs().max() <= SUMS


def test_packed_queries_in_a_bank_of_the_tile_pool():
    """One tile of query rows over so many of chunks that the last ones are handed out; the unscored rows come with no mask."""
    r = np.random.default_rng(5)
    ops, bank, kr, dco, q, _ = _case(31, 6, 4, r.integers(1, 33, size=66000), 9)
    print(f"[case] packed, {kr.shape[0]} chunks", flush=True)
    assert kr.shape[0] >= 16 * 256 * 256
    s, d, _ = ops.route_topk(bank, 0, q, None, "cosine", 1.0, 32)
    for b in (0, 7, 30):
        alone, _, _ = ops.route_topk(bank, 0, q[b:b + 1], None, "cosine", 1.0, 32)
        assert (alone - s[b:b + 1]).abs().max() <= SUMS
    qs = q[7].float()
    qs = (qs / qs.norm(dim=-1, keepdim=True)).view(6, 4, 4, 128).sum(2).to(torch.bfloat16).float()
    for doc, score in zip(d[7].tolist(), s[7].tolist()):
        true = (kr[dco[doc]:dco[doc + 1]].float().reshape(-1, 512) @ qs.reshape(6, 512).T).max() / 16
        assert abs(float(true) - score) <= 2 * SUMS
