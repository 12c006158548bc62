"""Batches of short queries that share row blocks in the routing scan: units of 8 and 4 rows in the streaming forms, of 8 in the large tiles."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu
# fp32 sums of 1024 products of bf16 operands in another order: 2 * 1024 * 2^-24 of the sum of the products' magnitudes, which is at most
# one (the mean over heads of unit vectors' products)
SUMS = 2 * 1024 * 2.0 ** -24


def _form(B, S, chunks, gathers=False):
    """(rows a query is a multiple of, whether the large tiles take them)."""
    from msa_amd import _lib
    unit, by_units = C.c_int32(), C.c_int32()
    assert _lib.load().msa_diag_row_packing(B, S, chunks, gathers, C.addressof(unit), C.addressof(by_units)) == 0
    return unit.value, bool(by_units.value)


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


# units of four and of eight in the streaming forms, of eight in the large tiles, and row blocks of a query's own where the others gain nothing
SMALL = {(4, False): [(28, 2, 8), (10, 3, 8), (16, 4, 8), (32, 1, 8), (32, 4, 4)], (8, False): [(7, 5, 8), (16, 8, 8), (3, 37, 8), (5, 24, 8)], (8, True): [(300, 2, 2)],
         (32, False): [(2, 57, 2), (13, 9, 8), (32, 5, 8), (9, 100, 8), (5, 33, 8), (40, 17, 4), (33, 7, 1), (4, 260, 8)]}


@pytest.mark.parametrize("form,B,S,Hkv", [(f, *c) for f, cases in SMALL.items() for c in cases])
def test_packed_queries(form, B, S, Hkv):
    assert _form(B, S, 31 * 71) == form
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


@pytest.mark.parametrize("form,B,S", [((4, False), 10, 3), ((4, False), 28, 2), ((8, False), 7, 5), ((8, True), 300, 2)])
def test_no_numbers(form, B, S):
    """What is no number counts for nothing in a maximum: a chunk of them, a document of such chunks and a query are what they are where a
    query has row blocks of its own."""
    print(f"[case] no numbers B={B} S={S}", flush=True)
    chunks = [20, 1, 32, 8, 44, 12, 4, 160] * 8
    ops, bank, kr, dco, q, _ = _case(B, S, 2, chunks, 5 + B)
    assert _form(B, S, kr.shape[0]) == form
    kr[2] = kr[20] = kr[700, 1, 7] = float("nan")               # one of a document's chunks, a document's only one, a value of one
    bank.set_layer(0, kr)
    q[1], q[2, 0], q[3, S - 1, 5] = float("nan"), float("nan"), float("nan")      # a query, a token, a head
    s, d, _ = ops.route_topk(bank, 0, q, None, "cosine", 1.0, 64)
    assert (s[1] == -torch.inf).all() and (s[0].isfinite().sum(), s[2].isfinite().sum()) == (len(chunks) - 1,) * 2
    assert (s.gather(1, (d == 1).long().argmax(1, keepdim=True)) == -torch.inf).all()                        # (all 64 documents come back)
    for b in range(min(B, 6)):
        alone, _, _ = ops.route_topk(bank, 0, q[b:b + 1], None, "cosine", 1.0, 64)
        assert torch.allclose(alone[0], s[b], rtol=0, atol=SUMS)


def _large(B, S, seed):
    """A bank of 300 tiles of chunks, the last one ragged, and what a call over it gives: (layers' bank, kr, queries, mask, the best 64 scores, all)."""
    r = np.random.default_rng(seed)
    chunks = r.integers(1, 41, size=4200)
    chunks = chunks[np.cumsum(chunks) <= 300 * 256 - 77].tolist()
    chunks.append(300 * 256 - 77 - sum(chunks))
    chunks = [c for c in chunks if c]
    ops, bank, kr, dco, q, mask = _case(B, S, 2, chunks, seed)
    mask[B - 1, S // 3] = True
    mask[B // 2] = False                       # nothing scored, in the middle
    doc = torch.repeat_interleave(torch.arange(len(chunks), device="cuda"), torch.tensor(chunks, device="cuda"))
    qn = q.float()
    qn = (qn / qn.norm(dim=-1, keepdim=True)).view(B, S, 2, 4, 128).sum(3).to(torch.bfloat16).float().view(B, S, 256)
    best = torch.full((B, len(chunks)), -torch.inf, device="cuda")
    for b in range(B):
        if mask[b].any():
            best[b].scatter_reduce_(0, doc, (qn[b, mask[b]] @ kr.float().view(-1, 256).T).amax(0) / 8, "amax")
    return ops, bank, kr, chunks, q, mask, best


def _check(s, d, best, live):
    want = best.topk(64, dim=1).values
    assert (s[live] - want[live]).abs().max() <= 2 * SUMS and (best.gather(1, d.long())[live] - s[live]).abs().max() <= 2 * SUMS
    assert torch.isinf(s[~live]).all()


@pytest.mark.parametrize("B,S", [(33, 7), (13, 9), (17, 20), (40, 17), (5, 33), (13, 37), (32, 37), (9, 100), (6, 200), (20, 1000)])
def test_queries_of_several_units_in_the_large_tiles(B, S):
    """1, 2, 3, 3, 5, 5, 5, 13, 25 and 125 units a query, which cross wavefronts' rows and tiles of rows at all places."""
    print(f"[case] units B={B} S={S}", flush=True)
    ops, bank, kr, chunks, q, mask, best = _large(B, S, 11 + B + S)
    assert _form(B, S, kr.shape[0]) == (8, True)
    bank.workspace(B, S, 8, 64, "cuda").fill_(0xFF)
    s, d, _ = ops.route_topk(bank, 0, q, mask, "cosine", 1.0, 64)
    _check(s, d, best, mask.any(dim=1))


@pytest.mark.parametrize("B,S", [(13, 9), (9, 100)])
def test_queries_in_units_beside_a_gather(B, S):
    """The large tiles carry a gather: all of both calls' results are those of the two by themselves."""
    print(f"[case] units and a gather B={B} S={S}", flush=True)
    ops, bank, kr, chunks, q, mask, best = _large(B, S, 12 + B + S)
    assert _form(B, S, kr.shape[0], True) == (8, True)
    g = torch.Generator().manual_seed(5)
    rows = [torch.randn(kr.shape, generator=g).to(torch.bfloat16).pin_memory() for _ in range(2)]
    bank.set_layer(0, kr, *rows)
    sel = torch.randint(0, len(chunks), (5, 7), generator=g).int()
    sel[1, :3], sel[2, 4], sel[3, 0] = sel[0, :3], sel[2, 3], -1         # shared by samples, twice in one, none
    sel = sel.cuda()
    want, rows_want = ops.route_topk(bank, 0, q, mask, "cosine", 1.0, 64), ops.gather_kv_device(bank, 0, sel, 35 * 40)
    bank.workspace(B, S, 8, 64, "cuda").fill_(0xFF)
    got, (k, v, cu) = ops.route_topk_gather(bank, 0, q, mask, "cosine", 1.0, 64, 0, sel, 35 * 40)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and torch.equal(cu, rows_want[2])
    n = int(cu[-1])
    assert n > 0 and torch.equal(k[:n], rows_want[0][:n]) and torch.equal(v[:n], rows_want[1][:n])
    _check(got[0], got[1], best, mask.any(dim=1))


def test_packed_queries_in_a_bank_of_the_tile_pool():
    """One tile of query rows over so many of chunks that the last ones are handed out; the unscored rows come with no mask."""
    r = np.random.default_rng(5)
    ops, bank, kr, dco, q, _ = _case(31, 6, 4, r.integers(1, 33, size=66000), 9)
    print(f"[case] packed, {kr.shape[0]} chunks", flush=True)
    assert kr.shape[0] >= 16 * 256 * 256 and _form(31, 6, kr.shape[0]) == (8, True)
    s, d, _ = ops.route_topk(bank, 0, q, None, "cosine", 1.0, 32)
    for b in (0, 7, 30):
        alone, _, _ = ops.route_topk(bank, 0, q[b:b + 1], None, "cosine", 1.0, 32)
        assert (alone - s[b:b + 1]).abs().max() <= SUMS
    qs = q[7].float()
    qs = (qs / qs.norm(dim=-1, keepdim=True)).view(6, 4, 4, 128).sum(2).to(torch.bfloat16).float()
    for doc, score in zip(d[7].tolist(), s[7].tolist()):
        true = (kr[dco[doc]:dco[doc + 1]].float().reshape(-1, 512) @ qs.reshape(6, 512).T).max() / 16
        assert abs(float(true) - score) <= 2 * SUMS
