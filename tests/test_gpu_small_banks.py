"""Routing over small banks: the fp32 form that splits K over a workgroup's wavefronts at its edges (chunks that are no multiple of 32,
row blocks shared out over workgroups, queries without a scored token, per-chunk scores) against float64, single candidate lists,
and the gather's plan with documents that many samples share."""
import numpy as np
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


def make(doc_chunks, B, S, seed, host=False):
    from msa_amd import ops
    g = torch.Generator().manual_seed(seed)
    off = np.concatenate([[0], np.cumsum(doc_chunks)])
    C = int(off[-1])
    kr = torch.nn.functional.normalize(torch.randn((C, 8, 128), generator=g), dim=-1)
    q = torch.randn((B, S, 32, 128), generator=g)
    bank = ops.Bank(1, off.tolist(), [7 * i + 1 for i in range(len(doc_chunks))], 8, 128, torch.float32)
    kv = [torch.randn((C, 8, 128), generator=g).pin_memory() for _ in range(2)] if host else [None, None]
    bank.set_layer(0, kr.cuda(), *kv)
    return bank, kr, q, off, kv


# (largest document, documents, queries, tokens): 1 chunk; 31 to 33 and their neighbours; more row blocks than a workgroup keeps (1 x
# 1200 tokens: 38 blocks); blocks of many queries; the line to the tiles (chunks x rows = 2^21) from both sides;
# documents of more chunks than a workgroup has, of which it sees several
@pytest.mark.parametrize("top,docs,B,S", [(1, 1, 1, 1), (1, 31, 2, 33), (1, 32, 1, 64), (1, 33, 3, 70), (9, 40, 1, 1200), (5, 300, 40, 5), (17, 800, 2, 130),
                                          (16, 2100, 1, 65), (16, 2100, 1, 128), (16, 2040, 1, 128),
                                          (90, 12, 1, 1000), (40, 16, 3, 70), (33, 30, 2, 64)])
def test_split_scores(top, docs, B, S):
    from msa_amd import ops
    rng = np.random.default_rng(docs)
    doc_chunks = rng.integers(1, top + 1, size=docs).tolist()
    bank, kr, q, off, _ = make(doc_chunks, B, S, docs + S)
    mask = torch.ones((B, S), dtype=torch.bool)
    if B > 1:
        mask[1, : (S + 1) // 2] = False
        mask[B - 1, :] = False                           # no scored token at all
        mask[B - 1, S - 1] = B == 2
    want = cf.chunk_scores(q, mask, kr)
    got = ops.chunk_scores(bank, 0, q.cuda(), mask.cuda()).cpu().double()
    seen = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), seen)
    # 1024 products of unit vectors in fp32: 1e-5 of the largest score
    assert (got - want)[seen].abs().max() <= 1e-5 * want[seen].abs().max()
    per_doc = torch.stack([want[:, off[d]:off[d + 1]].amax(1) for d in range(docs)], 1)
    k = min(16, docs)
    scores, doc, gid = (t.cpu() for t in ops.route_topk(bank, 0, q.cuda(), mask.cuda(), topk=k))
    for b in range(B):
        if not mask[b].any():
            assert torch.isinf(scores[b]).all()
            continue
        assert (scores[b].double() - per_doc[b].topk(k).values).abs().max() <= 1e-5 * per_doc[b].abs().max()
        assert (per_doc[b][doc[b].long()] - scores[b].double()).abs().max() <= 1e-5 * per_doc[b].abs().max()
        assert torch.equal(gid[b], 7 * doc[b].long() + 1) and len(set(doc[b].tolist())) == k


@pytest.mark.parametrize("B,k", [(1, 1), (3, 16), (33, 17), (20, 33), (32, 64), (70, 64)])
def test_gather_plan_of_shared_documents(B, k):
    """Few documents for many picks: nearly all are shared, some repeat within a sample, some are out of range."""
    from msa_amd import ops
    rng = np.random.default_rng(B * k)
    doc_chunks = rng.integers(1, 6, size=80).tolist()
    bank, _, _, off, kv = make(doc_chunks, 1, 1, B, host=True)
    sel = torch.from_numpy(rng.integers(-2, 83, size=(B, k)).astype(np.int32))
    keep = [sorted({d for d in row if 0 <= d < 80}) for row in sel.tolist()]
    want = [torch.cat([t[off[d]:off[d + 1]] for row in keep for d in row] + [t[:0]]) for t in kv]
    n = want[0].shape[0]
    k_out, v_out, cu = ops.gather_kv_device(bank, 0, sel.cuda(), max(1, n))
    assert cu.tolist() == np.concatenate([[0], np.cumsum([sum(doc_chunks[d] for d in row) for row in keep])]).tolist()
    assert torch.equal(k_out[:n].cpu(), want[0]) and torch.equal(v_out[:n].cpu(), want[1])


@pytest.mark.parametrize("dtype,L", [(torch.float32, 1), (torch.float32, 200), (torch.bfloat16, 255)])
def test_single_pass_decode_attention(dtype, L):
    """Contexts that are not split: the output comes from the first launch; a sample without keys yields zeros."""
    from msa_amd import ops
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(s, generator=g).to(dtype) for s in ((3, 32, 128), (3 * L, 8, 128), (3 * L, 8, 128)))
    lens = torch.tensor([L, 0, max(1, L // 2)], dtype=torch.int32)
    out = ops.sparse_attn(q.cuda(), k.cuda(), v.cuda(), (torch.arange(3) * L).cuda(), lens.cuda(), L).cpu().double()
    assert (out[1] == 0).all()
    for b in (0, 2):
        kk, vv = (t[b * L:b * L + int(lens[b])].double().repeat_interleave(4, dim=1) for t in (k, v))
        p = torch.softmax((q[b].double()[None] * kk).sum(-1) * 128 ** -0.5, dim=0)
        want = (p[..., None] * vv).sum(0)
        assert (out[b] - want).abs().max() <= (1e-5 if dtype == torch.float32 else 1e-2) * want.abs().max()


@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_decode_attention_through_the_ring(G):
    """bf16 rows at the edges of a step's 32 keys, a round of four steps and a split, cut out of one block of keys, whose other rows
    are NaN.  Bound: the output's rounding (half a unit of eight bits, 2^-8 of it) and the weights' (two bf16 parts, 2^-16 of the sum
    of |p v|, twice for the fp32 sums), also beside the infinite value."""
    from msa_amd import ops
    lens = [1, 31, 32, 33, 127, 128, 129, 0, 255, 257, 1030, 2100]
    g = torch.Generator().manual_seed(G)
    q = (2 * torch.randn((len(lens), 2 * G, 128), generator=g)).bfloat16()
    off = [2 * b + sum(lens[:b]) for b in range(len(lens))]
    k, v = (torch.full((off[-1] + lens[-1] + 2, 2, 128), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    for o, n in zip(off, lens):
        k[o:o + n], v[o:o + n] = (torch.randn((n, 2, 128), generator=g).bfloat16() for _ in range(2))
    v[off[4] + 100, 0, 5] = float("inf")
    out = ops.sparse_attn(q.cuda(), k.cuda(), v.cuda(), torch.tensor(off).cuda(), torch.tensor(lens, dtype=torch.int32).cuda(), max(lens)).cpu().double()
    for b, (o, n) in enumerate(zip(off, lens)):
        kk, vv = (t[o:o + n].double().repeat_interleave(G, dim=1) for t in (k, v))
        p = torch.softmax((q[b].double()[None] * kk).sum(-1) * 128 ** -0.5, dim=0)
        want = (p[..., None] * vv).sum(0)
        fin = torch.isfinite(want)
        assert torch.equal(out[b][~fin], want[~fin])
        bound = want.abs() * 2 ** -8 + (p[..., None] * vv.abs()).sum(0) * 2 ** -15
        assert ((out[b] - want).abs() <= bound)[fin].all()


def _attention(q, k, v):
    p = torch.softmax((q.double()[:, None] * k.double()[None]).sum(-1) * 128 ** -0.5, dim=1)       # [rows, keys, heads]
    return (p[..., None] * v.double()[None]).sum(1)


@pytest.mark.parametrize("dtype,sq,L", [(torch.bfloat16, 1, 700), (torch.bfloat16, 1, 4400), (torch.float32, 1, 700), (torch.float32, 1, 4400),
                                        (torch.bfloat16, 12, 100), (torch.bfloat16, 12, 700), (torch.bfloat16, 12, 4400)])
def test_infinite_values_in_the_last_split(dtype, sq, L):
    """One sample, one infinite value among its last keys: splits of 256 keys or more, none of them sixteen or a multiple, single
    rows and query blocks (the last key but one: a tile's last row also stands in for those behind it).  The head's column is
    infinite and nothing else changes.  Bounds as for single passes above."""
    from msa_amd import ops
    g = torch.Generator().manual_seed(L + sq)
    q, k, v = (torch.randn(s, generator=g).to(dtype) for s in ((sq, 8, 128), (L, 2, 128), (L, 2, 128)))
    v[L - (1 if sq == 1 else 2), 1, 7] = float("inf")
    cu = torch.tensor([0, sq], dtype=torch.int32).cuda() if sq > 1 else None
    out = ops.sparse_attn(q.cuda(), k.cuda(), v.cuda(), torch.zeros(1, dtype=torch.int64).cuda(), torch.tensor([L], dtype=torch.int32).cuda(), L, cu_q=cu,
                          max_sq=sq, causal=False).cpu().double()
    want = _attention(q, k.repeat_interleave(4, dim=1), v.repeat_interleave(4, dim=1))
    assert torch.isinf(want[:, 4:, 7]).all() and torch.equal(torch.isfinite(out), torch.isfinite(want))
    fin = torch.isfinite(want)
    assert (out[~fin] == want[~fin]).all()
    assert (out - want)[fin].abs().max() <= (1e-5 if dtype == torch.float32 else 1e-2) * want[fin].abs().max()


@pytest.mark.parametrize("infinite", [False, True])
@pytest.mark.parametrize("G", [1, 2])
def test_weights_of_one_and_two_heads_keep_their_bits(G, infinite):
    """Groups of one and two heads: three keys whose weights are 1, p and 1 and whose values cancel but for 2^-18 of their size, so
    that the output's rounding shows nothing and the weights' everything: 16 bits of p leave errors of 2^-18.  Bound: 2^-20 of the sum
    of |p v| (p from the hardware's 2^x of an argument of up to 6 rounded twice to fp32: 2^-21.5; the fp32 sums) and the rounding of
    the output.  With an infinite value in another column as well."""
    from msa_amd import ops
    B, H = 64, 2 * G
    g = torch.Generator().manual_seed(G)
    q, k, v = torch.zeros((B, H, 128)), torch.zeros((3 * B, 2, 128)), torch.zeros((3 * B, 2, 128))
    q[..., 0] = 1.0
    k[1::3, :, 0] = (-40 * torch.rand((B, 2), generator=g)).bfloat16().float()         # score 0, k / sqrt(128), 0
    p = torch.exp(k[1::3, :, 0].double() * 128 ** -0.5)[..., None]
    v[1::3] = torch.randn((B, 2, 128), generator=g).bfloat16().float()
    v[0::3] = (-(p * v[1::3].double())).bfloat16().float()
    v[2::3] = (-(p * v[1::3].double() + v[0::3].double())).bfloat16().float()
    want = ((v[0::3] + p * v[1::3].double() + v[2::3]) / (2 + p)).repeat_interleave(G, dim=1)
    size = ((v[0::3].abs() + p * v[1::3].double().abs() + v[2::3].abs()) / (2 + p)).repeat_interleave(G, dim=1)
    if infinite:
        v[1::3, 1, 64] = float("inf")
        want[:, G:, 64] = float("inf")
    out = ops.sparse_attn(q.bfloat16().cuda(), k.bfloat16().cuda(), v.bfloat16().cuda(), (3 * torch.arange(B)).cuda(),
                          torch.full((B,), 3, dtype=torch.int32).cuda(), 3).cpu().double()
    fin = torch.isfinite(want)
    assert torch.equal(out[~fin], want[~fin])
    assert ((out - want).abs() <= want.abs() * 2 ** -8 + size * 2 ** -20)[fin].all()


@pytest.mark.parametrize("B,L", [(1, 300), (3, 1024), (3, 1100), (16, 1300), (24, 2815), (24, 2816), (48, 1500)])
def test_split_plans_and_partials(B, L):
    """2 to 18 partials a head, four and sixteen a batch of the combining kernel and their neighbours, in plans of one and of two
    workgroups a compute unit (24 samples of 2 heads from 2816 keys on).  Bounds as in the test of the ring."""
    from msa_amd import ops
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(s, generator=g).bfloat16() for s in ((B, 8, 128), (B * L, 2, 128), (B * L, 2, 128)))
    lens = torch.tensor([L - 7 * b for b in range(B)], dtype=torch.int32)
    out = ops.sparse_attn(q.cuda(), k.cuda(), v.cuda(), (L * torch.arange(B)).cuda(), lens.cuda(), L).cpu().double()
    for b in range(0, B, max(1, B // 4)):
        kk, vv = (t[b * L:b * L + int(lens[b])].double().repeat_interleave(4, dim=1) for t in (k, v))
        p = torch.softmax((q[b].double()[None] * kk).sum(-1) * 128 ** -0.5, dim=0)
        want = (p[..., None] * vv).sum(0)
        assert ((out[b] - want).abs() <= want.abs() * 2 ** -8 + (p[..., None] * vv.abs()).sum(0) * 2 ** -15).all()


# both sides of each line between the ring and the vector units: 512 rows and heads, 128 keys with one head, 1024 with two
@pytest.mark.parametrize("G,B,L", [(1, 4, 128), (1, 4, 129), (1, 256, 100), (1, 257, 100), (1, 3, 2100), (2, 5, 128), (2, 20, 2048), (2, 256, 90), (2, 257, 90),
                                   (2, 257, 1024), (2, 257, 1025)])
def test_small_groups_on_both_sides_of_the_line(G, B, L):
    """Ragged samples out of one block of keys whose other rows are NaN, one of them empty, one with an infinite value in its last key.
    Bounds as in the test of the ring."""
    from msa_amd import ops
    g = torch.Generator().manual_seed(B + L)
    q = (2 * torch.randn((B, 2 * G, 128), generator=g)).bfloat16()
    lens = [L, 0, *(1 + int(x) for x in torch.randint(0, L, (B - 2,), generator=g))]
    k, v = (torch.full((B * (L + 1), 2, 128), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    off = [b * (L + 1) for b in range(B)]
    for o, n in zip(off, lens):
        k[o:o + n], v[o:o + n] = (torch.randn((n, 2, 128), generator=g).bfloat16() for _ in range(2))
    v[off[2] + lens[2] - 1, 1, 9] = float("inf")
    out = ops.sparse_attn(q.cuda(), k.cuda(), v.cuda(), torch.tensor(off).cuda(), torch.tensor(lens, dtype=torch.int32).cuda(), L).cpu().double()
    for b, (o, n) in enumerate(zip(off, lens)):
        kk, vv = (t[o:o + n].double().repeat_interleave(G, dim=1) for t in (k, v))
        p = torch.softmax((q[b].double()[None] * kk).sum(-1) * 128 ** -0.5, dim=0)
        want, size = (p[..., None] * vv).sum(0), (p[..., None] * vv.abs()).sum(0)
        fin = torch.isfinite(want)
        assert fin.all() == (b != 2) and torch.equal(out[b][~fin], want[~fin])
        assert ((out[b] - want).abs() <= want.abs() * 2 ** -8 + size * 2 ** -15)[fin].all(), (b, n)
