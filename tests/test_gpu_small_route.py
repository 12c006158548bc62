"""The forms of routing and gather that small memories take, at the edges of their ranges: fp32 scoring through the ring, top-k of one and of
many lists, and the gather of up to 64 documents in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[small_route] {msg}", flush=True)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import ops
    return ops


def _bank(ops, docs, per, seed, host=False):
    g = torch.Generator(device="cuda").manual_seed(seed)
    counts = [per if per > 0 else 1 + (i * 7) % 5 for i in range(docs)]
    off = torch.tensor([0] + counts).cumsum(0)
    kr = torch.randn((int(off[-1]), 8, 128), generator=g, device="cuda")
    kr /= kr.norm(dim=-1, keepdim=True)
    bank = ops.Bank(1, off.to(torch.int32), torch.arange(docs) + 1, 8, 128, torch.float32)
    store = [torch.randn(kr.shape, pin_memory=True) for _ in range(2)] if host else [None, None]
    bank.set_layer(0, kr, *store)
    return bank, kr, off, store, g


# 191 / 192 / 256 / 257 workgroups of 32 chunks: one or two a compute unit; 31 and 33 chunks; blocks of several queries
@pytest.mark.parametrize("chunks,B,S", [(31, 1, 1), (33, 2, 40), (191 * 32, 1, 64), (192 * 32 - 5, 1, 64), (256 * 32, 2, 33), (256 * 32 + 1, 1, 64),
                                        (512 * 32 + 7, 3, 20), (700, 9, 128)])
def test_fp32_scores(ops, chunks, B, S):
    """fp32 sums of 1024 products: 1e-6 of the largest score, far below the distance of neighbouring documents here."""
    _say(f"fp32 scores chunks={chunks} B={B} S={S}")
    bank, kr, _, _, g = _bank(ops, chunks, 1, 1)
    q = torch.randn((B, S, 32, 128), generator=g, device="cuda")
    scores, docs, _ = ops.route_topk(bank, 0, q, None, topk=min(16, chunks))
    qd = q.double()
    qd = (qd / qd.norm(dim=-1, keepdim=True)).view(B, S, 8, 4, 128).sum(3).reshape(B * S, 1024) / 32
    want = (qd @ kr.double().view(-1, 1024).t()).view(B, S, chunks).amax(1)
    top = want.topk(min(16, chunks), 1)[0]
    assert (scores.double() - top).abs().max() < 1e-6
    assert (want.gather(1, docs.long()) - top).abs().max() < 1e-6


@pytest.mark.parametrize("docs", [1, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 2048 * 16 + 1, 2048 * 17, 2048 * 35 + 3])
def test_topk_of_every_list_length(ops, docs):
    """Documents of one chunk whose score is exact (a power of two or a sum of a few): the order is the score's, ties by document."""
    _say(f"topk docs={docs}")
    kr = torch.zeros((docs, 8, 128), device="cuda")
    r = torch.randperm(docs, generator=torch.Generator().manual_seed(docs)).cuda()
    kr[:, 0, 0] = (r // 3).float() / (1 << 17)                       # three documents a score
    bank = ops.Bank(1, torch.arange(docs + 1, dtype=torch.int32), torch.arange(docs) + 1, 8, 128, torch.float32)
    bank.set_layer(0, kr)
    q = torch.zeros((2, 3, 32, 128), device="cuda")
    q[:, 0, :4, 0] = 1.0
    for k in (1, 16, 64):
        _, got, _ = ops.route_topk(bank, 0, q, None, mode="scaled_dot", topk=k)
        order = torch.sort(-(r // 3), stable=True)[1][:k].to(torch.int32)
        want = torch.full((k,), -1, dtype=torch.int32, device="cuda")
        want[:len(order)] = order
        assert torch.equal(got[0], want) and torch.equal(got[1], want)


# lists of 2048 documents on 256 compute units: 258, 256 and 257 of them, up to two, four and eighteen a query
@pytest.mark.parametrize("docs,B", [(2049, 129), (2048, 256), (100, 257), (7000, 65), (2048 * 17 + 1, 15)])
def test_topk_of_many_lists(ops, docs, B):
    """Scores as above, rising for one query and falling for the next."""
    _say(f"topk docs={docs} B={B}")
    kr = torch.zeros((docs, 8, 128), device="cuda")
    r = torch.randperm(docs, generator=torch.Generator().manual_seed(docs)).cuda()
    kr[:, 0, 0] = (r // 3).float() / (1 << 17)                       # three documents a score
    bank = ops.Bank(1, torch.arange(docs + 1, dtype=torch.int32), torch.arange(docs) + 1, 8, 128, torch.float32)
    bank.set_layer(0, kr)
    q = torch.zeros((B, 1, 32, 128), device="cuda")
    q[0::2, :, :4, 0], q[1::2, :, :4, 0] = 1.0, -1.0
    for k in (1, 16, 64):
        _, got, _ = ops.route_topk(bank, 0, q, None, mode="scaled_dot", topk=k)
        for sign in (0, 1):
            want = torch.sort(-(r // 3) if sign == 0 else r // 3, stable=True)[1][:k].to(torch.int32)
            assert torch.equal(got[sign::2], want.expand(len(range(sign, B, 2)), -1))


@pytest.mark.parametrize("B,k,capacity", [(1, 1, 100), (1, 64, 400), (2, 32, 400), (4, 16, 400), (3, 5, 400), (4, 16, 37), (1, 17, 3), (5, 16, 400)])
def test_gather_of_few_documents(ops, B, k, capacity):
    """Against the rows themselves: documents of several samples, missing and repeated picks, rows behind the capacity."""
    _say(f"gather B={B} k={k} capacity={capacity}")
    bank, _, off, (hk, hv), g = _bank(ops, 30, 0, 2, host=True)
    sel = torch.randint(-1, 30, (B, k), generator=g, device="cuda", dtype=torch.int32)
    out = [torch.full((capacity, 8, 128), 7.0, device="cuda") for _ in range(2)]
    K, V, cu = ops.gather_kv_device(bank, 0, sel, capacity, out=tuple(out))
    torch.cuda.synchronize()
    rows, want_cu = [], [0]
    for b in range(B):
        for d in sorted(set(x for x in sel[b].tolist() if x >= 0)):
            rows += range(int(off[d]), int(off[d + 1]))
        want_cu.append(min(len(rows), capacity))
    assert cu.tolist() == want_cu
    n = min(len(rows), capacity)
    assert torch.equal(K[:n].cpu(), hk[rows[:n]]) and torch.equal(V[:n].cpu(), hv[rows[:n]])
    assert bool((K[n:] == 7).all()) and bool((V[n:] == 7).all())
