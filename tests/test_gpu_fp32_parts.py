"""fp32 routing on the bf16 matrix cores (values in three parts): edges of the columns and row blocks, the lines to the other forms, infinities
and NaN, and a workspace that holds no parts, against float64."""
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


def make(C, B, S, seed):
    from msa_amd import ops
    g = torch.Generator().manual_seed(seed)
    kr = torch.nn.functional.normalize(torch.randn((C, 8, 128), generator=g), dim=-1)
    q = torch.randn((B, S, 32, 128), generator=g)
    off = list(range(0, C, 3)) + [C]
    return ops.Bank(1, off, list(range(len(off) - 1)), 8, 128, torch.float32), kr, q, off


# (chunks, queries, tokens): columns of 32 with a rest, one to 256 of them and one more; one row block to 32; queries that share a workgroup's blocks;
# several workgroups a column; both sides of the line
@pytest.mark.parametrize("C,B,S", [(1, 1, 1), (31, 1, 32), (33, 2, 33), (300, 16, 32), (300, 1, 64), (700, 3, 200), (2000, 1, 128), (2720, 3, 32), (3300, 2, 96), (4200, 1, 128),
                                   (8000, 1, 64), (8192, 2, 40), (8193, 1, 64), (1500, 12, 32), (8191, 1, 1024), (100, 1, 1025)])
def test_scores(C, B, S):
    from msa_amd import ops
    bank, kr, q, off = make(C, B, S, C + S)
    bank.set_layer(0, kr.cuda(), None, None)
    mask = torch.ones((B, S), dtype=torch.bool)
    if B > 1:
        mask[0, : S // 2] = False
        mask[1, :] = False
    want = cf.chunk_scores(q, mask, kr)
    got = ops.chunk_scores(bank, 0, q.cuda(), mask.cuda()).cpu().double()
    seen = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), seen)
    # 1024 products of values that hold 24 bits and sums in fp32
    assert (got - want)[seen].abs().max() <= 1e-6 * want[seen].abs().max()
    k = min(8, len(off) - 1)
    scores, doc, _ = (t.cpu() for t in ops.route_topk(bank, 0, q.cuda(), mask.cuda(), topk=k))
    per_doc = torch.stack([want[:, a:b].amax(1) for a, b in zip(off, off[1:])], 1)
    for b in range(B):
        if mask[b].any():
            assert (scores[b].double() - per_doc[b].topk(k).values).abs().max() <= 1e-6 * per_doc[b].abs().max()


def test_infinities_and_nan():
    """A product with an infinity keeps its sign, a row whose sum is no number counts for nothing (as in a maximum that ignores NaN)."""
    from msa_amd import ops
    inf, nan = float("inf"), float("nan")
    bank, kr, q, _ = make(200, 2, 40, 5)
    q = q.abs() + 0.1                                      # all products positive
    kr[3, 0, 0], kr[40, 2, 9], kr[41, 1, 1], kr[41, 7, 127], kr[77, 5, 5], kr[199, 7, 127] = inf, -inf, inf, -inf, nan, 3e38
    bank.set_layer(0, kr.cuda(), None, None)
    got = ops.chunk_scores(bank, 0, q.cuda()).cpu()
    assert got[:, 3].tolist() == [inf, inf] and got[:, 40].tolist() == [-inf, -inf]
    assert got[:, 41].tolist() == [-inf, -inf] and got[:, 77].tolist() == [-inf, -inf]
    rest = [c for c in range(200) if c not in (3, 40, 41, 77)]
    assert torch.isfinite(got[:, rest]).all()


def test_a_workspace_without_room_for_the_parts():
    from msa_amd import _lib, ops
    C, B, S = 500, 2, 64
    bank, kr, q, off = make(C, B, S, 9)
    bank.set_layer(0, kr.cuda(), None, None)
    lib, qd = _lib.load(), q.cuda()
    need = bank.workspace_bytes(B, S, 32, 16, chunk_plane=True)
    want = ops.chunk_scores(bank, 0, qd).cpu()
    out = torch.empty((B, C), device="cuda")
    for bytes_ in (need, need - B * S * 2048):
        ws = torch.empty(bytes_, dtype=torch.uint8, device="cuda")
        ops.check(lib.msa_chunk_scores(bank.handle, 0, ops.ptr(qd), None, B, S, 32, 0, 1.0, ops.ptr(out), ops.ptr(ws), bytes_, ops._stream()), "msa_chunk_scores")
        assert (out.cpu() - want).abs().max() <= 2e-6 * want.abs().max()
    assert lib.msa_chunk_scores(bank.handle, 0, ops.ptr(qd), None, B, S, 32, 0, 1.0, ops.ptr(out), ops.ptr(ws), 4096, ops._stream()) != 0


def test_smallest_values():
    """Keys whose second and third parts are below the smallest normal number."""
    from msa_amd import ops
    bank, kr, q, _ = make(64, 1, 32, 7)
    kr = kr * 1e-35
    bank.set_layer(0, kr.cuda(), None, None)
    want = cf.chunk_scores(q, torch.ones((1, 32), dtype=torch.bool), kr)
    got = ops.chunk_scores(bank, 0, q.cuda()).cpu().double()
    # products below 2^-126 are rounded to multiples of 2^-149: 1024 of them, six to a product
    assert (got - want).abs().max() <= 1e-6 * want.abs().max() + 8 * 6 * 1024 * 2.0**-149
