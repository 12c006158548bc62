"""fp32 decode attention: one head, two heads or a whole group a workgroup, on both sides of the lines between them, against float64."""
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


# (rows, keys, query heads, KV heads): rows x heads x splits around 256 and 512, one to eight splits, groups of one to eight heads, fewer keys
# than a workgroup has slots
@pytest.mark.parametrize("B,L,Hq,Hkv", [(1, 1, 32, 8), (1, 192, 32, 8), (8, 256, 32, 8), (8, 257, 32, 8), (9, 33, 32, 8), (16, 250, 32, 8), (17, 65, 32, 8),
                                        (2, 513, 32, 8), (2, 2049, 32, 8), (3, 2049, 32, 8), (1, 100, 8, 8), (33, 31, 8, 8), (4, 300, 16, 8), (16, 40, 16, 8),
                                        (33, 40, 16, 8), (4, 129, 64, 8), (5, 700, 64, 8), (9, 64, 64, 8)])
def test_heads_a_workgroup(B, L, Hq, Hkv):
    from msa_amd import ops
    g = torch.Generator().manual_seed(B * L + Hq)
    lens = [L] + [int(n) for n in torch.randint(0, L + 1, (B - 1,), generator=g)]
    k, v = (torch.randn((B, L, Hkv, 128), generator=g) for _ in range(2))
    q = torch.randn((B, Hq, 128), generator=g)
    for b, n in enumerate(lens):                           # what lies behind a sample's keys must not be seen
        k[b, n:], v[b, n:] = float("nan"), float("inf")
    if B > 1 and lens[1] > 0:
        v[1, lens[1] - 1, 0, 7] = float("inf")             # an infinite value stays one, in its own place
    out = ops.sparse_attn(q.cuda(), k.cuda().view(-1, Hkv, 128), v.cuda().view(-1, Hkv, 128), (torch.arange(B, dtype=torch.int64) * L).cuda(),
                          torch.tensor(lens, dtype=torch.int32).cuda(), L).cpu()
    for b, n in enumerate(lens):
        if n == 0:
            assert not out[b].any()
            continue
        got, vb = out[b:b + 1], v[b, :n].clone()
        if b == 1:
            assert torch.isinf(got[0, :Hq // Hkv, 7]).all() and int(torch.isinf(got).sum()) == Hq // Hkv
            vb[n - 1, 0, 7], got = 0.0, got.clone()
            got[0, :Hq // Hkv, 7] = cf.attention(q[b:b + 1], k[b, :n], vb)[0, :Hq // Hkv, 7].float()
        assert cf.rel_err(got, cf.attention(q[b:b + 1], k[b, :n], vb)) < 1e-5          # fp32 sums
