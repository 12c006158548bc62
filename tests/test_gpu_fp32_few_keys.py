"""fp32 decode attention of groups of one and two heads over few keys: both sides of the lines between four and eight wavefronts, rows on both sides of the
lines in their number, against float64."""
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (4, 4), (16, 8), (2, 1)])
@pytest.mark.parametrize("B", [1, 17, 40, 65])
@pytest.mark.parametrize("L", [1, 17, 64, 104, 105, 128, 129])
def test_few_keys(B, L, Hq, Hkv):
    from msa_amd import ops
    g = torch.Generator().manual_seed(B * L + Hq)
    lens = [L] + [int(n) for n in torch.randint(0, L + 1, (B - 1,), generator=g)]
    k, v = (torch.randn((B, L, Hkv, 128), generator=g) for _ in range(2))
    q = torch.randn((B, Hq, 128), generator=g)
    for b, n in enumerate(lens):                           # what lies behind a sample's keys must not be seen
        k[b, n:], v[b, n:] = float("nan"), float("inf")
    out = ops.sparse_attn(q.cuda(), k.cuda().view(-1, Hkv, 128), v.cuda().view(-1, Hkv, 128), (torch.arange(B, dtype=torch.int64) * L).cuda(),
                          torch.tensor(lens, dtype=torch.int32).cuda(), L).cpu()
    for b, n in enumerate(lens):
        if n == 0:
            assert not out[b].any()
        else:
            assert cf.rel_err(out[b:b + 1], cf.attention(q[b:b + 1], k[b, :n], v[b, :n])) < 1e-5          # fp32 sums
