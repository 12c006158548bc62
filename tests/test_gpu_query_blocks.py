"""Blocks of query rows on both sides of the line between the one-pass kernel and the split keys, samples shorter than the splits, and a workspace
that holds the splits by rows only, against the oracle."""
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


# (rows of the samples, keys in front of them): one workgroup a KV head, a tile more, both sides of the lines at 8, 32 and 64 tiles, one key to 16 splits
@pytest.mark.parametrize("lens,mem", [([16], 0), ([16], 411), ([16], 413), ([16, 700, 20], 5), ([33], 255), ([128], 684), ([128], 685), ([129], 1200), ([256, 17], 2000), ([64] * 4, 1260),
                                      ([64] * 4, 1261), ([20, 31, 500], 5000), ([600], 4200)])
def test_against_the_oracle(lens, mem):
    from msa_amd import _lib, ops
    print(f"[query_blocks] {lens} behind {mem}", flush=True)
    lib, D, Hq, Hkv = _lib.load(), 128, 32, 8
    g = torch.Generator().manual_seed(sum(lens) + mem)
    B, tq, kv = len(lens), sum(lens), [n + max(0, mem - 97 * b) for b, n in enumerate(lens)]
    q = torch.randn((tq, Hq, D), generator=g).bfloat16()
    k, v = (torch.randn((sum(kv), Hkv, D), generator=g).bfloat16() for _ in range(2))
    cu, off = torch.tensor([0] + lens).cumsum(0).int(), torch.tensor([0] + kv).cumsum(0)[:-1]
    qd, kd, vd, cud, offd, kld = q.cuda(), k.cuda(), v.cuda(), cu.cuda(), off.cuda(), torch.tensor(kv).int().cuda()
    got = [ops.sparse_attn(qd, kd, vd, offd, kld, max(kv), cu_q=cud, max_sq=max(lens)).cpu()]
    full, out = lib.msa_attn_workspace_bytes(tq, Hq, Hkv, D, max(kv)), torch.empty_like(qd)
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    call = lambda n: lib.msa_sparse_attn(ops.ptr(qd), ops.ptr(cud), ops.ptr(kd), ops.ptr(vd), ops.ptr(offd), ops.ptr(kld), B, tq, max(lens), max(kv), Hq, Hkv, D,
                                         ops.dtype_code(qd.dtype), D ** -0.5, 1, ops.ptr(out), ops.ptr(ws), n, ops._stream())
    per = tq * Hq * (D + 2) * 4
    least = next(n for n in range(per, full + 1024, per) if call(min(n + 512, full)) == 0)      # the least that is taken
    for n in {min(least + 512, full), full}:
        assert call(n) == 0
        got.append(out.cpu())
    for b, n in enumerate(lens):
        want = cf.attention(q[cu[b]:cu[b + 1]], k[off[b]:off[b] + kv[b]], v[off[b]:off[b] + kv[b]], causal=True)
        for o in got:
            assert cf.rel_err(o[cu[b]:cu[b + 1]], want) < 1e-2


def test_no_keys_are_refused():
    from msa_amd import _lib, ops
    q, k = torch.zeros((16, 32, 128), device="cuda").bfloat16(), torch.zeros((1, 8, 128), device="cuda").bfloat16()
    cu = torch.tensor([0, 16]).int().cuda()
    with pytest.raises(_lib.MsaError):
        ops.sparse_attn(q, k, k, torch.zeros(1, dtype=torch.int64, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda"), 0, cu_q=cu, max_sq=16)
