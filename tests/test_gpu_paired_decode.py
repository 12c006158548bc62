"""Decoding samples of different lengths dealt in pairs: both sides of the rule's lines, up to 64 samples, a second round that is not full,
empty and full caches, and a workspace that holds the even splits only."""
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


def lengths(kind, B, cap, g):
    if kind == "equal":
        return [cap - 1] * B
    if kind == "one long":
        return [1] * (B - 1) + [cap]
    n = torch.randint(0, cap + 1, (B,), generator=g).tolist()
    n[0], n[B // 2] = 0, cap
    return n


@pytest.mark.parametrize("B,Hkv,G,cap", [(16, 8, 4, 2000), (16, 8, 4, 1999), (15, 8, 4, 640), (5, 8, 4, 1920), (7, 8, 4, 1500), (13, 4, 8, 1440), (64, 8, 4, 160),
                                         (63, 2, 4, 700), (50, 8, 4, 170), (4, 8, 4, 8000), (17, 4, 4, 1200), (9, 4, 8, 2240), (65, 2, 4, 700)])
def test_paired(B, Hkv, G, cap):
    from msa_amd import _lib, ops
    lib, D, Hq = _lib.load(), 128, Hkv * G
    g = torch.Generator().manual_seed(B * 7 + Hkv)
    qkv = torch.randn((B, (Hq + 2 * Hkv) * D), generator=g).bfloat16().cuda()
    qw, kw = (1 + 0.1 * torch.randn(D, generator=g)).bfloat16().cuda(), (1 + 0.1 * torch.randn(D, generator=g)).bfloat16().cuda()
    rope = ops.rope_tables(1024, D, 1e6, device="cuda")
    kc0, vc0 = (torch.randn((B, cap, Hkv, D), generator=g).bfloat16().cuda() for _ in range(2))
    kv_off = torch.arange(B, dtype=torch.int64, device="cuda") * cap
    for kind in ("ragged", "equal", "one long"):
        print(f"[paired_decode] B={B} Hkv={Hkv} G={G} cap={cap} {kind}", flush=True)
        lens = torch.tensor(lengths(kind, B, cap, g), dtype=torch.int32)
        pos = torch.randint(0, 1100, (B,), generator=g).cuda()
        kc1, vc1, l1 = kc0.clone(), vc0.clone(), lens.cuda()
        q = ops.qk_norm_rope_append(qkv, Hq, Hkv, D, pos, qw, kw, 1e-6, rope, kc1, vc1, l1)
        want = ops.sparse_attn(q, kc1.view(-1, Hkv, D), vc1.view(-1, Hkv, D), kv_off, l1, cap, causal=True)
        full = lib.msa_attn_workspace_bytes(B, Hq, Hkv, D, cap)
        for short in (False, True):
            kc2, vc2, l2 = kc0.clone(), vc0.clone(), lens.cuda()
            if short:                                      # the least that is taken
                ws, out = torch.empty(full, dtype=torch.uint8, device="cuda"), torch.empty((B, Hq, D), dtype=torch.bfloat16, device="cuda")
                call = lambda n: lib.msa_decode_attn_fused(ops.ptr(qkv), qkv.shape[1], ops.ptr(pos), ops.ptr(qw), ops.ptr(kw), 1e-6, ops.ptr(rope[0]), ops.ptr(rope[1]), 1024,
                                                           B, Hq, Hkv, D, ops.ptr(kc2), ops.ptr(vc2), cap, ops.ptr(l2), D ** -0.5, ops.ptr(out), ops.ptr(ws), n, ops._stream())
                per = B * Hq * (D + 2) * 4
                least = next(n for n in range(per, full + 512, per) if call(min(n + 512, full)) == 0)
                assert least <= full
                got = out
            else:
                got = ops.decode_attn_fused(qkv, Hq, Hkv, D, pos, qw, kw, 1e-6, rope, kc2, vc2, l2)
            assert l2.cpu().tolist() == l1.cpu().tolist()
            assert torch.equal(kc2, kc1) and torch.equal(vc2, vc1)
            # of the largest value: two roundings to bf16, 2^-9 each where they fall apart, and fp32 sums in another order
            assert cf.rel_err(got.cpu(), want.cpu()) <= 2.0**-8 + 1e-5
