"""Samples much shorter than their caches in a launch that has the workgroups for pairs: both sides of the line between dealing pieces in pairs and fewer
pieces, one sample beyond it, one to twelve pieces a sample, empty and full caches, and a captured step whose samples grow over the line."""
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


def operands(B, Hkv, G, cap, seed=0):
    from msa_amd import ops
    g = torch.Generator().manual_seed(B * 7 + Hkv + seed)
    rnd = lambda *s: torch.randn(s, generator=g).bfloat16().cuda()
    qw, kw = (1 + 0.1 * torch.randn(128, generator=g)).bfloat16().cuda(), (1 + 0.1 * torch.randn(128, generator=g)).bfloat16().cuda()
    return rnd(B, (Hkv * G + 2 * Hkv) * 128), qw, kw, ops.rope_tables(1024, 128, 1e6, device="cuda"), rnd(B, cap, Hkv, 128), rnd(B, cap, Hkv, 128), g


def both(qkv, qw, kw, rope, kc, vc, lens, pos, Hq, Hkv):
    """The fused step, and the same in two calls: q and the appended cache, then attention by rows."""
    from msa_amd import ops
    B, cap = kc.shape[:2]
    kc1, vc1, l1 = kc.clone(), vc.clone(), lens.clone()
    q = ops.qk_norm_rope_append(qkv, Hq, Hkv, 128, pos, qw, kw, 1e-6, rope, kc1, vc1, l1)
    want = ops.sparse_attn(q, kc1.view(-1, Hkv, 128), vc1.view(-1, Hkv, 128), torch.arange(B, dtype=torch.int64, device="cuda") * cap, l1, cap, causal=True)
    kc2, vc2, l2 = kc.clone(), vc.clone(), lens.clone()
    got = ops.decode_attn_fused(qkv, Hq, Hkv, 128, pos, qw, kw, 1e-6, rope, kc2, vc2, l2)
    assert torch.equal(l1, l2) and torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    # of the largest value: two roundings to bf16, 2^-9 each where they fall apart, and fp32 sums in another order
    assert cf.rel_err(got.cpu(), want.cpu()) <= 2.0**-8 + 1e-5


# (samples, KV heads, group, capacity, the line): one piece a sample, four, eight, nine of which five are left, twelve
@pytest.mark.parametrize("B,Hkv,G,cap,worth", [(64, 8, 4, 1024, 300), (16, 8, 4, 2400, 1200), (8, 8, 4, 4160, 2400), (8, 4, 8, 8200, 4800), (7, 8, 4, 2048, 450),
                                               (5, 8, 4, 2000, 600), (13, 8, 4, 700, 200)])
def test_both_sides(B, Hkv, G, cap, worth):
    qkv, qw, kw, rope, kc, vc, g = operands(B, Hkv, G, cap)
    for kind in ("below", "one above", "none", "few keys", "full"):
        print(f"[short_samples] B={B} Hkv={Hkv} cap={cap} {kind}", flush=True)
        n = torch.randint(0, worth, (B,), generator=g).int()
        n[0], n[B - 1] = worth - 1, 0
        if kind == "one above":
            n[B // 2] = worth
        if kind in ("none", "few keys"):
            n = torch.full((B,), 0).int() if kind == "none" else torch.arange(B).int() % 5
        if kind == "full":
            n[B // 2] = cap
        both(qkv, qw, kw, rope, kc, vc, n.cuda(), torch.randint(0, 1100, (B,), generator=g).cuda(), Hkv * G, Hkv)


def test_a_captured_step_that_grows_over_the_line():
    from msa_amd import ops
    B, Hkv, G, cap = 16, 8, 4, 2400
    qkv, qw, kw, rope, kc, vc, g = operands(B, Hkv, G, cap, 1)
    lens, pos = torch.full((B,), 1197, dtype=torch.int32, device="cuda"), torch.randint(0, 1000, (B,), generator=g).cuda()
    eager = [t.clone() for t in (kc, vc, lens)]
    step = lambda k, v, n: ops.decode_attn_fused(qkv, Hkv * G, Hkv, 128, pos, qw, kw, 1e-6, rope, k, v, n)
    scratch = [t.clone() for t in (kc, vc, lens)]
    step(*scratch)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(kc, vc, lens)
    for i in range(6):
        graph.replay()
        want = step(*eager)
        torch.cuda.synchronize()
        assert lens.cpu().tolist() == eager[2].cpu().tolist() == [1198 + i] * B
        assert torch.equal(out, want) and torch.equal(kc, eager[0]) and torch.equal(vc, eager[1])
