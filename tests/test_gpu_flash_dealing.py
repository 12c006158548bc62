"""The wide flash form's dealing of blocks: every block once whatever the samples' lengths, from one workgroup a key head to 256 (several groups of
them), empty samples, more samples than lanes, keys that end before their rows, against the 32-column form; and the choice between the forms."""
import pytest
import torch

from oracle import closed_form as cf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Hq,Hkv", [(4, 1), (4, 2), (6, 3), (16, 8), (8, 8), (64, 64), (260, 260)])
def test_every_block_once(Hq, Hkv, causal):
    from msa_amd import _lib, ops
    lib, D = _lib.load(), 128
    g = torch.Generator().manual_seed(Hq + causal)
    for lens, extra in (([1], 0), ([700], 30), ([0, 65, 0, 640, 1, 0], 5), ([3] * 90 + [900] + [1] * 50, 64), ([513, 64, 256, 1025, 255], -40), ([129] * 70, 0)):
        if Hq > 64 and sum(lens) > 1000:
            continue
        print(f"[flash_dealing] H={Hq}/{Hkv} causal={causal} {len(lens)} samples, {sum(lens)} rows, extra {extra}", flush=True)
        kv = [max(1, n + extra) for n in lens]
        q = torch.randn((sum(lens), Hq, D), generator=g).bfloat16().cuda()
        k, v = (torch.randn((sum(kv), Hkv, D), generator=g).bfloat16().cuda() for _ in range(2))
        cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
        off, kl = (torch.tensor([0] + kv).cumsum(0)[:-1]).cuda(), torch.tensor(kv).int().cuda()
        outs = []
        try:
            for form in (1, 2):
                _lib.check(lib.msa_flash_set_form(form), "msa_flash_set_form")
                out = torch.full_like(q, float("nan"))
                _lib.check(lib.msa_flash_attn(ops.ptr(q), ops.ptr(cu), ops.ptr(k), ops.ptr(v), ops.ptr(off), ops.ptr(kl), len(lens), sum(lens), Hq, Hkv, D, D ** -0.5, int(causal),
                                              ops.ptr(out), ops._stream()), "msa_flash_attn")
                torch.cuda.synchronize()
                outs.append(out.cpu())
        finally:
            lib.msa_flash_set_form(0)
        assert torch.isfinite(outs[1]).all()
        # of the largest value: weights and outputs rounded to bf16 (2^-9 each) in both
        assert cf.rel_err(outs[1], outs[0]) <= 4 * 2.0**-9


@pytest.mark.parametrize("lens,form", [([4096] * 2, 2), ([3500, 2000, 2500] * 2, 2), ([3500, 2000, 2500], 1), ([4000], 2), ([3400], 1), ([2048], 1), ([1100], 1), ([1000, 1048], 1), ([1500, 500], 1), ([400] * 6, 1), ([1999] * 5, 1), ([2048] * 4, 2), ([1024] * 8, 2), ([5000], 1), ([2200, 1780], 2), ([1540] * 2 + [1200] * 4, 2)])
def test_choice(lens, form):
    from msa_amd import _lib, ops
    lib, D, Hq, Hkv = _lib.load(), 128, 32, 8
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are for 256 compute units")
    print(f"[flash_dealing] choice {lens}", flush=True)
    q = torch.randn((sum(lens), Hq, D), device="cuda").bfloat16()
    k, v = (torch.randn((sum(lens), Hkv, D), device="cuda").bfloat16() for _ in range(2))
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    off, kl = cu[:-1].long(), torch.tensor(lens).int().cuda()
    # (one and two samples within two rounds of the 32-column form: the second round runs backwards)
    run = lambda: ops.sparse_attn(q, k, v, off, kl, max(lens), cu_q=cu, max_sq=max(lens))
    got = run()
    try:
        forced = {}
        for f in (1, 2):
            lib.msa_flash_set_form(f)
            forced[f] = run()
    finally:
        lib.msa_flash_set_form(0)
    assert not torch.equal(forced[1], forced[2]) and torch.equal(got, forced[form])
    assert cf.rel_err(forced[2].cpu(), forced[1].cpu()) <= 4 * 2.0**-9
