"""The decoders' prefill attention in the attention model's kernels (sinks, gates, strided queries, groups, keys behind earlier ones) against
float64 on the values as they are: one rounding of the output to bf16 and softmax weights in bf16, 2^-9 each over many keys."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[flash_rows] {msg}", flush=True)


def _want(q, k, v, off, sink, gate, scale, H, G, counts, pos):
    out, at = torch.empty((q.shape[0], H, 128), dtype=torch.float64, device="cuda"), 0
    for s, (n, p) in enumerate(zip(counts, pos)):
        o, L = int(off[s]), n + p
        kk, vv = (t[o:o + L].double().view(L, G, 128).repeat_interleave(H // G, 1) for t in (k, v))
        seen = torch.arange(L, device="cuda")[None, :] <= torch.arange(p, L, device="cuda")[:, None]
        for h in range(H):
            sc = (q[at:at + n].double().view(n, H, 128)[:, h] @ kk[:, h].t() * scale).masked_fill_(~seen, -torch.inf)
            m = sc.amax(1, keepdim=True)
            m = m if sink is None else m.clamp(min=float(sink[h]))
            e = (sc - m).exp()
            out[at:at + n, h] = e @ vv[:, h] / (e.sum(1, keepdim=True) + (0 if sink is None else (sink[h].double() - m).exp()))
        at += n
    out = out if gate is None else out * torch.sigmoid(gate.double())[:, :, None]
    return out.view(q.shape[0], -1)


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("H,G,counts,pos,sinks,gated", [
    (4, 4, [513], [0], True, False), (8, 1, [600], [0], False, True), (4, 2, [512, 1, 700, 64], [0, 900, 65, 3], True, True),
    (8, 2, [520, 33], [1, 0], False, False), (2, 2, [1029], [130], True, True)])
def test_against_float64(form, H, G, counts, pos, sinks, gated):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import _lib, seq_ops
    _say(f"form={form} H={H} G={G} counts={counts} pos={pos} sinks={sinks} gated={gated}")
    g = torch.Generator(device="cuda").manual_seed(H + len(counts))
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    T, n, L = sum(counts), len(counts), [c + p for c, p in zip(counts, pos)]
    q = rnd(T, H * 128 + 24).bfloat16()[:, 16:16 + H * 128]
    k, v = rnd(sum(L) + 5, G * 128).bfloat16(), rnd(sum(L) + 5, G * 128).bfloat16()
    off = torch.tensor([0] + L[:-1]).cumsum(0).cuda() + 5
    # sinks from far below every score to far above
    sink = torch.linspace(-200.0, 200.0, H, device="cuda") if sinks else None
    gate = rnd(T, H + 8).bfloat16()[:, :H] if gated else None
    batch = seq_ops.StepBatch(counts, list(range(n)), pos, "cuda")
    assert seq_ops.takes_flash_rows(q, k, v, H, G, 128, 128, 0, batch)
    try:
        _lib.load().msa_flash_set_form(form)
        got = seq_ops.flash(q, k, v, off, sink, 0.09, H, batch, G, 2048, gate)
    finally:
        _lib.load().msa_flash_set_form(0)
    want = _want(q, k, v, off, sink, gate, 0.09, H, G, counts, pos)
    assert ((got.double() - want).norm() / want.norm()).item() < 5e-3
    for h in range(H):                                   # every head by itself: a large sink leaves next to nothing
        a, b = got.double()[:, 128 * h:128 * h + 128], want[:, 128 * h:128 * h + 128]
        assert (a - b).norm() <= 5e-3 * b.norm() + 1e-30


def test_what_stays_with_the_general_kernel():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import seq_ops
    q, k = torch.zeros((600, 512), device="cuda").bfloat16(), torch.zeros((600, 512), device="cuda").bfloat16()
    batch = seq_ops.StepBatch([600], [0], [0], "cuda")
    ok = lambda chunk=0, q=q, k=k, b=batch, D=128: seq_ops.takes_flash_rows(q, k, k, 512 // D, 512 // D, D, D, chunk, b)
    assert ok() and ok(600)
    assert not ok(599) and not ok(D=64) and not ok(b=seq_ops.StepBatch([300, 300], [0, 1], [0, 0], "cuda"))
    assert not ok(k=torch.zeros((600, 520), device="cuda").bfloat16()[:, :512])
    assert not ok(q=torch.zeros((600, 516), device="cuda").bfloat16()[:, :512])
    assert not ok(b=seq_ops.StepBatch([560] + [1] * 40, list(range(41)), [0] * 41, "cuda"))     # one long portion among short ones
