"""Attention of single rows that prepares its queries, and appends its key and value, itself: against the two launches.

The norms' sums of squares are formed in another order (1e-6 of them), so a prepared value may round to the neighbouring bf16 one, in a few of
a thousand; the scores then differ by up to 2^-8 of a term, and so little of the outputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(lens, H, G, D, E, own, cap, seed):
    from msa_amd import seq_ops
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    B = len(lens)
    proj = rnd(B, H * D + G * D + G * E + H + 8).bfloat16()
    cut = lambda at, n: proj[:, at:at + n]
    q, k, v, gate = cut(0, H * D), cut(H * D, G * D), cut(H * D + G * D, G * E), cut(H * D + G * D + G * E, H)
    batch = seq_ops.StepBatch([1] * B, list(range(B, 0, -1)), [n - 1 for n in lens], "cuda:0")
    caches = [rnd(B + 2, cap, G, D).bfloat16(), rnd(B + 2, cap, G, E).bfloat16()]
    for i, n in enumerate(lens):                                     # what stands behind the keys, the row's own place included, counts nothing
        for c in caches:
            c[B - i, n - (1 if own else 0):] = float("nan")
    norms = [1 + 0.1 * rnd(D) for _ in range(2)]
    return seq_ops, batch, q, {"k": k, "v": v, "k_norm": norms[1]} if own else {}, gate, caches, norms[0]


@pytest.mark.parametrize("lens,H,G,D,E,pairs,chunk,own", [((1,), 16, 4, 128, 128, 64, 0, True), ((4097,), 16, 4, 128, 128, 64, 8192, True),
                                                          ((32, 33, 31, 1, 64, 65, 700), 32, 8, 128, 128, 64, 0, True), ((2000,) * 16, 32, 8, 128, 128, 64, 0, True),
                                                          ((129, 128, 127, 1025), 8, 8, 128, 128, 64, 128, True), ((300, 17), 40, 2, 128, 128, 64, 0, True),
                                                          ((500, 3), 32, 8, 128, 128, 64, 0, False), ((90, 33), 8, 4, 64, 128, 32, 0, True),
                                                          ((90, 33), 8, 4, 128, 128, 32, 0, True)])
def test_single_rows(lens, H, G, D, E, pairs, chunk, own):
    """Heads of 64 and those that are rotated by half take the launch of their own: the same results bit for bit."""
    cap = max(lens) + (0 if len(lens) == 1 else 9)
    seq_ops, batch, q, kv, gate, caches, q_norm = _operands(lens, H, G, D, E, own, cap, len(lens) + H)
    freqs = (10000.0 ** -(torch.arange(pairs, dtype=torch.float64) / pairs)).cuda()
    two, one = [c.clone() for c in caches], [c.clone() for c in caches]
    print(f"[rope_decode] {lens[:4]} H={H} G={G} D={D} chunk={chunk} own={own}", flush=True)
    want = seq_ops.kv_attn(seq_ops.qk_rope_append(q, q_norm, freqs, 1e-5, *two, batch, **kv), *two, D ** -0.5, batch, chunk, gate)
    for _ in range(2):
        got = seq_ops.rope_kv_attn(q, q_norm, freqs, 1e-5, *one, D ** -0.5, batch, chunk, gate, **kv)
        assert got.isfinite().all() and want.isfinite().all()
        if D == 64 or 2 * pairs < D:
            assert torch.equal(got, want)
        assert ((got.float() - want.float()).norm() / want.float().norm()).item() < 4e-3
        assert torch.equal(one[1].isnan(), two[1].isnan()) and torch.equal(one[1].nan_to_num(), two[1].nan_to_num())
        a, b = one[0].float(), two[0].float()
        assert torch.equal(a.isnan(), b.isnan())
        a, b = a.nan_to_num(), b.nan_to_num()
        step = torch.ldexp(torch.ones_like(b), torch.frexp(b).exponent - 8)
        assert ((a - b).abs() <= step).all()
        if own:
            rows = torch.tensor([n - 1 for n in lens]), torch.tensor(list(range(len(lens), 0, -1)))
            assert (a[rows[1], rows[0]] != b[rows[1], rows[0]]).float().mean() < 1e-2


def test_refused():
    seq_ops, batch, q, kv, gate, caches, q_norm = _operands((5,), 8, 4, 128, 128, True, 8, 1)
    freqs = torch.zeros(64, dtype=torch.float64, device="cuda")
    for bad in (dict(freqs=freqs.float()), dict(q=q[:, :-128]), dict(k=kv["k"][:, :-8]), dict(gate=gate[:, :-1])):
        args = {**dict(q=q, q_norm=q_norm, freqs=freqs, eps=1e-5, k_cache=caches[0], v_cache=caches[1], scale=0.1, batch=batch, gate=gate), **kv, **bad}
        with pytest.raises(Exception):
            seq_ops.rope_kv_attn(**args)
