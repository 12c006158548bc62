"""What a decode step's first launches and the delta rule's folded low rank do, at the edges of their sizes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[decode_starts] {msg}", flush=True)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import ops
    return ops


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape,W", [((1, 1), 8), ((16, 1), 2560), ((3, 7), 2056), ((70001,), 16)])
def test_embed_rows(ops, dtype, shape, W):
    _say(f"embed_rows {shape} W={W} {dtype}")
    table = torch.randn((37, W), device="cuda").to(dtype)
    tok = torch.randint(0, 37, shape, device="cuda")
    assert torch.equal(ops.embed_rows(table, tok), table[tok])
    rows, wide = ops.embed_rows(table, tok - 37, f32=True, wrap=True)
    assert torch.equal(rows, table[tok]) and torch.equal(wide, table[tok].float())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,W", [([1], 8), ([1] * 16, 2560), ([5, 1, 300], 1024), ([7, 2], 30), ([600], 72)])
def test_embed_norm_is_lookup_and_residual_norm(ops, dtype, counts, W):
    _say(f"embed_norm counts={counts} W={W} {dtype}")
    from msa_amd import seq_ops
    n, T = len(counts), sum(counts)
    table = torch.randn((50, W), device="cuda").to(dtype)
    tok = torch.randint(-50, 50, (T,), device="cuda")
    batch = seq_ops.StepBatch(counts, list(range(n))[::-1], [3] * n, "cuda")
    vec = lambda: torch.randn(W, device="cuda")
    norm, shift, prev = seq_ops.DynTanhNorm(vec(), vec(), 0.7), vec(), torch.randn((n, W), device="cuda")
    prev2 = prev.clone()
    x, h, hs = seq_ops.embed_norm(tok, table, batch, norm, shift, prev)
    x2, h2, hs2 = seq_ops.residual_norm(table[tok].float(), batch, dtype, norm=norm, shift=shift, prev=prev2)
    for a, b in ((x, x2), (h, h2), (hs, hs2), (prev, prev2)):
        assert torch.equal(a, b)
    x, h, hs = seq_ops.embed_norm(tok, table, batch, norm)
    assert torch.equal(x, x2) and torch.equal(h, h2) and hs is None


@pytest.mark.parametrize("B,H,G,D,E,R", [(1, 16, 16, 64, 128, 64), (16, 4, 2, 128, 128, 128), (3, 2, 1, 16, 8, 8), (2, 3, 3, 24, 40, 136),
                                         (5, 4, 4, 128, 64, 264), (1, 1, 1, 1, 1, 16), (70, 2, 1, 100, 120, 48), (16, 32, 16, 128, 128, 128)])
def test_delta_step_with_its_low_rank(ops, B, H, G, D, E, R):
    """Against the fp32 rule on the products in fp32: the output's own rounding to bf16 (2^-9), the state's sums in another order."""
    _say(f"delta_step B={B} H={H} G={G} D={D} E={E} R={R}")
    from msa_amd import seq_ops
    g = torch.Generator(device="cuda").manual_seed(B + D)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    pad = lambda n: -(-n // 8) * 8
    n_a = pad(H * D)
    ch = 2 * G * D + H * E
    proj = rnd(B, pad(ch) + 2 * pad(R) + pad(H)).bfloat16()
    qkv, a_low, g_low = proj[:, :ch], proj[:, pad(ch):pad(ch) + R], proj[:, pad(ch) + pad(R):pad(ch) + pad(R) + R]
    b = proj[:, pad(ch) + 2 * pad(R):][:, :H]
    w = (rnd(n_a + H * E, R) * R ** -0.5).bfloat16()
    A_log, bias, norm = rnd(H).sigmoid(), rnd(H * D) - 2, 1 + 0.1 * rnd(E)
    state = 0.3 * rnd(B, H, D, E)
    state2 = state.clone()
    batch = seq_ops.StepBatch([1] * B, list(range(B)), [9] * B, "cuda")
    got = seq_ops.delta_step(qkv, a_low, g_low, w, n_a, b, A_log, bias, norm, 1e-5, H, G, D, E, state, batch)
    a, gate = a_low.float() @ w[:H * D].float().t(), g_low.float() @ w[n_a:].float().t()
    want = seq_ops.delta(qkv.float().contiguous(), a, b.float().contiguous(), gate, A_log, bias, norm, 1e-5, H, G, D, E, state2, batch)
    assert ((got.float() - want).norm() / want.norm()).item() < 3e-3
    assert ((state - state2).norm() / state2.norm()).item() < 1e-5
