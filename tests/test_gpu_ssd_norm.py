"""The state-space recurrence with the norm of its output in the launch that makes it, against the two launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,H,P,N,G", [((4096,), 32, 64, 128, 8), ((4001, 4500, 700, 1), 32, 64, 128, 8), ((8190,), 8, 32, 64, 4), ((2100,) * 4, 40, 8, 32, 8),
                                            ((2070, 2048, 33, 2000, 190), 10, 56, 120, 5),
                                            ((4000, 4100), 20, 64, 96, 4), ((2500, 2600, 100), 25, 56, 64, 5)])
def test_folded_norm(counts, H, P, N, G):
    """The same bits as the two launches: their squares are added in the same order.  (32 lanes to a row, the models', then 8, 5, 14, 40 and 35:
    halves of a wavefront and whole ones.)"""
    from msa_amd import _lib, seq_ops
    g = torch.Generator(device="cuda").manual_seed(sum(counts))
    T, inner = sum(counts), H * P
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    proj = rnd(T, 2 * inner + 2 * G * N + (H + 15) // 8 * 8).bfloat16()
    z, xbc, dt = proj[:, :inner], proj[:, inner:2 * inner + 2 * G * N], proj[:, 2 * inner + 2 * G * N:2 * inner + 2 * G * N + H]
    small = (rnd(H) - 4.0, torch.rand(H, generator=g, device="cuda"), rnd(H))
    w = 1 + 0.1 * rnd(inner)
    batch = seq_ops.StepBatch(list(counts), list(range(len(counts), 0, -1)), [0] * len(counts), "cuda:0")
    states = [0.1 * torch.ones((len(counts) + 2, H, N, P), device="cuda") for _ in range(2)]
    assert _lib.load_seq().msa_seq_ssd_norm_folds(batch.max_rows, batch.n_seq, H, P, N, G, G)
    print(f"[ssd_norm] {counts} H={H} P={P} N={N} G={G}", flush=True)
    want = seq_ops.group_rmsnorm(seq_ops.ssd(xbc, z, dt, *small, H, P, N, G, states[0], batch, True), w, G, 1e-5)
    got = seq_ops.ssd_norm(xbc, z, dt, *small, H, P, N, G, states[1], batch, True, w, G, 1e-5)
    assert torch.equal(got, want) and torch.equal(*states)


def test_what_is_not_folded():
    from msa_amd import _lib
    folds = _lib.load_seq().msa_seq_ssd_norm_folds
    assert folds(8192, 1, 32, 64, 128, 8, 8)
    for args in ((1024, 1, 32, 64, 128, 8, 8), (8192, 1, 80, 64, 128, 8, 8), (8192, 1, 32, 128, 128, 8, 8), (8192, 1, 32, 64, 136, 8, 8), (8192, 1, 32, 64, 128, 8, 4),
                 (8192, 1, 32, 60, 128, 8, 8), (0, 1, 32, 64, 128, 8, 8)):
        assert not folds(*args)
