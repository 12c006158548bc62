"""The latents of a step's rows appended beside the products of its queries: the same as the two launches, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,heads,dim,rank", [((1,), 16, 128, 256), ((1,) * 16, 32, 128, 512), ((3, 1, 7), 2, 64, 72), ((1, 1), 1, 128, 64), ((2, 14), 200, 8, 8),
                                                   ((1,) * 5, 1, 2048, 4096), ((4, 2), 3, 40, 20)])
def test_appended_beside_products(counts, heads, dim, rank):
    """(1, 2048) takes the weight ring and (4, 2) latents that are no whole vectors, each in launches of their own."""
    from msa_amd import seq_ops
    g = torch.Generator(device="cuda").manual_seed(rank)
    T = sum(counts)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    proj = rnd(T, heads * dim + rank + 8).bfloat16() if rank % 8 == 0 else rnd(T, heads * dim + 24).bfloat16()
    q, lat = proj[:, :heads * dim], proj[:, heads * dim:heads * dim + rank]
    w, norm = (rnd(heads * rank, dim) * dim ** -0.5).bfloat16(), 1 + 0.1 * rnd(rank)
    n, cap = len(counts), 40
    at = [5 * i for i in range(n)]
    at[-1] = cap - counts[-1]                                            # up to the last row
    batch = seq_ops.StepBatch(list(counts), list(range(n, 0, -1)), [a % (cap - counts[i] + 1) for i, a in enumerate(at)], "cuda:0")
    caches = [torch.full((n + 2, cap, rank), 3.0, device="cuda").bfloat16() for _ in range(2)]
    seq_ops.latent_append(lat, norm, 1e-5, caches[0], batch)
    want = seq_ops.rows_linear(q, w, groups=heads)
    for _ in range(2):
        got = seq_ops.rows_linear_append(q, w, heads, lat, norm, 1e-5, caches[1], batch)
        assert torch.equal(got, want) and torch.equal(*caches)


def test_refused():
    from msa_amd import seq_ops
    batch = seq_ops.StepBatch([1], [0], [7], "cuda:0")
    z = lambda *s, t=torch.bfloat16: torch.zeros(s, dtype=t, device="cuda")
    ok = dict(x=z(1, 256), w=z(128, 128), groups=2, latents=z(1, 64), norm=z(64, t=torch.float32), eps=1e-5, cache=z(1, 8, 64), batch=batch)
    seq_ops.rows_linear_append(**ok)
    for bad in (dict(latents=z(1, 64, t=torch.float32)), dict(latents=z(2, 64)), dict(norm=z(64)), dict(cache=z(1, 7, 64)), dict(cache=z(1, 8, 72)), dict(x=z(1, 128)),
                dict(x=z(17, 256))):
        with pytest.raises(Exception):
            seq_ops.rows_linear_append(**{**ok, **bad})
