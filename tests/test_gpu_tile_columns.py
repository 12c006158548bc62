"""Products of blocks whose last columns leave the 256 x 256 tiles for the smaller ones: every end on both sides of the cut, inside wider
tensors, against a float32 product."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows, depth, columns): 32, 8 and 256 columns behind eight or 24 tiles' width, rows that are no multiple of a tile, no whole round in front,
# as many behind as stay in tiles, and a depth that is not cut
SHAPES = [(8192, 1024, 6176), (8192, 1024, 2056), (8192, 1024, 2304), (8191, 1024, 2304), (6001, 1024, 3072), (4096, 2560, 4608), (4095, 1024, 4240), (4096, 1024, 4352),
          (8192, 1024, 2048), (8192, 1024, 3072), (8192, 960, 2304)]


@pytest.mark.parametrize("T,K,N", SHAPES)
@pytest.mark.parametrize("end", ["store", "gelu_before", "gelu_behind", "gelu_odd", "glu"])
def test_ends(T, K, N, end):
    from msa_amd import ops
    if end == "glu" and N % 16:
        return
    g = torch.Generator(device="cuda").manual_seed(T + N)
    x = torch.randn((T, K + 8), generator=g, device="cuda").bfloat16()[:, :K]                  # a column range of a wider tensor
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    want = x.float() @ w.float().t()
    kw = {}
    if end == "glu":
        kw = {"glu": (1.5, 1.702, 1.0)}
        gate, up = want[:, 0::2].clamp(max=1.5), want[:, 1::2].clamp(-1.5, 1.5)
        want = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
    elif end != "store":
        n = {"gelu_before": 1152, "gelu_behind": N - N % 128, "gelu_odd": N}[end]
        kw = {"gelu_n": n}
        want[:, :n] = torch.nn.functional.gelu(want[:, :n], approximate="tanh")
    wide = torch.full((T + 2, want.shape[1] + 16), 7.0, device="cuda", dtype=torch.bfloat16)
    out = wide[1:-1, 8:-8]
    ops.tile_linear(x, w, out=out, **kw)
    got = out.float()
    # one rounding of the result, and of a gated end's sums: 2^-8 of either at most
    assert ((got - want).norm() / want.norm()).item() < 4e-3
    assert ((got - want).abs() <= 2 ** -6 * want.abs() + 2 ** -6).all()
    out.fill_(7.0)
    assert bool((wide == 7.0).all())
