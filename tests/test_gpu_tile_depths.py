"""Products whose last columns may leave the 256 x 256 tiles, on both sides of the greatest depth at which they do, against a float32 product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [2560, 2624, 4096])
@pytest.mark.parametrize("T,N", [(8192, 2304), (8192, 6176), (4096, 4608)])
def test_depths(T, N, K):
    from msa_amd import ops
    g = torch.Generator(device="cuda").manual_seed(K + N)
    x = torch.randn((T, K), generator=g, device="cuda").bfloat16()
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    want = x.float() @ w.float().t()
    got = ops.tile_linear(x, w).float()
    # one rounding of the result
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2 ** -10).all()
