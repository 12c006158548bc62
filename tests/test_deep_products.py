"""Deep plain products of fewer rows than half a round of whole tiles: which ones the tiles take, and what they give."""
import pytest
import torch

from msa_amd import ops, seq_ops


class _On:
    """An operand as the routing sees it."""
    dtype, is_cuda, requires_grad, device = torch.bfloat16, True, False, torch.device("cuda:0")

    def __init__(self, *shape):
        self.shape = shape

    dim = lambda self: len(self.shape)
    numel = lambda self: self.shape[0] * self.shape[1]
    is_contiguous = lambda self: True
    stride = lambda self, i: (self.shape[1], 1)[i]
    data_ptr = lambda self: 4096


@pytest.mark.parametrize("T,K,N,taken", [(448, 8192, 2560, True), (447, 8192, 2560, False), (448, 8128, 2560, False), (2816, 9728, 2560, True),
                                         (2817, 9728, 2560, False), (513, 8192, 1536, False), (1793, 8192, 4096, False), (1536, 8192, 4096, True),
                                         (500, 8192, 2568, False), (500, 32832, 2560, False)])
def test_line(T, K, N, taken):
    assert ops.tile_linear_ok(_On(T, K), _On(N, K), end=False) == taken
    assert not ops.tile_linear_ok(_On(T, K), _On(N, K)) or T * N >= ops.TILE_MIN


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,N", [(448, 8192, 2560), (513, 9728, 2560), (2340, 9728, 2560), (2600, 8256, 2560)])
def test_products(T, K, N):
    """One rounding of the result: 1.7e-3 over many values."""
    print(f"[case] deep product {T} x {K} x {N}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((T, K + 32), generator=g, device="cuda").bfloat16()[:, 8:K + 8]
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    assert ops.tile_linear_ok(x, w, end=False)
    want, got = x.float() @ w.float().t(), ops.tile_linear(x, w)
    assert ((got.float() - want).norm() / want.norm()).item() < 3e-3
    # a step's products of fewer rows have another form in front of this one
    assert torch.equal(seq_ops.product(x, w), got if T >= ops.FLOW_FIRST else ops.flow_linear(x, w))
    lin = torch.nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16)
    lin.weight.data.copy_(w)
    with torch.no_grad():
        assert torch.equal(ops.linear(lin, x.contiguous()), got)
