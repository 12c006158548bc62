"""Products of few tokens (``ops.block_linear``, behind ``seq_ops.product`` and its forms) against fp32: edges of every tile, depths of one
K tile and of more than are on their way, row strides, the ends, the rule that takes a call there, and a captured call.

One rounding to bf16 leaves a relative error of up to 2^-9 a value, 1.7e-3 over many; the gated unit and gelu round the product, then
the result, the gate's part passed on by a factor of up to 1.3 over many values: sqrt(1 + 1 + 1.3^2) of one."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL, TOL_END = 3e-3, 4e-3


def _say(msg):
    print(f"[block_gemm] {msg}", flush=True)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import ops
    return ops


def _operands(T, K, N, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((T, K), generator=g, device="cuda").bfloat16()
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    return x, w, x.float() @ w.float().t()


def _err(got, want):
    return ((got.float() - want).norm() / want.norm()).item()


# 64 x 32 tiles: the first five; 64 x 64: the next two; 128 x 64: the next two; 128 x 128: the others
SHAPES = [(1, 64, 16), (31, 128, 80), (33, 192, 1040), (65, 320, 1024), (300, 2560, 1024), (573, 1024, 1040), (300, 1088, 2064), (2048, 1024, 1072),
          (573, 576, 3072), (573, 1024, 4080), (1990, 192, 6176), (6001, 128, 4096)]


@pytest.mark.parametrize("T,K,N", SHAPES)
def test_products(ops, T, K, N):
    _say(f"T={T} K={K} N={N}")
    x, w, want = _operands(T, K, N, 1)
    wide = torch.full((T + 1, K + 24), float("nan"), device="cuda").bfloat16()     # what lies beside x is not read
    wide[:T, 8:K + 8] = x
    assert _err(ops.block_linear(wide[:T, 8:K + 8], w), want) < TOL
    n = (N // 2 + 7) // 8 * 8
    got = ops.block_linear(x, w, gelu_n=n)
    assert _err(got[:, :n], torch.nn.functional.gelu(want[:, :n], approximate="tanh")) < TOL_END
    assert _err(got[:, n:], want[:, n:]) < TOL
    limit, alpha, shift = 1.5, 1.702, 1.0
    gate, up = want[:, 0::2].clamp(max=limit), want[:, 1::2].clamp(-limit, limit)
    assert _err(ops.block_linear(x, w, glu=(limit, alpha, shift)), gate * torch.sigmoid(alpha * gate) * (up + shift)) < TOL_END


def test_route(ops, monkeypatch):
    from msa_amd import seq_ops
    taken = []
    inner = ops.block_linear
    monkeypatch.setattr(ops, "block_linear", lambda x, w, **k: (taken.append(tuple(x.shape)), inner(x, w, **k))[1])
    for T, K, N, here in ((64, 1024, 1024, True), (6001, 128, 4096, True), (8192, 256, 2048, False), (300, 2560, 8192, False), (40, 96, 64, False),
                          (40, 64, 72, False)):
        _say(f"route T={T} K={K} N={N}")
        x, w, want = _operands(T, K, N, 2)
        taken.clear()
        assert _err(seq_ops.product(x, w), want) < TOL and bool(taken) == here
        seq_ops.product_gelu(x, w, 16)
        if N % 16 == 0:
            seq_ops.product_glu(x, w, 7.0)
        assert len(taken) == (3 if here else 0)
    x, w, want = _operands(40, 64, 64, 3)
    taken.clear()
    for y in (seq_ops.product(x, w.clone().requires_grad_()), seq_ops.product(x.t().contiguous().t(), w), seq_ops.product(x[:, :64], w.t().contiguous().t())):
        assert _err(y.detach(), want) < TOL
    assert not taken                                     # gradients, and operands that the kernel does not read


def test_captured(ops):
    x, w, want = _operands(300, 1024, 2304, 4)
    out = ops.block_linear(x, w)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = ops.block_linear(x, w)
    for _ in range(3):
        held.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(held, out)
    assert _err(out, want) < TOL


def test_route_of_captured_calls(ops):
    """A captured call pays for no host: the line is the kernels' own."""
    shapes = {(64, 1024, 1024): True, (17, 1024, 6176): True, (1000, 2048, 1024): True, (32, 2560, 2560): False, (1500, 128, 4096): False,
              (573, 1024, 8192): False}
    operands = {s: _operands(*s, 5) for s in shapes}
    assert all(ops.block_linear_ok(x, w) for x, w, _ in operands.values())
    graph, took = torch.cuda.CUDAGraph(), {}
    keep = torch.zeros(1, device="cuda")
    with torch.cuda.graph(graph):
        keep.add_(1)
        for s, (x, w, _) in operands.items():
            took[s] = ops.block_linear_ok(x, w)
    assert took == shapes
