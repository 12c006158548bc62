"""Products of some hundred tokens in one round of mid-sized tiles (``ops.flow_linear`` and its C entry) against fp32: every tile whole and
ragged, pieces of K, depths of one K tile and fewer than the ring holds, row strides, the ends, the rule that takes a call there, a captured call.

One rounding to bf16 leaves a relative error of up to 2^-9 a value, 1.7e-3 over many; the gated unit and gelu round the product, then
the result, the gate's part passed on by a factor of up to 1.3 over many values: sqrt(1 + 1 + 1.3^2) of one."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu
TOL, TOL_END = 3e-3, 4e-3


def _operands(T, K, N, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((T, K), generator=g, device="cuda").bfloat16()
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    return x, w, x.float() @ w.float().t()


def _err(got, want):
    return ((got.float() - want).norm() / want.norm()).item()


def _flow(x, w, pieces=True, **end):
    """The C entry, with the workspace it asks for (behind which nothing is written) or none."""
    from msa_amd import _lib
    lib, (T, K), N = _lib.load(), x.shape, w.shape[0]
    glu, gelu_n = end.get("glu"), end.get("gelu_n", 0)
    mode = _lib.TILE_GLU if glu else _lib.TILE_GELU if gelu_n else _lib.TILE_STORE
    out = torch.full((T + 1, (N // 2 if glu else N) + 8), 7.0, device="cuda").bfloat16()
    need = lib.msa_flow_workspace_bytes(T, K, N, mode) if pieces else 0
    ws = torch.full((need + 64,), 9, dtype=torch.uint8, device="cuda")
    e = _lib.TileEnd(mode, gelu_n, *(glu or (0.0, 0.0, 0.0)))
    _lib.check(lib.msa_flow_linear(x.data_ptr(), x.stride(0), T, K, w.data_ptr(), N, C.byref(e), out.data_ptr(), out.shape[1], ws.data_ptr() if need else None, need,
                                   torch.cuda.current_stream().cuda_stream), "msa_flow_linear")
    torch.cuda.synchronize()
    assert (out[T] == 7).all() and (out[:, -8:] == 7).all() and (ws[need:] == 9).all()
    return out[:T, :-8], need


# 64 x 32 tiles, the last two in 3 and 6 pieces; 64 x 64, in 4; 64 x 96, in 5; 64 x 128, in 6; 128 x 96; 128 x 128, in 6; 128 x 160, in 5; 192 x 128;
# 192 x 160; 192 x 192; 256 x 128, in 3
SHAPES = [(1, 64, 16), (31, 128, 80), (33, 320, 1040), (1, 1408, 64), (17, 4864, 2000), (34, 128, 8272), (33, 3520, 3280), (33, 64, 8224), (67, 2816, 2624),
          (97, 64, 8208), (113, 4160, 2128), (131, 192, 8544), (573, 1024, 4080), (195, 64, 11136), (220, 8704, 2448), (263, 128, 10960), (144, 5952, 5936),
          (326, 64, 11040), (783, 192, 9280), (517, 256, 13232), (402, 64, 12400), (1000, 9728, 2560)]


@pytest.mark.parametrize("T,K,N", SHAPES)
def test_products(T, K, N):
    print(f"[flow_gemm] T={T} K={K} N={N}", flush=True)
    x, w, want = _operands(T, K, N, 1)
    wide = torch.full((T + 1, K + 24), float("nan"), device="cuda").bfloat16()     # what lies beside x is not read
    wide[:T, 8:K + 8] = x
    got, need = _flow(wide[:T, 8:K + 8], w)
    assert _err(got, want) < TOL
    if need:
        whole, none = _flow(x, w, pieces=False)
        assert none == 0 and _err(whole, want) < TOL
    n = (N // 2 + 7) // 8 * 8
    got, _ = _flow(x, w, gelu_n=n)
    assert _err(got[:, :n], torch.nn.functional.gelu(want[:, :n], approximate="tanh")) < TOL_END
    assert _err(got[:, n:], want[:, n:]) < TOL
    limit, alpha, shift = 1.5, 1.702, 1.0
    gate, up = want[:, 0::2].clamp(max=limit), want[:, 1::2].clamp(-limit, limit)
    assert _err(_flow(x, w, glu=(limit, alpha, shift))[0], gate * torch.sigmoid(alpha * gate) * (up + shift)) < TOL_END


def test_more_than_a_round():
    x, w, want = _operands(2000, 64, 19456, 2)
    assert _err(_flow(x, w)[0], want) < TOL


def test_route(monkeypatch):
    from msa_amd import ops, seq_ops
    taken, inner = [], ops.flow_linear
    monkeypatch.setattr(ops, "flow_linear", lambda x, w, **k: (lambda y: (taken.append(y is not None), y)[1])(inner(x, w, **k)))
    for T, K, N, here in ((450, 2560, 2560, True), (100, 9728, 2560, True), (700, 9728, 2560, True), (1000, 9728, 2560, False), (1000, 1024, 6144, True), (1500, 1024, 6144, True),
                          (16, 9728, 2560, False), (159, 2560, 12288, False), (2305, 1024, 3072, False), (64, 1024, 1024, False), (450, 2592, 2560, False)):
        print(f"[flow_gemm] route T={T} K={K} N={N}", flush=True)
        x, w, want = _operands(T, K, N, 3)
        taken.clear()
        assert _err(seq_ops.product(x, w), want) < TOL and any(taken) == here
        if here:
            taken.clear()
            gelu = seq_ops.product_gelu(x, w, 64)
            assert _err(gelu[:, 64:], want[:, 64:]) < TOL and any(taken)
            taken.clear()
            seq_ops.product_glu(x, w, 7.0)
            assert any(taken)
    x, w, want = _operands(450, 2560, 2560, 4)
    odd = torch.empty(450 * 2560 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(450, 2560).copy_(x)
    for a, b in ((x, w.clone().requires_grad_()), (x.t().contiguous().t(), w), (x, w.t().contiguous().t()), (odd, w)):
        taken.clear()
        assert _err(seq_ops.product(a, b).detach(), want) < TOL and not any(taken)      # gradients, and operands that the kernel does not read
    assert ops.flow_linear(x.cpu(), w) is None


@pytest.mark.parametrize("T,K,N", [(64, 1024, 1024), (450, 2560, 2560), (1536, 8192, 2560)])      # block_linear's, flow_linear's and tile_linear's
def test_more_than_values(T, K, N):
    """A tangent, a batch of vmap, and what a class or a mode sees of a call are torch's own product's."""
    import torch.autograd.forward_ad as fwd
    from torch.utils._python_dispatch import TorchDispatchMode
    from msa_amd import seq_ops
    x, w, want = _operands(T, K, N, 6)
    t = torch.randn(x.shape, device="cuda").bfloat16()
    turned = t.float() @ w.float().t()
    with fwd.dual_level():
        for a in (fwd.make_dual(x, t), fwd.make_dual(x[:, :], t)):
            y, tangent = fwd.unpack_dual(seq_ops.product(a, w))
            assert _err(y, want) < TOL and tangent is not None and _err(tangent, turned) < TOL
    y, tangent = torch.func.jvp(lambda x: seq_ops.product(x, w), (x,), (t,))
    assert _err(y, want) < TOL and _err(tangent, turned) < TOL
    both = torch.vmap(lambda x: seq_ops.product(x, w))(torch.stack([x, t]))
    assert _err(both[0], want) < TOL and _err(both[1], turned) < TOL

    class Own(torch.Tensor):
        pass

    class Seen(TorchDispatchMode):
        calls = 0

        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            Seen.calls += 1
            return f(*args, **(kwargs or {}))

    assert type(seq_ops.product(x.as_subclass(Own), w)) is Own
    with Seen():
        seq_ops.product(x, w)
    assert Seen.calls
    assert _err(seq_ops.product(x, torch.nn.Parameter(w, requires_grad=False)), want) < TOL


@pytest.mark.parametrize("T,K,N", [(450, 2560, 2560), (300, 9728, 2560)])
def test_captured(T, K, N):
    from msa_amd import ops
    x, w, want = _operands(T, K, N, 5)
    out = ops.flow_linear(x, w)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = ops.flow_linear(x, w)
    for _ in range(3):
        held.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(held, out)
        torch.mm(x, w.t())
    assert _err(out, want) < TOL


def test_refused():
    from msa_amd import _lib
    lib = _lib.load()
    x, w, _ = _operands(32, 128, 64, 6)
    out = torch.empty((32, 64), dtype=torch.bfloat16, device="cuda")
    e = _lib.TileEnd(_lib.TILE_STORE, 0, 0.0, 0.0, 0.0)
    ok = dict(x=x.data_ptr(), ldx=128, T=32, K=128, w=w.data_ptr(), N=64, end=C.byref(e), out=out.data_ptr(), ldo=64, ws=None, need=0, st=None)
    for bad in (dict(x=None), dict(T=0), dict(K=96), dict(N=60), dict(ldx=120), dict(ldx=132), dict(ldo=56), dict(x=x.data_ptr() + 2), dict(end=None),
                dict(end=C.byref(_lib.TileEnd(_lib.TILE_ADD, 0, 0.0, 0.0, 0.0))), dict(end=C.byref(_lib.TileEnd(_lib.TILE_GELU, 12, 0.0, 0.0, 0.0)))):
        assert lib.msa_flow_linear(*{**ok, **bad}.values()) != 0
