"""Products of a block of tokens (``ops.tile_linear``) against fp32: edges of the 256 x 256 tiles, one K tile and many, tiles multiplied in
pieces, row strides, and every end (store, add, silu-mul, clamped unit, gelu; the heads' norm and rotary are tested with ``qkv_proj``).

One rounding to bf16 leaves a relative error of up to 2^-9 a value, 1.7e-3 over many; the fp32 sums are far below it.  The gated ends and
gelu may round the sums before and the result behind: three roundings for a gated unit, the gate's passed on by a factor of up to 1.3
over many values, sqrt(1 + 1 + 1.3^2) of one."""
import pytest
import torch

from msa_amd._lib import MsaError

pytestmark = pytest.mark.gpu
TOL = 3e-3
TOL_END = 4e-3


def _say(msg):
    print(f"[tile_gemm] {msg}", flush=True)


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


# several tiles a workgroup, their ends under the next one's steps from K = 704 on: the last three
# (2100 x 4096 x 2576: 99 tiles on 256 compute units, in pieces of K; 257 x 1024 x 16400: 130 tiles, whole)
SHAPES = [(1, 64, 8), (255, 64, 256), (256, 128, 256), (257, 192, 264), (17, 320, 1000), (300, 4096, 2048), (2100, 4096, 2576), (257, 1024, 16400),
          (6001, 704, 5144), (9000, 640, 4360), (5000, 1024, 6664)]


@pytest.mark.parametrize("T,K,N", SHAPES)
def test_store_and_add(ops, T, K, N):
    _say(f"T={T} K={K} N={N}")
    x, w, want = _operands(T, K, N, 1)
    assert _err(ops.tile_linear(x, w), want) < TOL
    # columns of wider tensors: what lies beside them stays as it was
    wide_x = torch.full((T, K + 24), float("nan"), device="cuda").bfloat16()
    wide_x[:, 8:K + 8] = x
    wide = torch.full((T + 1, N + 16), 7.0, device="cuda").bfloat16()
    out = wide[:T, 8:N + 8]
    base = torch.randn((T, N), device="cuda").bfloat16()
    out.copy_(base)
    ops.tile_linear(wide_x[:, 8:K + 8], w, out=out, add=True)
    assert _err(out, want + base.float()) < TOL
    out.fill_(7.0)
    assert bool((wide == 7.0).all())


@pytest.mark.parametrize("T,K,N", [(1, 64, 16), (129, 128, 272), (513, 256, 1040), (2100, 4096, 2592), (6001, 1024, 5136), (6001, 704, 5200)])
def test_silu_mul(ops, T, K, N):
    _say(f"silu-mul T={T} K={K} N={N}")
    x, gate, want_gate = _operands(T, K, N // 2, 2)
    up = (torch.randn((N // 2, K), device="cuda") * K ** -0.5).bfloat16()
    got = ops.tile_linear(x, ops.interleave_gate_up(gate, up), silu_mul=True)
    assert _err(got, torch.nn.functional.silu(want_gate) * (x.float() @ up.float().t())) < TOL_END


@pytest.mark.parametrize("T,K,N", [(1, 64, 16), (129, 128, 272), (2100, 4096, 2592), (6001, 1024, 5136), (6001, 704, 5200)])
def test_glu(ops, T, K, N):
    """Rows in (gate, up) pairs; sums up to 4 against a limit of 1.5, so that both are clamped."""
    _say(f"glu T={T} K={K} N={N}")
    x, w, want = _operands(T, K, N, 6)
    got = ops.tile_linear(x, w, glu=(1.5, 1.702, 1.0))
    gate, up = want[:, 0::2].clamp(max=1.5), want[:, 1::2].clamp(-1.5, 1.5)
    assert _err(got, gate * torch.sigmoid(1.702 * gate) * (up + 1.0)) < TOL_END


@pytest.mark.parametrize("T,K,N,n", [(1, 64, 8, 8), (129, 128, 264, 136), (257, 256, 512, 128), (2100, 4096, 2576, 1304), (6001, 1024, 5144, 3072), (6001, 704, 5200, 1408)])
def test_gelu(ops, T, K, N, n):
    _say(f"gelu T={T} K={K} N={N} n={n}")
    x, w, want = _operands(T, K, N, 7)
    want[:, :n] = torch.nn.functional.gelu(want[:, :n], approximate="tanh")
    assert _err(ops.tile_linear(x, w, gelu_n=n), want) < TOL_END


def test_extreme_gates(ops):
    """silu of sums far out: the exponential overflows and the product stays 0 or the sum itself."""
    x = torch.zeros((16, 64), device="cuda").bfloat16()
    x[:, 0] = torch.linspace(-3e4, 3e4, 16, device="cuda").bfloat16()
    gate, up = torch.zeros((8, 64), device="cuda").bfloat16(), torch.zeros((8, 64), device="cuda").bfloat16()
    gate[:, 0], up[:, 0] = 1.0, 1.0
    got = ops.tile_linear(x, ops.interleave_gate_up(gate, up), silu_mul=True).float()
    want = torch.nn.functional.silu(x[:, :1].float()) * x[:, :1].float()
    assert torch.allclose(got, want.expand(-1, 8), rtol=2 ** -8)


@pytest.mark.parametrize("T,front,back", [(2055, 2, 0), (700, 0, 5)])
def test_heads_in_pieces(ops, T, front, back):
    """The projection's tiles multiplied in pieces give what the one-piece call gives."""
    from msa_amd import _lib
    K, Hq, Hkv = 4096, 8, 2
    _say(f"heads T={T} front={front} back={back}")
    N = (front + Hq + 2 * Hkv + back) * 128
    x, w, _ = _operands(T, K, N, 3)
    pos = torch.arange(T, device="cuda") % 500
    nw = [1 + 0.1 * torch.randn(128, device="cuda").bfloat16() for _ in range(2)]
    rope = ops.rope_tables(500, 128, 1e6, device="cuda")
    assert _lib.load().msa_tile_workspace_bytes(T, K, N) > 0
    split = ops.qkv_proj(x, w, Hq, Hkv, pos, nw[0], nw[1], 1e-6, rope, router_front=front, router_back=back)
    whole = [torch.empty_like(t) for t in split]
    ops.check(_lib.load().msa_qkv_proj(ops.ptr(x), T, K, ops.ptr(w), Hq, Hkv, front, back, ops.ptr(pos), ops.ptr(nw[0]), ops.ptr(nw[1]), 1e-6,
                                       ops.ptr(rope[0]), ops.ptr(rope[1]), 500, *(ops.ptr(t) for t in whole), ops._stream()), "msa_qkv_proj")
    for a, b in zip(split, whole):
        assert _err(a, b.float()) < TOL


def test_refusals(ops):
    x, w, _ = _operands(64, 128, 64, 4)
    with pytest.raises(ValueError):
        ops.tile_linear(x.float(), w)
    with pytest.raises(ValueError):
        ops.tile_linear(x[:, :64], w)
    with pytest.raises(ValueError):
        ops.tile_linear(x, w, add=True)
    with pytest.raises(MsaError):
        ops.tile_linear(x[:, :96].contiguous(), w[:, :96].contiguous())        # K is no multiple of 64
    with pytest.raises(MsaError):
        ops.tile_linear(x, w[:60])                                             # N is no multiple of 8
    with pytest.raises(MsaError):
        ops.tile_linear(torch.empty(64 * 128 + 8, device="cuda", dtype=torch.bfloat16)[4:-4].view(64, 128), w)


def test_module_route(ops):
    """The module's own call and the tiled product agree; hooks, biases and gradients keep the module's call."""
    x, w, want = _operands(4096, 1024, 4096, 5)
    lin = torch.nn.Linear(1024, 4096, bias=False).cuda().bfloat16()
    with torch.no_grad():
        lin.weight.copy_(w)
        assert ops.linear_ok(lin, x) and _err(ops.linear(lin, x), want) < TOL
        assert not ops.linear_ok(lin, x[:2300])       # 144 tiles, but not their outputs
        h = lin.register_forward_hook(lambda m, i, o: o * 0)
        assert not ops.linear_ok(lin, x) and not ops.linear(lin, x).any()
        h.remove()
        assert not ops.linear_ok(torch.nn.Linear(1024, 4096).cuda().bfloat16(), x)
    assert not ops.linear_ok(lin, x) and ops.linear(lin, x).requires_grad
