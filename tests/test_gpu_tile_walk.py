"""The walk of the tiled products over rounds of whole tiles and a last one cut into pieces of K, against fp32: a held tile finished under a
piece's steps, a piece too short for that, several pieces of one workgroup behind one another, outputs that pass the caches.

Tolerances: one rounding to bf16, 1.7e-3 over many values; a gated unit and gelu round the product first (``test_gpu_tile_gemm.py``)."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu
TOL, TOL_END = 3e-3, 4e-3
TILE, XCDS, PIECE = 256, 8, 256 * 256 * 4


def _say(msg):
    print(f"[tile_walk] {msg}", flush=True)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import ops
    return ops


def _walk(ops, T, K, N):
    """(complete rounds, pieces a tile of the last round, K tiles of a piece, items of a workgroup in it)"""
    from msa_amd import _lib
    units = torch.cuda.get_device_properties(0).multi_processor_count // XCDS
    tiles = -(-T // TILE) * -(-N // TILE)
    share = [tiles * (x + 1) // XCDS - tiles * x // XCDS for x in range(XCDS)]
    rem = max(s % units for s in share)
    need = _lib.load().msa_tile_workspace_bytes(T, K, N)
    split = need // (XCDS * rem * PIECE) if rem and need else 1
    return min(s // units for s in share), split, K // 64 // split, -(-rem * split // units)


def _operands(T, K, N, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((T, K), generator=g, device="cuda").bfloat16()
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    return x, w, x.float() @ w.float().t()


def _err(got, want):
    return ((got.float() - want).norm() / want.norm()).item()


def _call(ops, x, w, out, mode, gelu_n=0, glu=(0.0, 0.0, 0.0), pieces=True):
    from msa_amd import _lib
    (T, K), N = x.shape, w.shape[0]
    end = _lib.TileEnd(mode, gelu_n, *glu)
    ws = torch.empty(_lib.load().msa_tile_workspace_bytes(T, K, N), dtype=torch.uint8, device="cuda") if pieces else None
    ops.check(_lib.load().msa_tile_linear(ops.ptr(x), K, T, K, ops.ptr(w), N, C.byref(end), ops.ptr(out), out.shape[1], ops.ptr(ws),
                                          0 if ws is None else ws.numel(), ops._stream()), "msa_tile_linear")
    return out


# complete rounds, pieces a tile, K tiles a piece and items of a workgroup in the last round, on 256 compute units: pieces that a held tile is
# finished under; pieces too short for that; two of them to a workgroup; compute units without any (257 tiles)
SHAPES = [(5880, 4096, 4080), (6001, 2560, 19456), (8900, 8192, 2800), (200, 1024, 65776)]
WALKS = [(1, 2, 32, 1), (7, 4, 10, 1), (1, 3, 42, 2), (1, 4, 4, 1)]


def test_the_shapes_are_what_they_are_for(ops):
    walks = [_walk(ops, *s) for s in SHAPES]
    _say(str(walks))
    assert walks == WALKS or torch.cuda.get_device_properties(0).multi_processor_count != 256


@pytest.mark.parametrize("T,K,N", SHAPES)
def test_ends(ops, T, K, N):
    from msa_amd import _lib
    _say(f"T={T} K={K} N={N}")
    x, w, want = _operands(T, K, N, 1)
    assert _err(ops.tile_linear(x, w), want) < TOL
    base = torch.randn((T, N), device="cuda").bfloat16()
    out = base.clone()
    ops.tile_linear(x, w, out=out, add=True)
    assert _err(out, want + base.float()) < TOL
    n = N // 2 // 128 * 128
    act = torch.nn.functional.gelu(want[:, :n], approximate="tanh")
    got = ops.tile_linear(x, w, gelu_n=n)
    assert _err(got[:, :n], act) < TOL_END and _err(got[:, n:], want[:, n:]) < TOL
    limit, alpha, shift = 1.5, 1.702, 1.0
    gate, up = want[:, 0::2].clamp(max=limit), want[:, 1::2].clamp(-limit, limit)
    assert _err(ops.tile_linear(x, w, glu=(limit, alpha, shift)), gate * torch.sigmoid(alpha * gate) * (up + shift)) < TOL_END
    gate, up = want.view(T, N // 16, 2, 8).unbind(2)
    assert _err(ops.tile_linear(x, w, silu_mul=True), (torch.nn.functional.silu(gate) * up).reshape(T, -1)) < TOL_END


@pytest.mark.parametrize("T,K,N", SHAPES)
def test_ends_in_pieces_round_as_whole_ones(ops, T, K, N):
    """fp32 sums of another order differ by some 1e-6, which moves one in thousands to the other side of a rounding; an end that rounds
    the sums first and one that does not differ in a tenth of all results where a third of the tiles is cut."""
    from msa_amd import _lib
    x, w, _ = _operands(T, K, N, 2)
    for mode, width, kw in ((_lib.TILE_STORE, N, {}), (_lib.TILE_GELU, N, dict(gelu_n=N // 128 * 128)), (_lib.TILE_SILU_MUL, N // 2, {}),
                            (_lib.TILE_GLU, N // 2, dict(glu=(1.5, 1.702, 1.0)))):
        a, b = (_call(ops, x, w, torch.empty((T, width), device="cuda").bfloat16(), mode, pieces=p, **kw) for p in (True, False))
        share = (a != b).float().mean().item()
        _say(f"T={T} K={K} N={N} mode={mode}: {share:.5f} differ")
        assert share < 0.002


def test_heads(ops):
    from msa_amd import _lib
    T, K, front, Hq, Hkv, back = 5880, 4096, 4, 16, 4, 4
    N = (front + Hq + 2 * Hkv + back) * 128
    assert _walk(ops, T, K, N)[0] >= 1 and _walk(ops, T, K, N)[1] > 1
    x, w, want = _operands(T, K, N, 3)
    pos = torch.arange(T, device="cuda") % 500
    nw = [1 + 0.1 * torch.randn(128, device="cuda").bfloat16() for _ in range(2)]
    rope = ops.rope_tables(500, 128, 1e6, device="cuda")
    q, k, v, r = ops.qkv_proj(x, w, Hq, Hkv, pos, nw[0], nw[1], 1e-6, rope, router_front=front, router_back=back)
    heads = want.view(T, -1, 128)

    def turned(t, n):
        t = t * torch.rsqrt((t * t).mean(-1, keepdim=True) + 1e-6) * n.float()
        lo, hi = t.chunk(2, dim=-1)
        c, s = rope[0][pos][:, None], rope[1][pos][:, None]
        return torch.cat([lo * c - hi * s, hi * c + lo * s], dim=-1)
    at = front
    assert _err(q, turned(heads[:, at:at + Hq], nw[0])) < TOL
    assert _err(k, turned(heads[:, at + Hq:at + Hq + Hkv], nw[1])) < TOL
    assert _err(v, heads[:, at + Hq + Hkv:at + Hq + 2 * Hkv]) < TOL
    assert _err(r, torch.cat([heads[:, :front], heads[:, at + Hq + 2 * Hkv:]], dim=1)) < TOL


@pytest.mark.parametrize("T,K,N,pair", [(8208, 704, 8200, False), (8208, 640, 8200, False), (11600, 704, 11600, True)])
def test_outputs_past_the_caches(ops, T, K, N, pair):
    """Outputs of more than 128 MB are stored non-temporal."""
    _say(f"T={T} K={K} N={N}")
    assert T * N * (1 if pair else 2) > 128 << 20
    x, w, want = _operands(T, K, N, 4)
    if pair:
        gate, up = want[:, 0::2].clamp(max=1.5), want[:, 1::2].clamp(-1.5, 1.5)
        assert _err(ops.tile_linear(x, w, glu=(1.5, 1.702, 1.0)), gate * torch.sigmoid(1.702 * gate) * (up + 1.0)) < TOL_END
        gate, up = want.view(T, N // 16, 2, 8).unbind(2)
        assert _err(ops.tile_linear(x, w, silu_mul=True), (torch.nn.functional.silu(gate) * up).reshape(T, -1)) < TOL_END
    else:
        assert _err(ops.tile_linear(x, w), want) < TOL
        want[:, :4096] = torch.nn.functional.gelu(want[:, :4096], approximate="tanh")
        assert _err(ops.tile_linear(x, w, gelu_n=4096), want) < TOL_END
