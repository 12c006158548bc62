"""The calls that the host's extension module takes, against the same calls through the interpreter: the same launches, so the same bits; and
what that path refuses is refused with its errors."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from msa_amd import _lib, cache, ops, seq_ops


class _Declines:
    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture
def interpreted(monkeypatch):
    """Runs a call without the module."""
    def run(f):
        with monkeypatch.context() as m:
            m.setattr(ops, "host", lambda: _Declines())
            return f()
    return run


def test_pieces_and_cleared_slots():
    host = ops.host()
    words = torch.arange(40, dtype=torch.int64) * 3 + (7 << 32)
    got = host.pieces(words, [(0, 5, True), (3, 0, False), (4, 7, False), (39, 1, True)])
    assert torch.equal(got[0], words.view(torch.int32)[:5]) and got[1].numel() == 0 and got[1].dtype == torch.int64
    assert torch.equal(got[2], words[4:11]) and torch.equal(got[3], words[39:].view(torch.int32)[:1])
    for bad in ((words.int(), []), (words, [(38, 5, False)]), (words, [(0, 1)])):
        with pytest.raises(Exception):
            host.pieces(*bad)
    a, b = torch.ones(4, 3), torch.ones(4, 2, 2)
    host.clear([a, b], 2)
    host.clear([], 0)
    assert a.sum(1).tolist() == [3, 3, 0, 3] and b.sum((1, 2)).tolist() == [4, 4, 0, 4]
    with pytest.raises(ImportError):
        host.bind(None, "no such library", (1, 1, 1, 1, 1.0, 1.0))
    for bad in (([a], 4), ([1], 0), ([a], "0")):
        with pytest.raises(Exception):
            host.clear(*bad)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_an_opened_sequence_s_states_are_cleared(device):
    c = cache.SequenceStateCache([{"s": cache.StateSpec((3,), torch.float32), "rows": cache.StateSpec((2,), torch.bfloat16, per_token=True)}], device, 2, 5)
    for t in c.tensors[0].values():
        t.fill_(1.0)
    assert c.open("a") == 0 and c.tensors[0]["s"].sum(1).tolist() == [0, 3] and c.tensors[0]["rows"].sum() == 20


@pytest.mark.skipif(torch.cuda.device_count() == 1, reason="where there is a device, a fake tensor cannot name one that is not")
def test_states_of_another_device_are_cleared_there():
    """A launch goes to the current device: tensors of another one are cleared by the call that switches to theirs.  (Fake tensors name a second
    device without one; where no device is current, none is theirs.)"""
    cleared = []

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            if f is torch.ops.aten._foreach_zero_.default:
                cleared.extend((str(t.device), tuple(t.shape)) for t in args[0])
            return f(*args, **(kwargs or {}))

    with FakeTensorMode():
        c = cache.SequenceStateCache([{"s": cache.StateSpec((3,), torch.float32), "c": cache.StateSpec((2, 2), torch.bfloat16)}], "cuda:1", 3, 5)
        with Seen():
            assert c.open_all(["a", "b"]) == [0, 1]
    assert cleared == [("cuda:1", (3,))] * 2 + [("cuda:1", (2, 2))] * 2


@pytest.mark.parametrize("name", ["linear", "residual_norm", "rms_residual", "conv_silu", "group_rmsnorm", "ssd", "delta"])
def test_operands_without_an_address_raise(name):
    """A wrapper of vmap passes for a tensor of the device and has no storage: the error of asking it for an address comes back as one, in front of
    any launch."""
    host, bf, batch = ops.host(), torch.bfloat16, seq_ops.StepBatch([4], [0], [0], "cpu")
    with FakeTensorMode():
        r = lambda *s, t=torch.float32: torch.empty(s, dtype=t, device="cuda:0")
        b = (batch.address, batch.top)
        calls = {
            "linear": ((4, 64), lambda x: host.linear(x, r(16, 64, t=bf), _lib.TILE_STORE, 0, 0.0, 0.0, 0.0)),
            "residual_norm": ((4, 8), lambda y: host.residual_norm(*b, r(4, 8), y, y, r(8), r(8), r(8), 1.0, None, None, True, _lib.MSA_BF16)),
            "rms_residual": ((4, 8), lambda y: host.rms_residual(r(4, 8), y, r(8), 1e-5, None, r(4, 8), True, _lib.MSA_BF16)),
            "conv_silu": ((4, 8), lambda x: host.conv_silu(*b, x, r(8, 4), None, r(1, 3, 8))),
            "group_rmsnorm": ((4, 8), lambda v: host.group_rmsnorm(v, r(8), 1, 1e-5)),
            "ssd": ((4, 32), lambda x: host.ssd(*b, x, r(4, 16, t=bf), r(4, 2, t=bf), r(2), r(2), r(2), 2, 8, 8, 1, r(1, 2, 8, 8), False)),
            "delta": ((4, 32), lambda x: host.delta(*b, x, r(4, 16, t=bf), r(4, 2, t=bf), r(4, 16, t=bf), r(2), r(16), r(8), 1e-5, 2, 1, 8, 8, r(1, 2, 8, 8), False)),
        }
        shape, call = calls[name]
        with pytest.raises(RuntimeError, match="data pointer"):
            torch.vmap(call)(r(3, *shape, t=bf))


def same(a, b):
    return all((x is None) == (y is None) and (x is None or (x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y))) for x, y in zip(a, b))


@pytest.mark.gpu
def test_rule_of_the_small_tiles(interpreted):
    bf = lambda *s: torch.randn(s, device="cuda").bfloat16()
    for T, K, N in ((1, 64, 16), (122, 1024, 1024), (2048, 1024, 4096), (2049, 1024, 16), (6001, 128, 4096), (300, 2560, 8192), (40, 96, 64), (40, 64, 72),
                    (0, 64, 16), (17, 9728, 2560)):
        x, w, wide = bf(T, K), bf(N, K), bf(T + 1, K + 24)
        forms = [(x, w), (wide[:T, 8:K + 8], w), (wide[:T, 4:K + 4], w), (wide[:T, :K], w), (bf(T, K + 4)[:, :K], w), (x.float(), w), (x, w.float()), (x, w.half()),
                 (x, bf(K, N).t()), (x[None], w), (x, w[None]), (x.cpu(), w), (x, w.cpu()), (x, w.clone().requires_grad_()), (x.clone().requires_grad_(), w),
                 (bf(K, T).t(), w), (x, bf(N, K + 64))]
        for a, b in forms:
            for end in (False, True):
                with torch.no_grad():
                    free = ops.block_linear_ok(a, b, end)
                    assert free == interpreted(lambda: ops.block_linear_ok(a, b, end))
                assert ops.block_linear_ok(a, b, end) == interpreted(lambda: ops.block_linear_ok(a, b, end))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts", [[1], [70, 3, 130]])
def test_layers_calls(interpreted, dtype, counts):
    g = torch.Generator(device="cuda").manual_seed(sum(counts))
    r = lambda *s: torch.randn(s, generator=g, device="cuda")
    T, W, n = sum(counts), 96, len(counts)
    batch = seq_ops.StepBatch(counts, list(range(n))[::-1], [0] * n, "cuda")
    x, y, wide, bias = r(T, W), r(T, W).to(dtype), r(T, W + 8).to(dtype), r(W)
    gate, norm, shift, w = wide[:, 8:], seq_ops.DynTanhNorm(r(W), r(W), 0.7), r(W), r(W)
    H, P, N, G = 4, 16, 32, 2
    calls = {
        "residual_norm": lambda s: seq_ops.residual_norm(x, batch, dtype, y, gate, bias, norm, shift, s[0]),
        "no sublayer": lambda s: seq_ops.residual_norm(x, batch, dtype, norm=norm, shift=shift, prev=s[0], want_h=False),
        "no norm": lambda s: seq_ops.residual_norm(x, batch, dtype, y, gate, bias),
        "rms_residual": lambda s: seq_ops.rms_residual(x, dtype, gate, w, 1e-5, out=torch.empty_like(x)),
        "rms_residual, next norm": lambda s: seq_ops.rms_residual(x, dtype, y, w, 1e-5, bias, out=torch.empty_like(x)),
        "conv_silu": lambda s: (seq_ops.conv_silu(gate, s[1][0], bias, s[2], batch),),
        "conv_silu, no bias": lambda s: (seq_ops.conv_silu(y, s[1][0], None, s[2], batch),),
        "group_rmsnorm": lambda s: (seq_ops.group_rmsnorm(y, w, 4, 1e-5),),
        "ssd": lambda s: (seq_ops.ssd(*s[3], H, P, N, G, s[4], batch, False),),
        "ssd, chunked": lambda s: (seq_ops.ssd(*s[3], H, P, N, G, s[4], batch, dtype == torch.bfloat16),),
        "delta": lambda s: (seq_ops.delta(*s[5], 1e-5, H, G, 32, 16, s[6], batch, False),),
        "delta, chunked": lambda s: (seq_ops.delta(*s[5], 1e-5, H, G, 32, 16, s[6], batch, dtype == torch.bfloat16),),
    }
    held = [r(n, W), [r(W, 4)], r(n, 3, W), [r(T, H * P + 2 * G * N).to(dtype), r(T, H * P + 8).to(dtype)[:, 8:], r(T, H).to(dtype), r(H), r(H), r(H)], r(n, H, N, P),
            [r(T, 2 * G * 32 + H * 16).to(dtype), r(T, H * 32).to(dtype), r(T, H).to(dtype), r(T, H * 16).to(dtype), r(H), r(H * 32), r(16)], r(n, H, 32, 16)]
    copy = lambda: [[t.clone() if i != 1 else t for t in s] if type(s) is list and i != 3 else s if type(s) is list else s.clone() for i, s in enumerate(held)]
    for name, call in calls.items():
        print(f"[host path] {name} {counts} {dtype}", flush=True)
        a, b = copy(), copy()
        got, want = call(a), interpreted(lambda: call(b))
        assert same(got, want), name
        assert all(torch.equal(a[i], b[i]) for i in (0, 2, 4, 6)), name


@pytest.mark.gpu
def test_refusals():
    T, W = 5, 64
    x, y, f = torch.zeros((T, W), device="cuda"), torch.zeros((T, W), device="cuda").bfloat16(), torch.ones(W, device="cuda")
    batch, norm, state = seq_ops.StepBatch([T], [3], [0], "cuda"), seq_ops.DynTanhNorm(f, f, 1.0), torch.zeros((4, 3, W), device="cuda")
    bf = torch.bfloat16
    for call in (lambda: seq_ops.residual_norm(x.bfloat16(), batch, bf, norm=norm), lambda: seq_ops.residual_norm(x[:4], batch, bf, norm=norm),
                 lambda: seq_ops.residual_norm(x, batch, bf, y, y[:, :32], f), lambda: seq_ops.residual_norm(x, batch, bf, y.float(), y, f),
                 lambda: seq_ops.residual_norm(x, batch, bf, y, y, f[:8]), lambda: seq_ops.residual_norm(x, batch, bf, norm=norm, shift=f, prev=state[:3, 0]),
                 lambda: seq_ops.residual_norm(x, batch, bf, norm=norm, shift=f.cpu(), prev=state[:, 0].contiguous()),
                 lambda: seq_ops.rms_residual(x, bf, y.t().contiguous().t(), f, 1e-5, out=x), lambda: seq_ops.rms_residual(x, bf, y, f, 1e-5, out=x.bfloat16()),
                 lambda: seq_ops.conv_silu(y, torch.ones((W, 4), device="cuda"), None, state[:3].contiguous(), batch),
                 lambda: seq_ops.conv_silu(y, torch.ones((W, 3), device="cuda"), None, state, batch),
                 lambda: seq_ops.group_rmsnorm(y.t().contiguous().t(), f, 4, 1e-5), lambda: seq_ops.group_rmsnorm(y, f.double(), 4, 1e-5),
                 lambda: ops.block_linear(y.cpu(), y)):
        with pytest.raises(ValueError):
            call()
    for call in (lambda: seq_ops.group_rmsnorm(y, f, 7, 1e-5), lambda: ops.block_linear(y[:, :48].contiguous(), y[:, :48].contiguous())):
        with pytest.raises(_lib.MsaError):
            call()
    with pytest.raises(TypeError):
        seq_ops.residual_norm(x, batch, torch.float16, norm=norm)
