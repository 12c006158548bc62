"""Entry points that advance a state, called again with the same tensors: every call launches, and nothing of a call outlives it."""
import gc
import inspect
import weakref

import pytest
import torch


def test_nothing_is_memoised():
    """Keys of a cache keep tensors, and what is found there launches nothing."""
    from msa_amd import hybrid, hybrid_layers, memory_sparse_attention, model, ops, postnorm, seq_ops, step_decoder
    for m in (ops, seq_ops, hybrid, hybrid_layers, postnorm, step_decoder, model, memory_sparse_attention):
        for name, f in vars(m).items():
            members = [(f"{name}.{n}", x) for n, x in vars(f).items()] if inspect.isclass(f) and f.__module__ == m.__name__ else [(name, f)]
            assert not [n for n, x in members if hasattr(x, "cache_info")], m.__name__


class _Lib:
    def __init__(self):
        self.calls = 0

    def msa_seq_delta_step(self, *a):
        self.calls += 1
        return 0


def test_delta_step_launches_each_time_and_keeps_nothing(monkeypatch):
    from msa_amd import _lib, seq_ops
    lib = _Lib()
    monkeypatch.setattr(_lib, "load_seq", lambda: lib)
    for n in ("_cuda", "_dense", "_f32"):
        monkeypatch.setattr(seq_ops, n, lambda *a: None)
    monkeypatch.setattr(seq_ops, "_stream", lambda *a: 0)
    B, H, D, E, R = 2, 2, 16, 8, 8
    bf = lambda *s: torch.zeros(s).bfloat16()
    ten = [bf(B, 2 * H * D + H * E), bf(B, R), bf(B, R), bf(H * D + H * E, R), bf(B, H), torch.zeros(H), torch.zeros(H * D), torch.zeros(E), torch.zeros(B, H, D, E)]
    batch = seq_ops.StepBatch([1] * B, list(range(B)), [0] * B, "cpu")
    step = lambda t, b: seq_ops.delta_step(*t[:4], H * D, t[4], *t[5:8], 1e-5, H, H, D, E, t[8], b)
    first = step(ten, batch)
    assert step(ten, batch) is not first and lib.calls == 2
    refs = [weakref.ref(t) for t in (first, *ten, batch)]
    del first, ten, batch
    gc.collect()
    assert not [r for r in refs if r() is not None]


# ------------------------------------------------------------------------------------------------ on the device
@pytest.fixture
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,G,D,E,R", [(1, 16, 16, 64, 128, 64), (3, 4, 2, 128, 128, 128)])
def test_delta_steps_on_the_same_buffers(gpu, B, H, G, D, E, R):
    """Three tokens through one set of buffers, filled in place: outputs rounded to bf16 (2^-9), the state's sums in another order."""
    from msa_amd import seq_ops
    print(f"[repeated] B={B} H={H} D={D} E={E}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(B)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    ch, n_a = 2 * G * D + H * E, H * D
    w = (rnd(n_a + H * E, R) * R ** -0.5).bfloat16()
    A_log, bias, norm = rnd(H).sigmoid(), rnd(H * D) - 2, 1 + 0.1 * rnd(E)
    state = 0.3 * rnd(B, H, D, E)
    state2 = state.clone()
    batch = seq_ops.StepBatch([1] * B, list(range(B)), [9] * B, "cuda")
    qkv, a_low, g_low, b = (torch.empty((B, n), dtype=torch.bfloat16, device="cuda") for n in (ch, R, R, H))
    for _ in range(3):
        for t in (qkv, a_low, g_low, b):
            t.copy_(rnd(*t.shape))
        got = seq_ops.delta_step(qkv, a_low, g_low, w, n_a, b, A_log, bias, norm, 1e-5, H, G, D, E, state, batch)
        a, gate = a_low.float() @ w[:n_a].float().t(), g_low.float() @ w[n_a:].float().t()
        want = seq_ops.delta(qkv.float(), a, b.float(), gate, A_log, bias, norm, 1e-5, H, G, D, E, state2, batch)
        assert ((got.float() - want).norm() / want.norm()).item() < 3e-3
        assert ((state - state2).norm() / state2.norm()).item() < 1e-5


def _postnorm():
    from msa_amd.config import PostNormConfig
    from msa_amd.postnorm import PostNormForCausalLM
    from postnorm_models import ATTN, config, layer, random_weights, tensor_shapes
    cfg = config([layer("channel_delta", {"heads": 4, "kv_heads": 2, "dim": 64, "vdim": 128, "conv": 4}), layer("attention", ATTN)], width=256)
    return lambda: PostNormForCausalLM.from_tensors(PostNormConfig.from_dict(cfg), random_weights(tensor_shapes(cfg, (64, 64))), torch.bfloat16, "cuda:0")


def _hybrid():
    from hybrid_models import CONFIGS
    from msa_amd.config import HybridConfig
    from msa_amd.hybrid import HybridForCausalLM
    return lambda: HybridForCausalLM.random(HybridConfig.from_dict(CONFIGS["mixed"]), 0, torch.bfloat16, "cuda:0")


@pytest.mark.gpu
@pytest.mark.parametrize("make", [_postnorm, _hybrid])
def test_eager_steps_hold_no_memory(gpu, monkeypatch, make):
    """Eager decode steps leave the allocator where it was, and a model and its cache that are dropped are given back."""
    from msa_amd import seq_ops
    taken, inner = [], seq_ops.delta_step
    monkeypatch.setattr(seq_ops, "delta_step", lambda *a: (taken.append(1), inner(*a))[1])
    model = make()

    def held():
        gc.collect()
        torch.cuda.synchronize()
        return torch.cuda.memory_allocated()

    def life():
        m = model()
        cache = m.create_cache(2, 64)
        sizes = []
        for i in range(12):
            m.step(cache, [(k, [i % 7], [0]) for k in ("a", "b")])
            sizes.append(held())
        assert len(set(sizes[2:])) == 1, sizes
    life()                                                 # (what a process allocates once)
    print("[repeated] second model", flush=True)
    before = held()
    life()
    assert len(taken) == (24 if make is _postnorm else 0) and held() == before
