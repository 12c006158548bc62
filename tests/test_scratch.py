"""Scratch of a call belongs to that call: not to another that is enqueued between its launches (a thread, a stream), nor to a later one
while a captured graph still replays it."""
import pytest
import torch


class _Lib:
    """An entry point that asks for scratch, notes what it is given and, the first time, lets another call in before it returns."""

    def __init__(self, entry, size, need):
        self.given, self.inside = [], None
        setattr(self, entry, self._entry)
        setattr(self, size, lambda *a: need)

    def _entry(self, *a):
        self.given.append(a[self.at])
        if self.inside is not None:
            inside, self.inside = self.inside, None
            inside()
        return 0


def _skinny(ops, seq_ops):
    x, w = torch.zeros((16, 256)).bfloat16(), torch.zeros((64, 256)).bfloat16()
    return ("msa_skinny_linear_ws", "msa_skinny_linear_workspace_bytes", -3, lambda: ops.skinny_linear(x, w))


def _attention(ops, seq_ops):
    q, k = torch.zeros((2, 4, 128)).bfloat16(), torch.zeros((64, 2, 128)).bfloat16()
    off, n = torch.zeros(2, dtype=torch.int64), torch.full((2,), 30, dtype=torch.int32)
    return ("msa_sparse_attn", "msa_attn_workspace_bytes", -3, lambda: ops.sparse_attn(q, k, k, off, n, 32))


def _gru(ops, seq_ops):
    zug, b, state = torch.zeros((3, 48)), torch.zeros(16), torch.zeros((1, 16))
    batch = seq_ops.StepBatch([3], [0], [0], "cpu")
    return ("msa_seq_min_gru", "msa_seq_min_gru_workspace_bytes", -3, lambda: seq_ops.min_gru(zug, b, b, 16, state, batch))


@pytest.mark.parametrize("case", [_skinny, _attention, _gru])
def test_a_call_between_has_its_own(case, monkeypatch):
    from msa_amd import _lib, ops, seq_ops
    entry, size, at, call = case(ops, seq_ops)
    lib = _Lib(entry, size, 4096)
    lib.at = at
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(_lib, "load_seq", lambda: lib)
    for m, names in ((ops, ("_need_cuda",)), (seq_ops, ("_cuda", "_dense", "_f32"))):
        for n in names:
            monkeypatch.setattr(m, n, lambda *a: None)
        monkeypatch.setattr(m, "_stream", lambda *a: 0)
    lib.inside = call
    call()
    assert len(lib.given) == 2 and None not in lib.given and lib.given[0] != lib.given[1]


# ------------------------------------------------------------------------------------------------ on the device
def _calls(ops, seed):
    """Calls with scratch: a product whose K is cut over workgroups, decode attention over split keys, a routed selection."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").bfloat16()
    x, w = rnd(16, 9728), rnd(2560, 9728)
    q, k, v = rnd(4, 32, 128), rnd(4 * 3000, 8, 128), rnd(4 * 3000, 8, 128)
    off, n = torch.arange(4, device="cuda") * 3000, torch.full((4,), 2990, dtype=torch.int32, device="cuda")
    bank = ops.Bank(1, (torch.arange(301) * 8).to(torch.int32), torch.arange(300), 8, 128, torch.bfloat16)
    bank.set_layer(0, torch.nn.functional.normalize(rnd(2400, 8, 128).float(), dim=-1).bfloat16())
    qr = rnd(2, 64, 32, 128)
    from msa_amd import _lib
    assert _lib.load().msa_skinny_linear_workspace_bytes(16, 2560, 9728) > 0
    return lambda: [ops.skinny_linear(x, w), ops.sparse_attn(q, k, v, off, n, 3000), *ops.route_topk(bank, 0, qr, topk=16)]


@pytest.mark.gpu
def test_captured_calls_behind_larger_ones():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import ops
    calls = _calls(ops, 1)
    want = [t.clone() for t in calls()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = calls()
    print("[scratch] captured", flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    big = torch.randn((16, 32, 128), generator=g, device="cuda").bfloat16()
    kv = torch.randn((16 * 9000, 8, 128), generator=g, device="cuda").bfloat16()
    off, n = torch.arange(16, device="cuda") * 9000, torch.full((16,), 9000, dtype=torch.int32, device="cuda")
    for _ in range(3):
        ops.sparse_attn(big, kv, kv, off, n, 9000)                 # more scratch than the captured call's
        fill = [torch.full((size,), 0x7F, dtype=torch.uint8, device="cuda") for size in (1 << 12, 1 << 16, 1 << 20, 1 << 22, 1 << 24)]
        for t in held:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(held, want))
        assert all(bool((t == 0x7F).all()) for t in fill)          # and a replay writes nobody else's memory


@pytest.mark.gpu
def test_two_streams():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import ops
    sides = [_calls(ops, s) for s in (3, 4)]
    want = [[t.clone() for t in c()] for c in sides]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in sides]
    print("[scratch] two streams", flush=True)
    got = [[], []]
    for _ in range(20):
        for i, c in enumerate(sides):
            with torch.cuda.stream(streams[i]):
                got[i].append(c())
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(a, b) for outs in got[i] for a, b in zip(outs, want[i]))
