"""A step's description goes to the device in one copy: contents, lifetime, and who may read it when."""
import numpy as np
import pytest
import torch

from msa_amd import seq_ops


def check(b, counts, slots, pos, extra):
    n = len(counts)
    assert b.cu.tolist() == np.cumsum([0] + counts).tolist() and b.slot.tolist() == slots and b.pos.tolist() == pos
    assert b.row_seq.tolist() == [s for s in range(n) for _ in range(counts[s])]
    assert [e.tolist() for e in b.extra] == [list(e) for e in extra]
    assert b.cu.dtype == b.slot.dtype == b.row_seq.dtype == torch.int32 and b.pos.dtype == torch.int64
    assert all(t.data_ptr() % t.element_size() == 0 for t in (b.cu, b.slot, b.pos, b.row_seq, *b.extra))


def test_only_a_step_does_not_wait(monkeypatch):
    """A description is complete when it is handed out, for any stream; a model's own step, which reads it on the stream it was made
    on, asks for no wait."""
    asked, to = [], torch.Tensor.to

    def spy(self, *a, **k):
        if "non_blocking" in k:
            asked.append(k["non_blocking"])
        return to(self, *a, **k)
    monkeypatch.setattr(torch.Tensor, "to", spy)
    seq_ops.StepBatch([2, 1], [0, 1], [0, 0], "cpu")
    assert asked == [False]
    asked.clear()
    seq_ops.StepBatch([2, 1], [0, 1], [0, 0], "cpu", wait=False)
    assert asked == [True]
    from types import SimpleNamespace
    from msa_amd.step_decoder import StepDecoder
    cache = SimpleNamespace(length={}, slot_of={}, reserve=lambda n: None, advance=lambda k, n: None)
    cache.open = lambda k: (cache.length.setdefault(k, 0), cache.slot_of.setdefault(k, len(cache.slot_of)))
    model = SimpleNamespace(config=SimpleNamespace(vocab=9), device="cpu", forward_rows=lambda tokens, batch, *a, **k: tokens)
    asked.clear()
    assert StepDecoder.step(model, cache, [("a", [1, 2], [1]), ("b", [3], [0])]).tolist() == [1, 2, 3] and asked == [True]


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[4], [2, 3, 1]])
def test_other_streams_may_read_a_description(counts):
    """Made on a stream with a long queue, read on another one at once."""
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    a = torch.randn(8192, 8192, device="cuda")
    torch.cuda.synchronize()
    for i in range(3):
        with torch.cuda.stream(busy):
            for _ in range(4):
                a = torch.mm(a, a) * 1e-4
            b = seq_ops.StepBatch(counts, [i + s for s in range(len(counts))], [7 * i] * len(counts), "cuda")
        with torch.cuda.stream(other):
            check(b, counts, [i + s for s in range(len(counts))], [7 * i] * len(counts), ())


@pytest.mark.parametrize("counts", [[1], [5], [3, 1], [2, 7, 1], [1] * 16])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_step_batch_contents(counts, device):
    slots, pos = [3 * s + 1 for s in range(len(counts))][::-1], [2 ** 33 + s for s in range(len(counts))]
    extra = (np.arange(sum(counts), dtype=np.int64) - 2 ** 40, np.zeros(0, np.int64), np.asarray([7], np.int64))
    check(seq_ops.StepBatch(counts, slots, pos, device, extra), counts, slots, pos, extra)


@pytest.mark.gpu
def test_pinned_memory_outlives_the_copies():
    """Copies queued behind a long product: every batch still holds its own values although the host has gone on."""
    a = torch.randn(8192, 8192, device="cuda")
    for _ in range(8):
        a = torch.mm(a, a) * 1e-4
    extra = [(np.full(1000, i, np.int64),) for i in range(40)]
    batches = [seq_ops.StepBatch([2, 3], [i, i + 1], [i, 0], "cuda", extra[i], wait=False) for i in range(40)]
    for i, b in enumerate(batches):
        check(b, [2, 3], [i, i + 1], [i, 0], extra[i])


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_offsets_of_keys_one_sequence_behind_the_other(device):
    for counts, pos in (([1], [0]), ([5], [7]), ([3, 1, 4], [0, 2 ** 33, 9]), ([1] * 16, list(range(16)))):
        b = seq_ops.StepBatch(counts, list(range(len(counts))), pos, device)
        ends = [p + c for p, c in zip(pos, counts)]
        assert b.key_off.tolist() == [sum(ends[:s]) for s in range(len(counts))]
        assert b.key_off.dtype == torch.int64 and b.key_off.device == b.pos.device and b.key_off.data_ptr() % 8 == 0
