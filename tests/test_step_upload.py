"""A step's description goes to the device in one copy that nothing waits for: contents and lifetime."""
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
    batches = [seq_ops.StepBatch([2, 3], [i, i + 1], [i, 0], "cuda", extra[i]) for i in range(40)]
    for i, b in enumerate(batches):
        check(b, [2, 3], [i, i + 1], [i, 0], extra[i])
