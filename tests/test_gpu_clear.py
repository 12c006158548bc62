"""Clearing the states of the sequences that a step opens: one launch for all of them."""
import pytest
import torch

from msa_amd import cache, ops


@pytest.mark.gpu
@pytest.mark.parametrize("slots", [[3], [0, 4, 2], list(range(19, -1, -1))])
def test_rows_of_many_tensors(slots):
    """Rows of one byte to several workgroups, whole and with a rest, aligned to 16, 4 and fewer bytes; more tensors and slots than a launch takes."""
    shapes = [(20, 3), (20, 4), (20, 1, 1), (20, 5000), (20, 4097, 3), (20, 2, 0), (20, 4096), (20, 8, 1024), (20, 7)] * 3
    types = [torch.float32, torch.bfloat16, torch.uint8]
    ts = [torch.ones(s, dtype=types[i % 3 if i < 9 else (i + i // 9) % 3], device="cuda") for i, s in enumerate(shapes)]
    ops.host().clear(ts, slots)
    torch.cuda.synchronize()
    for t in ts:
        want = torch.ones_like(t)
        want[slots] = 0
        assert torch.equal(t, want)
    part = torch.ones((6, 8), device="cuda")[:, :4]               # rows that do not lie behind one another
    ops.host().clear([part, ts[0]], [1, 5])
    assert part.sum(1).tolist() == [4, 0, 4, 4, 4, 0]
    for bad in ([20], [0, "1"], [-21]):
        with pytest.raises(Exception):
            ops.host().clear(ts, bad)


@pytest.mark.gpu
def test_one_launch_makes_no_views():
    """Of six states and eight slots, forty-eight views would take the host as long as several launches."""
    ts = [torch.ones((9, 4 + i), device="cuda") for i in range(6)]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as p:
        ops.host().clear(ts, list(range(8)))
    assert all(t[:8].sum() == 0 and t[8].sum() == t.shape[1] for t in ts)
    assert not [e.key for e in p.key_averages() if e.key.startswith("aten::")]


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_opening_several(device):
    c = cache.SequenceStateCache([{"s": cache.StateSpec((3,), torch.float32), "rows": cache.StateSpec((2,), torch.bfloat16, per_token=True)}], device, 2, 5)
    c.open("a")
    for t in c.tensors[0].values():
        t.fill_(1.0)
    assert c.open_all(["b", "c", "d"]) == [1, 2, 3] and c.slots == 4 and c.length == {"a": 0, "b": 0, "c": 0, "d": 0}
    assert c.tensors[0]["s"].sum(1).tolist() == [3, 0, 0, 0] and c.tensors[0]["rows"].sum() == 20
    for bad in (["e", "a"], ["e", "e"]):
        with pytest.raises(KeyError):
            c.open_all(bad)
    assert "e" not in c.slot_of and c.open_all([]) == []
    c.close("b")
    assert c.open("e") == 1


def test_opening_several_compares_no_two_of_them():
    class Key:
        compared = 0

        def __init__(self, n):
            self.n = n

        def __hash__(self):
            return self.n

        def __eq__(self, other):
            Key.compared += 1
            return self.n == other.n

    c = cache.SequenceStateCache([{"s": cache.StateSpec((3,), torch.float32)}], "cpu", 300, 5)
    assert len(c.open_all([Key(n) for n in range(300)])) == 300 and Key.compared < 300
