"""Which calls take the faster forms of products, embeddings and attention: a call outside what a form reads stays with the general one."""
import pytest
import torch

from msa_amd import seq_ops


@pytest.fixture
def anywhere(monkeypatch):
    monkeypatch.setattr(seq_ops, "_cuda", lambda *a: None)


def test_prefill_attention_of_other_types(anywhere):
    q, k = torch.zeros((600, 512)), torch.zeros((600, 512))
    batch = seq_ops.StepBatch([600], [0], [0], "cpu")
    ok = lambda q, k, v: seq_ops.takes_flash_rows(q, k, v, 4, 4, 128, 128, 0, batch)
    assert ok(q.bfloat16(), k.bfloat16(), k.bfloat16())
    for a, b, c in ((q, k, k), (q.half(), k.half(), k.half()), (q.bfloat16(), k, k), (q.bfloat16(), k.bfloat16(), k)):
        assert not ok(a, b, c)                # (the general kernel refuses them)
