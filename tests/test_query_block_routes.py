"""Calls of query blocks that state no keys: taken by the one-pass kernel from 16384 rows x KV heads on (zeros come back), by the split-key entry point
below, which refuses them, wherever the line lies for calls with keys."""
import pytest
import torch


class _Lib:
    def msa_attn_workspace_bytes(self, *a):
        return 256

    def msa_flash_attn_fit(self, *a):
        self.taken = "one pass"
        return 0

    def msa_sparse_attn(self, *a):
        self.taken = "splits"
        return 0


@pytest.fixture
def call(monkeypatch):
    from msa_amd import _lib, ops
    lib = _Lib()
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(ops, "_need_cuda", lambda *a: None)
    monkeypatch.setattr(ops, "_stream", lambda *a: 0)

    def run(rows, B, Hq, Hkv, keys, dtype=torch.bfloat16):
        q, k = torch.empty((rows, Hq, 128), dtype=dtype), torch.empty((1, Hkv, 128), dtype=dtype)
        ops.sparse_attn(q, k, k, torch.zeros(B, dtype=torch.int64), torch.zeros(B, dtype=torch.int32), keys, cu_q=torch.zeros(B + 1, dtype=torch.int32), max_sq=64)
        return lib.taken
    return run


@pytest.mark.parametrize("G", [1, 2, 4, 8])
@pytest.mark.parametrize("Hkv", [1, 8, 32])
def test_no_keys(call, G, Hkv):
    for rows in (16, 100, 511, 512, 513, 1000, 2047, 2048, 2049, 16383, 16384):
        for B in (1, 20, 200):
            for keys in (0, -1):
                assert call(rows, B, G * Hkv, Hkv, keys) == ("one pass" if rows * Hkv >= 16384 else "splits"), (rows, B, keys)


def test_with_keys(call):
    # rows x heads / 20 and 1.6 keys a tile of 128 columns over 260 keys, up to 128 tiles
    for rows, B, Hq, Hkv, line in ((64, 1, 32, 8, 387), (64, 4, 32, 8, 413), (82, 4, 8, 8, 343), (400, 1, 32, 8, 1066), (2048, 1, 8, 8, 1283), (16, 1, 8, 8, 278)):
        assert call(rows, B, Hq, Hkv, line) == "one pass" and call(rows, B, Hq, Hkv, line + 1) == "splits", (rows, B, Hq, Hkv)
    assert call(2048, 1, 16, 8, 1 << 20) == "one pass" and call(33, 17, 32, 8, 1 << 20) == "one pass"
    assert call(4096, 1, 32, 8, 100, torch.float32) == "splits"
