"""fp32 attention rows of group sizes that no kernel has (3, 5, 6, 7 query heads a KV head) are refused whatever the number of rows, heads and splits."""
import pytest
import torch


@pytest.mark.parametrize("G", [3, 5, 6, 7])
@pytest.mark.parametrize("rows,Hkv,keys", [(1, 1, 40), (2, 8, 100), (8, 8, 192), (11, 8, 192), (16, 8, 100), (16, 8, 2000), (40, 8, 100), (5, 3, 700), (1, 8, 5000)])
def test_refused(G, rows, Hkv, keys):
    from msa_amd import _lib
    lib, Hq = _lib.load(), G * Hkv
    t = torch.zeros(1 << 10, dtype=torch.int64)
    p = (t.data_ptr() + 255) // 256 * 256                  # (nothing is read: the sizes alone decide)
    rc = lib.msa_sparse_attn(p, None, p, p, p, p, rows, rows, 1, keys, Hq, Hkv, 128, _lib.MSA_F32, 0.1, 1, p, p, 1 << 40, None)
    assert rc == -1 and b"group size" in lib.msa_last_error()
