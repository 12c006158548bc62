"""How the rows of a batch of short queries lie in the scan, over all batches and lengths that a call may have (on the host)."""
import ctypes as C


def test_row_packing_fits_its_form():
    from msa_amd import _lib
    lib = _lib.load()
    unit, by_units = C.c_int32(), C.c_int32()
    up = lambda n, m: -(-n // m) * m
    for B in [*range(1, 70), 100, 255, 256, 1000, 4096]:
        for S in [*range(1, 300), 511, 1000, 1024, 1025, 4000, 4090]:
            whole = B * up(S, 32)
            for gathers, chunks in ((0, 1), (1, 1), (0, 200_000), (1, 200_000), (0, 1_600_001)):
                assert lib.msa_diag_row_packing(B, S, chunks, gathers, C.addressof(unit), C.addressof(by_units)) == 0
                u, rows = unit.value, B * up(S, unit.value)
                if u == 32:
                    assert not by_units.value
                    continue
                assert rows < whole and whole > 64
                if by_units.value:             # fewer large tiles; the kernel's reciprocal of a query's units divides exactly
                    per, total = up(S, 8) // 8, up(up(rows, 32), 256) // 8
                    assert u == 8 and up(rows, 256) < up(whole, 256) and total < 1 << 21 and per * total < 1 << 32
                    magic = (1 << 32) // per + 1
                    assert per == 1 or all((n * magic) >> 32 == n // per for n in {0, per - 1, per, total // 2, total - 1, total // per * per - 1})
                else:                          # a smaller form; one unit of four rows is a whole query
                    assert rows <= (64 if whole <= 128 else 128) and (u == 8 or S <= 4)
                    assert not (gathers and whole > 128)       # (the small forms carry no gather)
