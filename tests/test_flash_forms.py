"""Where the wide flash form takes its blocks in turn, that comes out even whatever the order of the samples; elsewhere they are dealt by length."""
import random

import pytest

COLUMNS32, DEALT, IN_TURN = range(3)


def longest_share(lens, G, n):
    """What the workgroup with most has, of the mean: blocks of 256 columns in turn, back and forth, a sample's late ones first; a block's start
    and end take as long as a tile and a half of its keys."""
    cost = [3 + min(m, (i + 1) * 256 // G) // 32 for m in lens for i in reversed(range(-(-m * G // 256)))]
    had = [0] * n
    for p, c in enumerate(cost):
        r, i = divmod(p, n)
        had[n - 1 - i if r % 2 else i] += c
    return max(had) * n / sum(cost)


@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (16, 4), (16, 16), (32, 32), (16, 8), (64, 8), (8, 8)])
def test_in_turn_is_even(Hq, Hkv):
    from msa_amd import _lib
    lib, r, n = _lib.load(), random.Random(Hq + Hkv), 256 // Hkv
    form = lambda lens: lib.msa_diag_flash_form(len(lens), sum(lens), max(lens), Hq, Hkv, 256, 0)
    taken = 0
    for _ in range(6000):
        B = r.randint(1, 12)
        top = r.randint(200, 9000)
        lens = [top] * B if r.random() < 0.6 else [r.randint(int(0.6 * top), top) for _ in range(B)]
        if form(lens) == IN_TURN:
            taken += 1
            assert longest_share(lens, Hq // Hkv, n) <= 1.2, lens
    assert taken > 20


@pytest.mark.parametrize("lens,Hq,Hkv,form", [([8192], 16, 16, IN_TURN), ([2048] * 4, 16, 16, IN_TURN), ([1024] * 8, 32, 8, IN_TURN), ([3000, 5000], 16, 4, DEALT),
                                              ([1780, 2200], 32, 8, DEALT), ([2200, 1780], 32, 8, DEALT), ([3950, 3950], 16, 4, DEALT), ([1344] * 3, 32, 8, DEALT),
                                              ([4000, 2500, 3000, 3500] * 4, 32, 8, DEALT), ([1000], 32, 8, COLUMNS32), ([3500, 2160], 32, 8, COLUMNS32)])
def test_forms(lens, Hq, Hkv, form):
    from msa_amd import _lib
    assert _lib.load().msa_diag_flash_form(len(lens), sum(lens), max(lens), Hq, Hkv, 256, 0) == form


@pytest.mark.parametrize("lens,Hq,Hkv,hint,plain", [([4096], 32, 8, IN_TURN, IN_TURN), ([64] * 200, 32, 8, IN_TURN, IN_TURN), ([16] * 1000, 32, 8, IN_TURN, IN_TURN),
                                                    ([1024] * 4, 32, 8, IN_TURN, DEALT), ([3000] * 3, 32, 8, DEALT, DEALT), ([3950] * 2, 16, 4, DEALT, DEALT),
                                                    ([3000, 5000], 16, 4, DEALT, DEALT), ([3000, 1000], 32, 8, COLUMNS32, DEALT), ([1000], 32, 8, COLUMNS32, COLUMNS32)])
def test_promised_forms(lens, Hq, Hkv, hint, plain):
    from msa_amd import _lib
    form = lambda top: _lib.load().msa_diag_flash_form(len(lens), sum(lens), top, Hq, Hkv, 256, 1)
    assert form(max(lens)) == hint and form(0) == plain
