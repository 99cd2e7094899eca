"""The slices of 16-bit decode attention (no device is touched)."""
import ctypes
import math
import random

import pytest

from triton_metal_amd import _lib


def slices(B, Hkv, rep, D, S, page, lens=False):
    n, sl = ctypes.c_int(), ctypes.c_int()
    rc = _lib.lib().tm_decode_attention_plan(B, Hkv * rep, Hkv, D, S, page, int(lens),
                                             ctypes.byref(n), ctypes.byref(sl))
    assert rc == 0
    unit = page * 32 // math.gcd(page, 32) if page else 32
    assert sl.value % unit == 0 and (n.value - 1) * sl.value < S <= n.value * sl.value
    return n.value


def rounds(B, Hkv, rep, D, n):
    """Rounds of resident waves: 3 rings of a wave fill a CU's LDS, 6 up to D = 64."""
    return B * Hkv * -(-rep // 16) * n / (256 * (6 if D <= 64 else 3))


@pytest.mark.parametrize("B,Hkv,rep,D,S,page,want", [
    (16, 8, 4, 128, 8192, 0, 6), (17, 8, 4, 64, 16384, 0, 11), (28, 4, 4, 64, 9000, 0, 13),
    (32, 8, 8, 128, 4096, 64, 3), (8, 8, 4, 128, 8192, 16, 12)])
def test_full_sequences_take_one_round(B, Hkv, rep, D, S, page, want):
    """No count that starts a second round where one round takes all slices."""
    n = slices(B, Hkv, rep, D, S, page)
    assert n == want and rounds(B, Hkv, rep, D, n) <= 1


@pytest.mark.parametrize("B,Hkv,rep,D,S,page,most", [
    (16, 8, 4, 128, 8192, 16, 2), (17, 8, 4, 64, 16384, 0, 2), (32, 8, 8, 128, 4096, 64, 2),
    (23, 8, 4, 128, 8727, 0, 3), (8, 8, 4, 128, 16384, 16, 2), (4, 8, 4, 128, 32768, 16, 1)])
def test_own_lengths_fill_their_rounds(B, Hkv, rep, D, S, page, most):
    """Lengths are not known on the host: with seq_lens two or three rounds from 64 (sequence,
    KV head) pairs, filled when every sequence is full."""
    r = rounds(B, Hkv, rep, D, slices(B, Hkv, rep, D, S, page, lens=True))
    assert 0.93 * most < r <= most


@pytest.mark.parametrize("Hkv,rep,S,page,most", [
    (1, 8, 8192, 16, 32), (8, 4, 8192, 16, 32), (1, 8, 4096, 16, 32), (8, 4, 32768, 0, 96)])
@pytest.mark.parametrize("lens", [False, True])
def test_few_sequences_do_not_outgrow_the_combining_kernel(Hkv, rep, S, page, most, lens):
    """More than the 32 slices that are merged at once only where the slices save more
    than merging them one by one takes (64 of 8192 positions: 26.7 us, 32: 23.4)."""
    assert most // 2 < slices(1, Hkv, rep, 128, S, page, lens) <= most


def test_the_full_workspace_holds_both_plans():
    L = _lib.lib()
    for B, Hkv, rep, D, S, page in ((16, 8, 4, 128, 8192, 16), (1, 1, 8, 128, 4096, 0),
                                    (64, 4, 1, 64, 300, 5), (2, 2, 2, 80, 40, 0)):
        need = max(slices(B, Hkv, rep, D, S, page, lens) for lens in (False, True))
        per = B * Hkv * rep * (D + 4) * 4
        base = L.tm_decode_attention_workspace_size(B, Hkv * rep, Hkv, D, S, page)
        assert L.tm_decode_attention_full_workspace_size(B, Hkv * rep, Hkv, D, S, page) == max(
            base, per * need if need > 1 else 0)
    assert L.tm_decode_attention_plan(0, 8, 8, 64, 128, 0, 0, None, None) == _lib.TM_ERR_INVALID_ARG


@pytest.mark.parametrize("lens", [False, True])
def test_the_short_search_finds_what_the_whole_one_does(lens):
    """Launches plan too, so only some slice counts are looked at: over random calls
    never more than 8% above the least cost of all counts up to 256, 1% on average."""
    rng = random.Random(3)
    over = []
    for _ in range(400):
        B, Hkv = int(2 ** rng.uniform(0, 7)), rng.choice((1, 2, 4, 8, 16))
        rep, D = rng.choice((1, 4, 8, 32)), rng.choice((64, 128))
        S, page = int(2 ** rng.uniform(7, 17)), rng.choice((0, 0, 16, 48, 64, 256))
        unit = page * 32 // math.gcd(page, 32) if page else 32

        def cost(n):  # of slices of n units each
            sl = n * unit
            k = -(-S // sl)
            return ((math.ceil(rounds(B, Hkv, rep, D, k)) + 0.25 * lens) * (sl + 100)
                    + 75 * (k > 1) + (3.5 if page else 4.5) * k * (k > 32)), k

        every = {}
        for n in range(1, 257):
            sl = -(-(-(-S // n)) // unit)
            if n > 1 and sl * unit < 64:
                break
            c, k = cost(sl)
            every[k] = c
        over.append(every[slices(B, Hkv, rep, D, S, page, lens)] / min(every.values()) - 1)
    assert max(over) < 0.08 and sum(over) < 0.01 * len(over), (max(over), sum(over) / len(over))
