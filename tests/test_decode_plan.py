"""The slices of 16-bit decode attention, read from the workspace that they need
(no device is touched)."""
import pytest

from triton_metal_amd import _lib


def slices(B, Hkv, rep, D, S, page):
    n = _lib.lib().tm_decode_attention_full_workspace_size(B, Hkv * rep, Hkv, D, S, page)
    per = B * Hkv * rep * (D + 4) * 4
    assert n % per == 0
    return max(1, n // per)


def rounds(B, Hkv, rep, D, n):
    """Rounds of resident waves: 3 rings of a wave fill a CU's LDS, 6 up to D = 64."""
    return -(-B * Hkv * -(-rep // 16) * n // (256 * (6 if D <= 64 else 3)))


@pytest.mark.parametrize("B,Hkv,rep,D,S,page,want", [
    (16, 8, 4, 128, 8192, 0, 6), (17, 8, 4, 64, 16384, 0, 11), (28, 4, 4, 64, 9000, 0, 13),
    (32, 8, 8, 128, 4096, 64, 3), (8, 8, 4, 128, 8192, 16, 12)])
def test_full_sequences_take_one_round(B, Hkv, rep, D, S, page, want):
    """Lengths are not known on the host: no count that starts a second round when
    every sequence is full where one round takes them all."""
    n = slices(B, Hkv, rep, D, S, page)
    assert n == want and rounds(B, Hkv, rep, D, n) == 1
