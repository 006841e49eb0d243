"""The scan's block width for a set of packed sequences (a pure function, no GPU needed): the form that
measured fastest, also where few sequences of unlike length leave wide blocks waiting for the longest."""
import numpy as np
import pytest

from qwen3_5_native import hip


def halves(lens, heads, cus=256):
    chunks = np.array([(n + 63) // 64 for n in lens], np.int32)
    return hip.load().q35_gdn_scan_halves(chunks.ctypes.data, len(lens), heads, cus)


@pytest.mark.parametrize("lens,heads,want", [
    ([936], 48, 2), ([936], 32, 1), ([8192], 32, 1), ([107], 16, 1),            # one sequence
    ([160] * 8, 48, 4), ([40] * 32, 48, 4), ([16] * 64, 32, 4),                  # packed, of one length
    ([193, 219, 68, 219, 154, 163, 185, 119], 48, 4),
    ([1807, 755, 432, 4357, 1469], 16, 1), ([704, 1891, 705], 32, 2), ([73, 849, 667], 32, 2),
    ([3201, 520, 867], 32, 2), ([143, 1644, 1298], 16, 1), ([709, 233, 39], 32, 2),
    ([2429, 2320, 1057], 48, 4), ([2166, 2395, 1265, 2673, 832], 32, 4)])
def test_scan_form(lens, heads, want):
    assert halves(lens, heads) == want


def test_scan_form_ignores_empty_sequences():
    assert halves([0, 936, 0], 48) == halves([936], 48)


@pytest.mark.parametrize("cus", [1, 8, 304])
def test_scan_form_ends_on_any_device(cus):
    for lens in ([1], [1] * 64, [65536, 1], [64] * 64, [4096] + [1] * 63):
        for heads in (1, 48, 1024):
            assert halves(lens, heads, cus) in (1, 2, 4)
