"""The causal conv's tokens per thread (a pure function, no GPU needed): by how the launch fills the device for
one sequence, and no runs of 32 for packed ones, whose last runs are shorter."""
import numpy as np
import pytest

from qwen3_5_native import hip


def run(lens, value_heads, packed=True, cus=256):
    starts = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    return hip.load().q35_conv_run(int(starts[-1]), len(lens) if packed else 0, starts.ctypes.data,
                                   (2 * 16 + value_heads) * 128, cus)


@pytest.mark.parametrize("T,value_heads,want", [(1, 48, 8), (64, 48, 8), (936, 48, 8), (3399, 48, 16), (4096, 32, 32)])
def test_one_sequence(T, value_heads, want):
    assert run([T], value_heads, packed=False) == want
    assert run([T], value_heads) in (want, 16)  # a packed call of one sequence


@pytest.mark.parametrize("lens,value_heads,want", [
    ([193, 219, 68, 219, 154, 163, 185, 119], 48, 8), ([40] * 32, 48, 8), ([255] * 8, 32, 8),
    ([320] * 8, 48, 16), ([1877] * 6, 32, 16), ([1151, 756, 1274], 48, 16), ([2351, 2870, 3352, 1243, 3332], 16, 16)])
def test_packed(lens, value_heads, want):
    assert run(lens, value_heads) == want


def test_empty_sequences():
    assert run([0, 0], 48) in (8, 16)
    assert run([0], 48, packed=False) in (8, 16, 32)
