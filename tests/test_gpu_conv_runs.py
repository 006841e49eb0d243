"""The causal conv's run lengths (8, 16 and 32 tokens a thread, chosen by how the launch fills the
chip) and the shorter last runs, at their edges: whole runs, one row more and one less, fewer rows
than the window. Every form equals the any-shape kernel, which a misaligned input takes, bit for bit."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import dev, empty, get_bf16, say, stream
from qwen3_5_native import hip

pytestmark = pytest.mark.gpu


def conv(src, at, ld, w, key_dim, value_dim, T):
    q, k, v = empty(T * key_dim * 2), empty(T * key_dim * 2), empty(T * value_dim * 2)
    hip.check(hip.api().cs1_gdn_conv(src.at(at * 2), ld, w.at(0), q.at(0), k.at(0), v.at(0), T, key_dim, value_dim,
                                     stream().handle), "conv")
    return [get_bf16(q, T * key_dim), get_bf16(k, T * key_dim), get_bf16(v, T * value_dim)]


@pytest.mark.parametrize("T,key_dim,value_dim", [
    (1, 128, 256), (2, 128, 256), (4, 128, 256), (5, 128, 256), (7, 128, 256), (8, 128, 256), (9, 128, 256), (250, 2048, 6144),
    (1312, 2048, 6144), (1313, 2048, 6144), (1319, 2048, 6144), (1321, 2048, 6144),
    (3392, 2048, 6144), (3399, 2048, 6144), (3409, 2048, 6144)])
def test_every_run_length_equals_the_any_shape_kernel(T, key_dim, value_dim):
    say(f"conv runs T={T} key_dim={key_dim} value_dim={value_dim}")
    ld = 2 * key_dim + value_dim + 16
    x = O.f32_to_bf16(np.random.default_rng(T).standard_normal(T * ld).astype(np.float32))
    w = dev(O.f32_to_bf16((np.random.default_rng(1).standard_normal((2 * key_dim + value_dim) * 4) * 0.5).astype(np.float32)))
    got = conv(dev(x), 0, ld, w, key_dim, value_dim, T)
    want = conv(dev(np.concatenate([x[:1], x])), 1, ld, w, key_dim, value_dim, T)
    for g, e in zip(got, want):
        np.testing.assert_array_equal(g, e)


@pytest.mark.parametrize("lens", [[700, 33, 400], [1], [319, 320], [640, 1, 0, 900, 8]])
def test_packed_runs_equal_single_sequences(lens):
    key_dim, value_dim = 2048, 4096
    ld = 2 * key_dim + value_dim
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    say(f"conv packed runs {lens}")
    rng = np.random.default_rng(T)
    x = O.f32_to_bf16(rng.standard_normal(T * ld).astype(np.float32))
    w, src = dev(O.f32_to_bf16((rng.standard_normal(ld * 4) * 0.5).astype(np.float32))), dev(x)
    q, k, v = empty(T * key_dim * 2), empty(T * key_dim * 2), empty(T * value_dim * 2)
    hip.check(hip.api().cs1_gdn_conv_varlen(src.at(0), ld, w.at(0), q.at(0), k.at(0), v.at(0), cu.ctypes.data,
                                            len(lens), None, key_dim, value_dim, stream().handle), "conv varlen")
    got = [get_bf16(b, T * d).reshape(T, d) for b, d in ((q, key_dim), (k, key_dim), (v, value_dim))]
    for r0, L in zip(cu, lens):
        if L:
            for g, e in zip(got, conv(src, int(r0) * ld, ld, w, key_dim, value_dim, L)):
                np.testing.assert_array_equal(g[r0:r0 + L].ravel(), e)
