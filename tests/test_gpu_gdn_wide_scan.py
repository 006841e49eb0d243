"""The scan with 64 value columns a block (chosen for packed sequences that need several rounds of narrower
blocks): the same bits as the one-half form, output and states, over chunk counts 0 to 5, one-row
sequences, shared and per-sequence initial states, and one long sequence."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import dev, empty, get, get_bf16, say, stream
from qwen3_5_native import hip

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("lens,h,hk,shared", [([64, 1, 0, 200, 129, 65, 320, 3], 6, 3, True), ([63, 64, 65], 2, 2, False),
                                              ([1], 4, 1, True), ([300, 17] * 8, 16, 8, False), ([1000], 3, 1, True)])
def test_four_halves_are_bit_identical(lens, h, hk, shared, forms):
    say(f"gdn wide scan lens={lens} h={h} hk={hk} shared={shared}")
    api, st = hip.api(), stream()
    n, cu = len(lens), np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(T + h)

    def bf(*shape):
        return dev(O.f32_to_bf16(rng.standard_normal(int(np.prod(shape))).astype(np.float32)))

    q, k, v = bf(T, hk, D), bf(T, hk, D), bf(T, h, D)
    beta = dev(O.f32_to_bf16(rng.random(T * h).astype(np.float32)))
    g = dev((-rng.random(T * h) * 0.2).astype(np.float32))
    s0 = dev((rng.standard_normal((1 if shared else n) * h * D * D) * 0.1).astype(np.float32))
    outs = []
    for halves in (1, 4):
        forms(scan_halves=halves)
        o, so = empty(T * h * D * 2), empty(n * h * D * D * 4)
        ws = empty(api.cs1_gdn_workspace_floats(64 * sum((x + 63) // 64 for x in lens), h) * 4)
        hip.check(api.cs1_gdn_prefill_varlen(q.at(0), k.at(0), v.at(0), g.at(0), beta.at(0), o.at(0), ws.at(0),
                                             cu.ctypes.data, n, h, hk, D ** -0.5, s0.at(0), 0 if shared else h * D * D,
                                             so.at(0), h * D * D, st.handle), "varlen")
        outs.append((get_bf16(o, T * h * D), get(so, np.float32, n * h * D * D)))
    np.testing.assert_array_equal(outs[0][0], outs[1][0])
    np.testing.assert_array_equal(outs[0][1], outs[1][1])
