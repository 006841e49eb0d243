"""cs1_attention_prefix_varlen at Dh 256, where a block's four 16-row groups may come from up to four
sequences or every sequence starts a block: one-row and empty sequences, group and tile remainders, a last block with unused
groups, more sequences than one launch takes, strided V. Every candidate equals its own windowed
call bit for bit, and rows of NaN in one candidate leave the others alone."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import dev, empty, get, get_bf16, say, stream
from qwen3_5_native import hip

pytestmark = pytest.mark.gpu
DH = 256


def packed(q, k, v, ldv, kp, vp, ldvp, P, gate, cu, hq, hk):
    T = int(cu[-1])
    out, lse = empty(T * hq * DH * 2), empty(hq * T * 4)
    bufs = [dev(x) for x in (q, k, v, kp, vp)] + [dev(gate) if gate is not None else None]
    hip.check(hip.api().cs1_attention_prefix_varlen(
        bufs[0].at(0), bufs[1].at(0), bufs[2].at(0), ldv, bufs[3].at(0), bufs[4].at(0), ldvp, P,
        bufs[5].at(0) if gate is not None else None, out.at(0), lse.at(0), cu.ctypes.data, len(cu) - 1, hq, hk, DH,
        DH ** -0.5, stream().handle), "prefix varlen")
    return get_bf16(out, T * hq * DH).reshape(T, hq, DH), get(lse, np.float32, hq * T).reshape(hq, T)


def window(q, k, v, kp, vp, P, gate, hq, hk):
    L = q.shape[0]
    W = P + L
    pad = np.zeros((P, hq, DH), np.uint16)
    bufs = [dev(np.concatenate([a, b])) for a, b in ((pad, q), (kp, k), (vp, v))]
    g = dev(np.concatenate([pad, gate])) if gate is not None else None
    out, lse = empty(W * hq * DH * 2), empty(hq * W * 4)
    hip.check(hip.api().cs1_attention_ex(bufs[0].at(0), bufs[1].at(0), bufs[2].at(0), hk * DH,
                                         g.at(0) if g is not None else None, out.at(0), lse.at(0), W, hq, hk, DH,
                                         DH ** -0.5, P, stream().handle), "window")
    return (get_bf16(out, W * hq * DH).reshape(W, hq, DH)[P:], get(lse, np.float32, hq * W).reshape(hq, W)[:, P:])


@pytest.mark.parametrize("hq,hk,P,gated,lens", [
    (24, 4, 64, True, [1]),
    (24, 4, 128, True, [1, 1, 1, 1, 1]),
    (16, 4, 64, False, [17, 0, 3, 16, 15, 33, 0]),
    (24, 4, 192, True, [0, 65, 64, 63, 1, 130, 2]),
    (8, 4, 64, True, [1 + (7 * i) % 19 for i in range(70)]),
    (2, 1, 256, True, [200, 31, 32]),
    # sequences that start a block each; kv heads that share XCDs, have one each, and do not divide them
    (16, 4, 64, True, [5, 5, 5]),
    (24, 4, 64, False, [16] * 16),
    (16, 8, 64, True, [70, 300, 1]),
    (4, 2, 128, True, [1000, 17]),
    (6, 3, 64, True, [129, 5, 0, 64]),
    (32, 16, 64, False, [90, 33]),
])
def test_packed_candidates_equal_windowed_calls(hq, hk, P, gated, lens):
    say(f"packed prefix attention hq={hq} hk={hk} P={P} lens={lens}")
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(T + P)

    def bf(*shape):
        return O.f32_to_bf16(rng.standard_normal(int(np.prod(shape))).astype(np.float32)).reshape(shape)

    q, k, v, gate = bf(T, hq, DH), bf(T, hk, DH), bf(T, hk, DH), bf(T, hq, DH) if gated else None
    kp, vp = bf(P, hk, DH), bf(P, hk, DH)
    # V as a column slice of wider rows
    wide, widep = bf(T, hk * DH + 64), bf(P, hk * DH + 8)
    wide[:, :hk * DH], widep[:, :hk * DH] = v.reshape(T, -1), vp.reshape(P, -1)
    got, lse = packed(q, k, wide, hk * DH + 64, kp, widep, hk * DH + 8, P, gate, cu, hq, hk)
    for i, L in enumerate(lens):
        if L:
            r = slice(int(cu[i]), int(cu[i + 1]))
            want, wl = window(q[r], k[r], v[r], kp, vp, P, gate[r] if gated else None, hq, hk)
            np.testing.assert_array_equal(got[r], want)
            np.testing.assert_array_equal(lse[:, r], wl)


def test_nan_rows_stay_in_their_candidate():
    hq, hk, P, lens = 8, 4, 64, [5, 40, 9]
    say(f"packed prefix attention with NaN rows, lens={lens}")
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    rng = np.random.default_rng(3)
    bf = lambda *s: O.f32_to_bf16(rng.standard_normal(int(np.prod(s))).astype(np.float32)).reshape(s)  # noqa: E731
    q, k, v, gate, kp, vp = bf(T, hq, DH), bf(T, hk, DH), bf(T, hk, DH), bf(T, hq, DH), bf(P, hk, DH), bf(P, hk, DH)
    clean, _ = packed(q, k, v, hk * DH, kp, vp, hk * DH, P, gate, cu, hq, hk)
    k2, v2 = k.copy(), v.copy()
    k2[5:45], v2[5:45] = 0x7FC0, 0x7FC0
    got, _ = packed(q, k2, v2, hk * DH, kp, vp, hk * DH, P, gate, cu, hq, hk)
    for r in (slice(0, 5), slice(45, 54)):
        np.testing.assert_array_equal(got[r], clean[r])
    assert np.isnan(O.bf16_to_f32(got[5:45])).any()


@pytest.mark.parametrize("T,hq,hk", [(1, 2, 1), (16, 16, 4), (63, 4, 2), (64, 16, 4), (65, 24, 4), (128, 8, 4), (129, 6, 1), (192, 2, 1)])
def test_one_to_three_tiles_match_the_emulator(T, hq, hk):
    """The first and the last step of a block, alone (one tile) and around whole steps."""
    say(f"attention Dh=256 T={T} hq={hq} hk={hk}")
    rng = np.random.default_rng(T)
    q, k, v, gate = (O.f32_to_bf16(rng.standard_normal(T * h * DH).astype(np.float32)) for h in (hq, hk, hk, hq))
    out, lse = empty(T * hq * DH * 2), empty(hq * T * 4)
    bufs = [dev(x) for x in (q, k, v, gate)]
    hip.check(hip.api().cs1_attention_ex(bufs[0].at(0), bufs[1].at(0), bufs[2].at(0), hk * DH, bufs[3].at(0), out.at(0),
                                         lse.at(0), T, hq, hk, DH, DH ** -0.5, 0, stream().handle), "ex")
    emu, else_ = O.attention_emul(q, k, v, hk * DH, gate, T, hq, hk, DH, DH ** -0.5, want_lse=True)
    d = np.abs(O.bf16_to_f32(get_bf16(out, T * hq * DH)) - O.bf16_to_f32(np.asarray(emu).ravel()))
    # the bars of the other attention tests: probabilities round to bf16 (2^-9 of values up to ~4)
    assert d.max() <= 2e-2 and d.mean() <= 2e-3
    np.testing.assert_allclose(get(lse, np.float32, hq * T).reshape(hq, T), else_, atol=1e-3, rtol=0)
