"""cs1_attn_prep with rotary tables on 16-byte addresses (vector loads) and off them (single values):
the same bytes, for every rotary width of a head, from no rotary dims to all of them."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import dev, empty, get_bf16, say, stream
from qwen3_5_native import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,Dh,Hq,Hk,half", [(1, 256, 1, 1, 32), (5, 256, 3, 1, 8), (37, 256, 4, 2, 128), (9, 128, 2, 2, 64),
                                             (33, 128, 5, 1, 24), (7, 256, 2, 1, 0), (7, 128, 0, 3, 16)])
def test_table_alignment_changes_nothing(T, Dh, Hq, Hk, half):
    say(f"attn_prep tables T={T} Dh={Dh} Hq={Hq} Hk={Hk} half={half}")
    ld = 2 * Hq * Dh + Hk * Dh
    rng = np.random.default_rng(T)
    row = dev(O.f32_to_bf16(rng.standard_normal(T * ld).astype(np.float32)))
    qw, kw = (dev(O.f32_to_bf16((rng.standard_normal(Dh) * 0.1).astype(np.float32))) for _ in range(2))
    tables = [np.asarray(t).ravel() for t in O.rotary_tables(np.arange(T, dtype=np.int64) * 3, half, 1e7)] if half else [np.zeros(8, np.uint16)] * 2
    got = []
    for off in (0, 1):
        cs, sn = [dev(np.concatenate([t[:off], t])) for t in tables]
        q, gate, k = empty(max(T * Hq * Dh * 2, 2)), empty(max(T * Hq * Dh * 2, 2)), empty(T * Hk * Dh * 2)
        hip.check(hip.api().cs1_attn_prep(row.at(0), row.at(2 * Hq * Dh * 2), ld, qw.at(0), kw.at(0),
                                          cs.at(off * 2), sn.at(off * 2), q.at(0), gate.at(0),
                                          k.at(0), T, Hq, Hk, Dh, half, 1e-6, stream().handle), "attn_prep")
        got.append([get_bf16(q, T * Hq * Dh), get_bf16(gate, T * Hq * Dh), get_bf16(k, T * Hk * Dh)])
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
    host = get_bf16(row, T * ld)
    if half:
        kr = np.concatenate([host[2 * Hq * Dh:], np.zeros(2 * Hq * Dh, np.uint16)])
        eq, eg, ek = O.attn_prep(host, kr, ld, get_bf16(qw, Dh), get_bf16(kw, Dh), *tables, T, Hq, Hk, Dh, half, 1e-6)
        np.testing.assert_array_equal(got[0][1], np.asarray(eg).ravel())
        for g, e in ((got[0][0], eq), (got[0][2], ek)):
            # an ulp of the normalised value, times two rounded rotary products (2 x 2^-8 of values up to ~4)
            d = np.abs(O.bf16_to_f32(g) - O.bf16_to_f32(np.asarray(e).ravel()))
            assert (d <= 2 * 2.0 ** -8 * np.maximum(np.abs(O.bf16_to_f32(np.asarray(e).ravel())), 1.0)).all()
