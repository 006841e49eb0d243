"""The two block forms of the Dh 128 attention (32 rows in eight waves, 16 rows in four), chosen by how the
launch fills the device: both sides of each line of the rule, tile and group remainders, against the
emulated reference kernel; windows, packed and prefix launches repeat the single calls bit for bit,
and so does a prefill of growing length, whichever form each takes."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import bf16_errors, dev, empty, get, get_bf16, say, stream
from qwen3_5_native import hip

pytestmark = pytest.mark.gpu
D = 128


def draw(T, hq, hk):
    rng = np.random.default_rng(T + hq)
    return [O.f32_to_bf16(rng.standard_normal(T * h * D).astype(np.float32)) for h in (hq, hk, hk, hq)]


def one(q, k, v, gate, T, hq, hk, base=0):
    out, lse = empty(T * hq * D * 2), empty(hq * T * 4)
    bufs = [dev(x) for x in (q, k, v, gate)]
    hip.check(hip.api().cs1_attention_ex(bufs[0].at(0), bufs[1].at(0), bufs[2].at(0), hk * D, bufs[3].at(0), out.at(0),
                                         lse.at(0), T, hq, hk, D, D ** -0.5, base, stream().handle), "ex")
    return get_bf16(out, T * hq * D).reshape(T, hq, D), get(lse, np.float32, hq * T).reshape(hq, T)


@pytest.mark.parametrize("T,hq,hk", [
    (1, 4, 1), (15, 4, 1), (16, 8, 2), (17, 8, 1), (31, 16, 4), (33, 16, 4), (96, 4, 1), (97, 8, 2), (127, 16, 4),
    (129, 4, 1), (512, 32, 8), (513, 32, 8), (1024, 16, 4), (1025, 16, 4), (1279, 8, 2), (1281, 16, 4)])
def test_forms_match_the_emulator(T, hq, hk):
    say(f"attention key groups T={T} hq={hq} hk={hk}")
    q, k, v, gate = draw(T, hq, hk)
    out, lse = one(q, k, v, gate, T, hq, hk)
    emu, else_ = O.attention_emul(q, k, v, hk * D, gate, T, hq, hk, D, D ** -0.5, want_lse=True)
    mx, mean = bf16_errors(out, O.bf16_to_f32(emu))
    # the bars of the other attention tests: probabilities round to bf16 (2^-9 of values up to ~4)
    assert mx <= 2e-2 and mean <= 2e-3
    np.testing.assert_allclose(lse, else_, atol=1e-3, rtol=0)


@pytest.mark.parametrize("T", [1024, 1100, 1300])
def test_windows_take_the_form_of_the_whole(T):
    hq, hk = 16, 4
    say(f"attention key groups window T={T}")
    q, k, v, gate = draw(T, hq, hk)
    full = one(q, k, v, gate, T, hq, hk)
    for base in (64, 512, (T - 1) // 64 * 64):  # windows start at multiples of 64
        win = one(q, k, v, gate, T, hq, hk, base)
        np.testing.assert_array_equal(win[0][base:], full[0][base:])
        np.testing.assert_array_equal(win[1][:, base:], full[1][:, base:])


@pytest.mark.parametrize("P,lens", [(0, [1025, 17, 0, 1300, 1024]), (1024, [1, 0, 40, 300])])
def test_packed_launches_mix_the_forms(P, lens):
    hq, hk = 16, 4
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    say(f"attention key groups packed P={P} lens={lens}")
    q, k, v, gate = (x.reshape(T, -1) for x in draw(T, hq, hk))
    _, kp, vp, _ = (x.reshape(max(P, 1), -1)[:P] for x in draw(max(P, 1), hq, hk))
    out, lse = empty(T * hq * D * 2), empty(hq * T * 4)
    dq, dk, dv, dg = (dev(x.reshape(-1)) for x in (q, k, v, gate))
    api, st = hip.api(), stream()
    if P:
        dkp, dvp = dev(kp.reshape(-1)), dev(vp.reshape(-1))
        hip.check(api.cs1_attention_prefix_varlen(dq.at(0), dk.at(0), dv.at(0), hk * D, dkp.at(0), dvp.at(0), hk * D, P,
                                                  dg.at(0), out.at(0), lse.at(0), cu.ctypes.data, len(lens), hq, hk, D,
                                                  D ** -0.5, st.handle), "prefix varlen")
    else:
        hip.check(api.cs1_attention_varlen(dq.at(0), dk.at(0), dv.at(0), hk * D, dg.at(0), out.at(0), lse.at(0),
                                           cu.ctypes.data, len(lens), hq, hk, D, D ** -0.5, st.handle), "varlen")
    got, got_lse = get_bf16(out, T * hq * D).reshape(T, hq, D), get(lse, np.float32, hq * T).reshape(hq, T)
    for a, n in zip(cu, lens):
        if n == 0:
            continue
        pad = np.zeros((P, hq * D), np.uint16)
        seq = [np.concatenate([x, y[a:a + n]]).reshape(-1) for x, y in ((pad, q), (kp, k), (vp, v), (pad, gate))]
        w, wl = one(*seq, P + n, hq, hk, P)
        np.testing.assert_array_equal(got[a:a + n], w[P:])
        np.testing.assert_array_equal(got_lse[:, a:a + n], wl[:, P:])


@pytest.mark.parametrize("hq,hk,whole,lengths", [(16, 4, 4096, [64, 500, 1024, 2048, 3000]), (32, 8, 2100, [1, 700, 1900])])
def test_rows_do_not_depend_on_the_length(hq, hk, whole, lengths):
    """Row r of a causal pass sees keys 0 .. r, however many rows follow it."""
    say(f"attention growing lengths hq={hq} T={whole}")
    x = draw(whole, hq, hk)
    full = one(*x, whole, hq, hk)
    for T in lengths:
        part = one(*(a.reshape(whole, -1)[:T].reshape(-1) for a in x), T, hq, hk)
        np.testing.assert_array_equal(part[0], full[0][:T])
        np.testing.assert_array_equal(part[1], full[1][:, :T])


def test_packed_long_sequences_equal_single_calls():
    """Enough long sequences for blocks of 32 rows; alone each takes blocks of 16."""
    hq, hk, lens = 16, 4, [2048, 2001, 2100, 1500]
    say(f"attention packed long {lens}")
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    x = [a.reshape(T, -1) for a in draw(T, hq, hk)]
    q, k, v, gate = (dev(a.reshape(-1)) for a in x)
    out, lse = empty(T * hq * D * 2), empty(hq * T * 4)
    hip.check(hip.api().cs1_attention_varlen(q.at(0), k.at(0), v.at(0), hk * D, gate.at(0), out.at(0), lse.at(0),
                                             cu.ctypes.data, len(lens), hq, hk, D, D ** -0.5, stream().handle), "varlen")
    got, got_lse = get_bf16(out, T * hq * D).reshape(T, hq, D), get(lse, np.float32, hq * T).reshape(hq, T)
    for a, n in zip(cu, lens):
        want, wl = one(*(y[a:a + n].reshape(-1) for y in x), n, hq, hk)
        np.testing.assert_array_equal(got[a:a + n], want)
        np.testing.assert_array_equal(got_lse[:, a:a + n], wl)
