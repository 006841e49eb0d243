"""cs1_gemm's own kernel at the edges of its tiles: every tile form, forced, unsplit and split (the second
pass), with rows and columns past the last whole tile, fewer k steps than the ring has stages, as
many and more, and more tiles than CUs; default plans of ragged shapes; a strided output; and what
the kernel does not take (K not a multiple of 64, N not of 8, operands off 16 bytes), which hipBLASLt
still runs."""
import ctypes

import numpy as np
import pytest

import oracle as O
from gpu_helpers import dev, get_bf16, say, stream
from qwen3_5_native import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gemm():
    stream()
    h = hip.api().cs1_gemm_create(32 << 20)
    assert h
    yield h
    hip.api().cs1_gemm_destroy(h)


def check(h, M, N, K, ldy=None, off=0):
    """Against the float64 product rounded once. A float32 sum of K products, in any order, is within
    K 2^-24 sum |x w| of it, and the bf16 rounding adds 2^-8 of the value."""
    ldy = ldy or N
    say(f"gemm M={M} N={N} K={K} ldy={ldy} offset={off}")
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    x = O.f32_to_bf16(rng.standard_normal(M * K + off).astype(np.float32))
    w = O.f32_to_bf16((rng.standard_normal(N * K) * 0.02).astype(np.float32))
    fill = np.full(M * ldy, 0x7F7F, np.uint16)
    dx, dw = dev(x), dev(w)
    outs = []
    for _ in range(2):
        y = dev(fill)
        hip.check(hip.api().cs1_gemm(h, dx.at(2 * off), dw.at(0), y.at(0), M, N, K, ldy, stream().handle), "gemm")
        outs.append(get_bf16(y, M * ldy).reshape(M, ldy))
    np.testing.assert_array_equal(outs[0], outs[1])
    assert (outs[0][:, N:] == 0x7F7F).all()
    xf = O.bf16_to_f32(x)[off:].reshape(M, K).astype(np.float64)
    wf = O.bf16_to_f32(w).reshape(N, K).astype(np.float64)
    want = xf @ wf.T
    bound = 2.0 ** -8 * np.abs(want) + K * 2.0 ** -24 * (np.abs(xf) @ np.abs(wf).T) + 1e-30
    d = np.abs(O.bf16_to_f32(outs[0][:, :N]).astype(np.float64) - want)
    assert (d <= bound).all(), float((d / bound).max())


def plan(h, M, N, K):
    tile, split = ctypes.c_int(), ctypes.c_int()
    hip.check(hip.api().q35_gemm_plan_of(h, M, N, K, N, tile, split), "plan")
    return tile.value, split.value


@pytest.fixture
def force(gemm):
    """The handle with one form and split forced, which runs that form or refuses the shape."""
    def set_form(tile, split):
        hip.check(hip.api().q35_gemm_force(gemm, tile, split), "force")
        return gemm

    yield set_form
    hip.check(hip.api().q35_gemm_force(gemm, -2, 1), "force")


FORMS = 18


def form(tile):
    bm, bn, stages = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert hip.api().q35_gemm_form(tile, bm, bn, stages) == 0
    return bm.value, bn.value, stages.value


def test_there_are_no_more_forms():
    n = ctypes.c_int()
    assert hip.api().q35_gemm_form(FORMS, n, n, n) == hip.HIP_ERROR_INVALID_VALUE


@pytest.mark.parametrize("tile", range(FORMS))
def test_form_edges(force, tile):
    """One tile and a ragged neighbour in both directions, at every depth around the ring's."""
    h = force(tile, 1)
    bm, bn, stages = form(tile)
    for M, N, steps in [(1, 8, 1), (bm, bn, stages), (bm + 1, bn + 8, stages - 1), (2 * bm - 1, 2 * bn - 8, stages + 1),
                        (bm + 17, bn + 24, 2 * stages + 1)]:
        check(h, M, N, 64 * steps)


@pytest.mark.parametrize("tile", range(FORMS))
def test_form_split_edges(force, tile):
    """The second pass, with parts of unequal length and a ragged last tile in both directions."""
    bm, bn, stages = form(tile)
    for M, N, steps, split in [(3, 16, 2, 2), (bm + 1, bn + 8, 7, 3), (2 * bm - 3, 2 * bn - 16, 2 * stages + 3, 2),
                               (bm, bn, 25, 12)]:
        check(force(tile, split), M, N, 64 * steps)


@pytest.mark.parametrize("tile", range(FORMS))
def test_form_takes_tiles_in_turn(force, tile):
    """More tiles than CUs: a block of the forms that fill a CU takes several, its ring running on."""
    h = force(tile, 1)
    bm, bn, stages = form(tile)
    rows = 17 if bm >= 64 else 34
    check(h, rows * bm + 5, 600 // rows // 2 * bn + 8, 64 * (stages + 1))


def test_forced_forms_refuse_what_does_not_fit(force):
    x = dev(np.zeros(64 * 128, np.uint16))
    args = (x.at(0), x.at(0), x.at(0), 64, 64, 64, 64, stream().handle)
    assert hip.api().cs1_gemm(force(0, 2), *args) == hip.HIP_ERROR_INVALID_VALUE  # one step cannot be split
    assert hip.api().cs1_gemm(force(FORMS, 1), *args) == hip.HIP_ERROR_INVALID_VALUE


@pytest.mark.parametrize("M,N,K", [
    (1, 8, 64), (16, 152, 128), (63, 264, 192), (1, 1368, 832), (1, 11648, 64), (31, 11656, 320),
    (3, 5440, 64), (35, 6248, 128), (43, 12216, 64), (81, 1992, 64), (76, 2312, 448), (141, 2256, 64),
    (67, 11320, 128), (458, 3208, 64), (577, 6256, 64), (577, 6256, 192), (146, 3336, 64), (139, 5112, 64),
    (265, 5792, 192), (789, 7888, 64), (388, 3408, 192), (996, 8552, 320), (648, 12344, 128), (391, 11688, 64),
    (1029, 11176, 128), (2049, 9000, 192), (333, 2560, 2432),
])
def test_gemm_default_plans(gemm, M, N, K):
    assert plan(gemm, M, N, K)[0] >= 0
    check(gemm, M, N, K)


@pytest.mark.parametrize("M,N,K", [(107, 2560, 9728), (333, 2560, 9728), (250, 1000, 5120)])
def test_gemm_default_splits(gemm, M, N, K):
    assert plan(gemm, M, N, K)[1] > 1
    check(gemm, M, N, K)


@pytest.mark.parametrize("M,N,K,ldy,off", [
    (70, 136, 256, 208, 0),   # a column slice of a wider output
    (70, 136, 192, 140, 0),   # ldy not a multiple of 8
    (70, 132, 192, 132, 0),   # N not a multiple of 8
    (70, 136, 200, 136, 0),   # K not a multiple of 64
    (70, 136, 192, 136, 4),   # x off a 16-byte address
])
def test_gemm_layouts(gemm, M, N, K, ldy, off):
    check(gemm, M, N, K, ldy, off)


def test_gemm_without_workspace():
    """A handle without workspace: no split sums, every shape still runs."""
    stream()
    h = hip.api().cs1_gemm_create(0)
    assert h
    try:
        check(h, 107, 512, 4096)
    finally:
        hip.api().cs1_gemm_destroy(h)
