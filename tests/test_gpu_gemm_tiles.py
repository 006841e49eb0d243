"""cs1_gemm's own kernel at the edges of its tiles: every tile form that the plan can choose (the
shapes were picked for it), the second pass of split products, rows and columns past the last
whole tile, one to several k steps (fewer than the ring's stages and more), more tiles than
CUs, a strided output, and what the kernel does not take (K not a multiple of 64, N not of 8,
operands off 16 bytes), which hipBLASLt still runs."""
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


@pytest.mark.parametrize("M,N,K", [
    (1, 8, 64), (16, 152, 128), (63, 264, 192),         # 64 x 64, one to three steps
    (1, 1368, 832),                                      # 64 x 64 in two parts
    (1, 11648, 64), (31, 11656, 320),                    # 32 x 256
    (3, 5440, 64), (35, 6248, 128), (43, 12216, 64),     # 64 x 128, 64 x 192
    (81, 1992, 64), (76, 2312, 448),                     # 128 x 80
    (141, 2256, 64), (67, 11320, 128), (458, 3208, 64),  # 128 x 128, 128 x 160, 128 x 192
    (577, 6256, 64), (577, 6256, 192),                   # 128 x 256
    (146, 3336, 64), (139, 5112, 64), (265, 5792, 192),  # 192 x 128, 192 x 160, 192 x 192
    (789, 7888, 64), (388, 3408, 192), (996, 8552, 320),  # 192 x 256, 256 x 128, 256 x 144
    (648, 12344, 128), (391, 11688, 64), (1029, 11176, 128),  # 256 x 160, 256 x 192, 256 x 256
    (2049, 9000, 192),                                   # more tiles than CUs, ragged on both sides
    (107, 2560, 9728), (333, 2560, 2432), (250, 1000, 5120),  # split products
])
def test_gemm_tile_edges(gemm, M, N, K):
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
