"""cs1_gemm_tune on operands that the own kernel cannot load (off a 16-byte address) re-chooses hipBLASLt's
kernel for such calls and leaves the shape's plan for aligned operands as it was."""
import ctypes

import numpy as np
import pytest

import oracle as O
from gpu_helpers import dev, empty, get_bf16, say, stream
from qwen3_5_native import hip

pytestmark = pytest.mark.gpu


def test_tune_on_unaligned_operands_keeps_the_plan():
    api, st = hip.api(), stream()
    M, N, K = 70, 136, 256
    say(f"gemm tune off 16 bytes M={M} N={N} K={K}")
    rng = np.random.default_rng(3)
    x = dev(O.f32_to_bf16(rng.standard_normal(M * K + 8).astype(np.float32)))
    w = dev(O.f32_to_bf16((rng.standard_normal(N * K) * 0.05).astype(np.float32)))
    h = api.cs1_gemm_create(32 << 20)
    assert h

    def plan():
        tile, split = ctypes.c_int(), ctypes.c_int()
        hip.check(api.q35_gemm_plan_of(h, M, N, K, N, tile, split), "plan")
        return tile.value, split.value

    def aligned():
        y = empty(M * N * 2)
        hip.check(api.cs1_gemm(h, x.at(0), w.at(0), y.at(0), M, N, K, N, st.handle), "gemm")
        return get_bf16(y, M * N)

    try:
        before, want = plan(), aligned()
        assert before[0] >= 0  # the own kernel runs the shape
        y = empty(M * N * 2)
        hip.check(api.cs1_gemm_tune(h, x.at(8), w.at(0), y.at(0), M, N, K, N, st.handle), "tune")
        assert plan() == before
        np.testing.assert_array_equal(aligned(), want)
        hip.check(api.cs1_gemm_tune(h, x.at(0), w.at(0), y.at(0), M, N, K, N, st.handle), "tune aligned")
        tuned = get_bf16(y, M * N)
        np.testing.assert_array_equal(aligned(), tuned)
    finally:
        api.cs1_gemm_destroy(h)
