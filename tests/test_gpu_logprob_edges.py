"""The log-probability kernel's single pass over a row of logits, alone and in the runner: a vocabulary of less
than one load per thread, of exactly one batch of all threads, of one 16-byte group more, and of several;
rows whose value hangs on one group at an edge; infinities, NaN and the type's lowest value."""
import ctypes

import numpy as np
import pytest

import oracle as O
from gpu_helpers import dev, empty, get, say, stream
import model_ref
from qwen3_5_native import hip
from qwen3_5_native import model as QM

pytestmark = pytest.mark.gpu

VOCABS = [8, 8184, 32768, 32776, 70008]


def kernel(logits, targets):
    """logits [R, V] bfloat16 bits, targets [R] -> [R] float32."""
    R, V = logits.shape
    fn = QM.load().q35m_test_row_logprobs
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    x, t, out = dev(logits), dev(np.asarray(targets, np.int32)), empty(4 * R)
    hip.check(fn(x.at(0), V, t.at(0), R, out.at(0), stream().handle), "row logprobs")
    return get(out, np.float32, R)


def reference(logits, targets):
    x = O.bf16_to_f32(logits).astype(np.float64)
    m = x.max(1, keepdims=True)
    m = np.where(np.isneginf(m), 0.0, m)
    with np.errstate(divide="ignore", invalid="ignore", over="ignore"):
        return x[np.arange(len(x)), targets] - m[:, 0] - np.log(np.exp(x - m).sum(1))


def close(got, want, V):
    # The sum is of V float32 exponentials, V / 1024 of them in a row per thread, then 6 + 16 merges, each
    # within 2^-24 of exact and expf within 2 ulp: relative error e below, absolute in the logarithm; the
    # two subtractions round to float32.
    e = (V / 1024 + 22 + 4) * 2.0 ** -24
    bound = e + 2.0 ** -22 * (1 + np.abs(want))
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / bound).max())


@pytest.mark.parametrize("vocab", VOCABS)
def test_rows_that_hang_on_one_group(vocab):
    """Each row's weight lies in one value at an edge of the batches: a group that is dropped, read twice or read
    from the next row changes the result by more than 0.1 (the rows between lie 25 higher)."""
    say(f"logprob edge groups vocab={vocab}")
    edges = sorted({p for g in (0, 1023, 1024, 2047, 3 * 1024, 4 * 1024 - 1, 4 * 1024, 8 * 1024 - 1, vocab // 8 - 1)
                    for p in (8 * g, 8 * g + 7) if 0 <= p < vocab})
    rng = np.random.default_rng(vocab)
    x = rng.standard_normal((2 * len(edges), vocab)).astype(np.float32)
    for i, p in enumerate(edges):
        x[2 * i, p] = 14.0  # against a sum of about 1.6 vocab
        x[2 * i + 1] += 25.0
    x = O.f32_to_bf16(x.reshape(-1)).reshape(x.shape)
    targets = rng.integers(0, vocab, len(x))
    close(kernel(x, targets), reference(x, targets), vocab)


@pytest.mark.parametrize("vocab", VOCABS)
def test_infinities_and_extreme_values(vocab):
    say(f"logprob extremes vocab={vocab}")
    rng = np.random.default_rng(vocab + 1)
    x = np.tile(rng.standard_normal(vocab).astype(np.float32), (8, 1))
    x[0, :vocab - vocab // 4] = -np.inf     # -inf in all of most threads' first batches
    x[1, 1:] = -np.inf                      # one finite value, at the front
    x[2, :-1] = -np.inf                     # and at the end
    x[3] = -3.3895313892515355e38           # the type's lowest value
    x[4, ::2] = -3.3895313892515355e38
    x[5] = 3.3895313892515355e38
    x[6, vocab // 2] = np.nan
    x[7] = -np.inf
    x = O.f32_to_bf16(x.reshape(-1)).reshape(x.shape)
    targets = np.array([vocab - 1, 0, vocab - 1, 3, 1, 5, 0, 0])
    got, want = kernel(x, targets), reference(x, targets)
    close(got[:6], want[:6], vocab)
    assert np.isnan(got[6:]).all()


@pytest.mark.parametrize("vocab", VOCABS)
def test_logprobs_at_vocabulary_edges(vocab):
    """The whole call; what the edges of the batches hold is the tests' above."""
    stream()
    say(f"logprob edges vocab={vocab}")
    cfg = QM.Config(layers=4, hidden=256, intermediate=512, vocab=vocab, heads=4, kv_heads=1, lin_k_heads=2,
                    lin_v_heads=4, lm_head=1)
    m = QM.Model(cfg, seed=3, max_tokens=64)
    ids = np.random.default_rng(vocab).integers(0, vocab, 33)
    got, want = m.logprobs(ids), model_ref.logprobs(m, ids)
    m.close()
    d = np.abs(got - want)
    # logits are bf16 (steps of 2^-8 relative); the hidden states differ by GEMM accumulation order
    assert np.isfinite(got).all() and d.max() <= 5e-2 and d.mean() <= 5e-3, (d.max(), d.mean())
