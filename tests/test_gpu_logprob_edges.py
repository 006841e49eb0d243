"""The log-probability kernel's single pass at the edges of its batches: a vocabulary of less than one
load per thread, of exactly one batch of all threads, of one 16-byte group more, and of several."""
import numpy as np
import pytest

from gpu_helpers import say, stream
import model_ref
from qwen3_5_native import model as QM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [8, 8184, 32768, 32776, 70008])
def test_logprobs_at_vocabulary_edges(vocab):
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
