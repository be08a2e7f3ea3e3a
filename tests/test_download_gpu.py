"""GPU test of logits on their way to the caller: fewer bytes than one pinned slot, a last slot that is not full, one to four threads, more
chunks than slots.  The reference is the same rows fetched one by one, whose products other kernels sum in another order; the greedy ids, which
the device finds by itself, say that every row is whole, and the same step again gives the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_seqs,vocab,rows", [(1, 16, 1), (1, 70000, 1), (3, 100003, 3), (2, 262144, 2), (8, 151936, 7), (64, 100000, 64)])
def test_logits_through_the_slots(max_seqs, vocab, rows):
    import nano_vllm_candle_amd as pkg

    vocab = vocab // 16 * 16
    m = pkg.Qwen3ForCausalLM.from_synthetic(pkg.Qwen3Config.tiny(vocab_size=vocab), seed=1)
    m.kv_alloc(max_seqs, max_seqs, 64)
    rng = np.random.default_rng(0)
    prompts = [rng.integers(0, vocab, 5) for _ in range(rows)]
    ids = list(range(rows))
    nxt, together = m.step(ids, prompts, True, want_logits=True)
    alone = np.concatenate([m.step([i], [prompts[i]], False, want_logits=True)[1] for i in ids])
    assert np.isfinite(together).all() and np.abs(together).max() > 0
    # the rows of a smaller step come from other kernels: equal up to their rounding, far below the distance of two rows
    assert np.abs(together - alone).max() < 1e-3 * np.abs(alone).max()
    assert (nxt == together.shape[1] - 1 - together[:, ::-1].argmax(1)).all()
    again = m.step(ids, prompts, True, want_logits=True)
    assert np.array_equal(again[1], together) and np.array_equal(again[0], nxt)
