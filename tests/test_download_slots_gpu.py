"""GPU test of logits on their way to the caller: one piece and less, pieces of one to four threads, more pieces than the pinned slots hold, an end that is not on 16 bytes,
arrays at odd places, again and again into the same slots.  The reference is the same rows a few at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,rows", [(256, 3), (32768, 8), (32784, 17), (32784, 40), (65552, 150)])
def test_every_row_arrives(vocab, rows):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=vocab, hidden_size=256, intermediate_size=256, num_hidden_layers=1, max_position_embeddings=256)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    m.kv_alloc(rows, rows, 1024)
    rng = np.random.default_rng(rows)
    seqs = [rng.integers(0, vocab, int(n)) for n in rng.integers(1, 9, rows)]
    ids = list(range(rows))
    m.step(ids, seqs, True)
    lists = [np.append(s, 5) for s in seqs]
    nxt, got = m.step(ids, lists, False, want_logits=True)
    assert np.array_equal(nxt, got.argmax(1))
    kept = got.copy()
    for _ in range(3):  # other answers in between
        m.step_score(ids, [np.append(s, 9) for s in seqs], False, [[len(s)] for s in seqs])
        assert np.array_equal(m.step(ids, lists, False, want_logits=True)[1], kept)
    assert np.array_equal(got, kept)
    for i in {0, rows // 2, rows - 1}:
        one = m.step([i], [lists[i]], False, want_logits=True)[1][0]
        # another kernel for one row: two 16-bit planes a product, 2^-15, one layer and the head
        assert np.abs(one - got[i]).max() < 2.0 ** -13 * np.abs(one).max()
    m.close()


@pytest.mark.parametrize("at", [1, 2, 3, 1021])  # floats behind the start of a page; what lies around stays
def test_arrays_at_odd_places(at):
    import ctypes as C

    import nano_vllm_candle_amd as pkg
    from nano_vllm_candle_amd import _lib

    cfg = pkg.Qwen3Config.tiny(vocab_size=32784, hidden_size=256, intermediate_size=256, num_hidden_layers=1, max_position_embeddings=256)
    rows, n = 17, 17 * 32784
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    m.kv_alloc(rows, rows, 1024)
    ids, seqs = list(range(rows)), [[5 + i, 9] for i in range(rows)]
    m.step(ids, [s[:1] for s in seqs], True)
    want_ids, want = m.step(ids, seqs, False, want_logits=True)
    memory = np.full(n + 4096, 7.0, np.float32)
    start = -memory.ctypes.data % 4096 // 4 + at
    next_ids = np.full(rows + 2, 77, np.uint32)
    u32p, seq_ids, ptrs, lens, _keep = m._step_args(ids, seqs)
    _lib.check(_lib.lib().nvllm_step(m.h, rows, seq_ids, ptrs, lens, 0, next_ids[1:].ctypes.data_as(u32p), memory[start:].ctypes.data_as(C.POINTER(C.c_float))), m.ctx.h)
    m.close()
    assert np.array_equal(memory[start:start + n].reshape(rows, -1), want) and np.array_equal(next_ids[1:-1], want_ids)
    assert (memory[:start] == 7).all() and (memory[start + n:] == 7).all() and next_ids[0] == next_ids[-1] == 77
