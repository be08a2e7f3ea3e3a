"""GPU test of what the wait for a step's logits costs the host: one thread waits, whatever their number that copies, and not all of a long step awake."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_one_thread_waits_for_a_long_step():
    import nano_vllm_candle_amd as pkg

    rows, vocab = 16, 65536  # 4.2 MB of logits: four threads copy
    cfg = pkg.Qwen3Config.tiny(vocab_size=vocab, hidden_size=4096, head_dim=128, num_attention_heads=32, num_key_value_heads=8, intermediate_size=12288, num_hidden_layers=10, max_position_embeddings=512)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    m.kv_alloc(rows, rows, 4096)
    rng = np.random.default_rng(0)
    seqs = [rng.integers(0, vocab, 256).astype(np.uint32) for _ in range(rows)]
    ids, last = list(range(rows)), [[255]] * rows
    for _ in range(2):
        m.step_score(ids, seqs, True, last)
    cpu, wall = time.process_time(), time.perf_counter()
    for _ in range(3):
        m.step_score(ids, seqs, True, last)
    cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    print(f"cpu {cpu * 1e3:.1f} ms, wall {wall * 1e3:.1f} ms")
    assert wall > 0.045  # a step is longer than the 10 ms that the wait stays awake for
    # the thread that enqueues and waits, the copies' threads for a part of a millisecond, the runtime's own; all four awake take more than three times the wall clock
    assert cpu < 1.6 * wall
    m.close()
