"""GPU test of decode attention in parts, merged by the part that ends last: as many parts as are merged at a time, one more and one less, rows of one part beside rows of
many, four and eight waves, 16 and 24 bits, heads of 64, query heads of more than one trip of the merge, and the counters of a step in the next one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,kv,heads,lens,bits", [
    (128, 8, 16, [895], 16), (128, 8, 16, [896], 16), (128, 8, 16, [1023], 16), (128, 8, 16, [1024], 16), (128, 8, 16, [2047], 16), (128, 8, 16, [2100], 16),  # 7 to 17 parts
    (128, 8, 16, [1, 127, 128, 513, 1500], 16), (128, 1, 16, [3, 600, 1030], 16), (128, 1, 16, [700, 2000], 24), (64, 2, 14, [40, 900, 1200], 16), (128, 2, 10, [5, 1300], 24)])
def test_parts(hd, kv, heads, lens, bits):
    import nano_vllm_candle_amd as pkg

    rows = len(lens)
    cfg = pkg.Qwen3Config.tiny(hidden_size=256, head_dim=hd, num_attention_heads=heads, num_key_value_heads=kv)
    m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
    if bits == 24:
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", 24)
    m.kv_alloc(sum(n // 256 + 1 for n in lens) + 9, rows + 1, 4096)
    rng = np.random.default_rng(rows + heads)
    seqs = [rng.integers(0, cfg.vocab_size, n + 1) for n in lens]
    for i in range(rows):
        m.step([i], [seqs[i][:-1]], True, want_logits=False)
    before = m.counter("merged_parts_launches")
    steps = [m.step(list(range(rows)), seqs, False, want_logits=True)[1] for _ in range(4)]
    assert m.counter("merged_parts_launches") - before == 4 * cfg.num_hidden_layers
    # whichever part merges, it takes them in their order
    assert all(np.array_equal(s.view(np.uint32), steps[0].view(np.uint32)) for s in steps)
    # the prompt's kernels sum in another order, from keys whose f16 may round the other way: 2^-11 of the largest logit, 2^-14 with the residuals
    bound = 2.0 ** (-11 if bits == 16 else -14)
    for i in range(rows):
        _, want = m.step([rows], [seqs[i]], True, want_logits=True)
        m.seq_free(rows)
        assert np.abs(steps[0][i] - want[0]).max() < bound * np.abs(want).max(), (i, lens[i])
    m.close()
