"""GPU test of a prompt chunk's fused QKV epilogue with a 24-bit cache: waves of one sequence and of several, starts that are no multiple of
four positions, a ragged last block of rows.  The reference is the same model with the row kernel instead."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [[1500], [1030, 3, 1, 62, 65, 129, 7], [61] * 20, [255, 257, 1, 511, 130]])
@pytest.mark.parametrize("k_bits", [16, 24])
def test_fused_epilogue_equals_the_row_kernel(lengths, k_bits):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=1024, intermediate_size=1024, head_dim=128, num_attention_heads=16, num_key_value_heads=8)
    rng = np.random.default_rng(len(lengths) + k_bits)
    prompts = [rng.integers(0, cfg.vocab_size, n) for n in lengths]
    ids = list(range(len(lengths)))
    out = {}
    for fused in (0, 1):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
        m.set_option("kv_v_bits", 24)
        m.set_option("kv_k_bits", k_bits)
        m.set_option("tile_fuse_qk", fused)
        m.kv_alloc(sum((n + 3) // 256 + 1 for n in lengths), len(lengths), 1101)  # chunks of 1101 rows: the second one starts anywhere
        out[fused] = [m.step(ids, prompts, True, want_logits=True)[1]]
        out[fused].append(m.step(ids, [np.append(p, 5) for p in prompts], False, want_logits=True)[1])  # reads all that was written
        m.close()
    # the same values but for the order of a head's sum of squares: half a unit of what the cache keeps, 2^-17 with K in 24 bits (its
    # residual products are good to 2^-15), 2^-12 with K in 16
    bound = 2.0 ** (-14 if k_bits == 24 else -11)
    for a, b in zip(out[0], out[1]):
        assert np.abs(a - b).max() < bound * np.abs(a).max(), np.abs(a - b).max() / np.abs(a).max()
