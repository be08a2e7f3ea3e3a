"""GPU test of the fused QKV product of short prompts (a workgroup is 16 rows of one head): row counts on both sides of its rule and ragged last
blocks, sequences that meet in a block, 16- and 24-bit caches.  The reference is the row kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 16 + 2 x 8 heads: 32 workgroups for every 16 rows, fused from 65 to 128 rows
@pytest.mark.parametrize("lengths", [[64], [65], [97], [128], [129], [31, 3, 50, 1], [16, 16, 48], [7] * 15])
@pytest.mark.parametrize("bits", [16, 24])
def test_fused_product_equals_the_row_kernel(lengths, bits):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(hidden_size=1024, intermediate_size=1024, head_dim=128, num_attention_heads=16, num_key_value_heads=8)
    rng = np.random.default_rng(len(lengths) + bits)
    prompts = [rng.integers(0, cfg.vocab_size, n) for n in lengths]
    ids = list(range(len(lengths)))
    out = {}
    for fused in (0, 1):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
        if bits == 24:
            m.set_option("kv_v_bits", 24)
            m.set_option("kv_k_bits", 24)
        m.set_option("tile_fuse_qk", fused)
        m.kv_alloc(2 * len(lengths) + 1, len(lengths), 512)
        out[fused] = [m.step(ids, prompts, True, want_logits=True)[1]]
        out[fused].append(m.step(ids, [np.append(p, 5) for p in prompts], False, want_logits=True)[1])  # reads all that was written
        m.close()
    # the same values but for the order of a head's sum of squares: 2^-17 with a 24-bit cache (its residual products are good to 2^-15),
    # 2^-12 of what a 16-bit one keeps where that rounds the other way
    bound = 2.0 ** (-14 if bits == 24 else -11)
    for a, b in zip(out[0], out[1]):
        assert np.abs(a - b).max() < bound * np.abs(a).max(), np.abs(a - b).max() / np.abs(a).max()
