"""GPU test of the q/k norm, rotation and cache writes of prompts by 16 rows and head, against the same in the product's epilogue: row counts at
the edges of 16 rows, sequences that begin anywhere in them, both cache forms, deferred norms of one and of many groups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [16, 24])
@pytest.mark.parametrize("lens", [[1], [15], [17], [90, 27], [33, 1, 2, 300], [255, 257], [1040, 5]])
def test_prompt(lens, bits):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=2048, hidden_size=1024, head_dim=128, num_hidden_layers=2, num_attention_heads=16, num_key_value_heads=8, intermediate_size=3072)
    rng = np.random.default_rng(sum(lens))
    seqs = [rng.integers(0, cfg.vocab_size, n + 1).astype(np.uint32) for n in lens]
    out = []
    for fuse in (0, 1):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
        if bits == 24:
            m.set_option("kv_v_bits", 24)
            m.set_option("kv_k_bits", 24)
        m.set_option("tile_fuse_qk", fuse)
        m.kv_alloc(sum(n // 256 + 2 for n in lens), len(lens), 4096)
        _, prompt = m.step(list(range(len(lens))), [s[:-1] for s in seqs], True, want_logits=True)
        _, after = m.step(list(range(len(lens))), seqs, False, want_logits=True)
        out.append(np.concatenate([prompt, after]))
        m.close()
    # f32 sums in another order, keys and values whose f16 may round the other way: 2^-11 of the largest logit, 2^-14 with the residuals
    assert np.abs(out[0] - out[1]).max() < 2.0 ** (-11 if bits == 16 else -14) * np.abs(out[1]).max()
