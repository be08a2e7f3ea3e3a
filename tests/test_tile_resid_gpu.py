"""GPU test of the products of a long prompt chunk that add the residual and prepare the next norm in their epilogue: row counts at the edges of
a block and of the rule, several prompts and chunks, both cache forms, against the same call with layer taps, which keeps slabs and norm launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


LAYERS = 3


def expected(hidden, rows, chunk):
    """o and down of all layers but the last, whose rows are few past its mixer, of every chunk of 128 workgroups of 32 rows"""
    parts = [chunk] * (rows // chunk) + [rows % chunk]
    return sum(2 * (LAYERS - 1) for r in parts if -(-r // 32) * (hidden // 128) >= 128)


# (hidden, heads, intermediate): K of 1024 and 2048 beside 3072 and 1152 (an odd number of 128)
@pytest.mark.parametrize("hidden,heads,inter", [(1024, 16, 3072), (1024, 8, 1152), (512, 8, 2048)])
@pytest.mark.parametrize("lens,chunk,bits", [([480], 4096, 16), ([481], 4096, 24), ([497], 4096, 16), ([992], 4096, 16), ([993], 4096, 16), ([700, 45], 4096, 24), ([1024], 4096, 16), ([1025], 4096, 16), ([1100, 3, 77], 4096, 24), ([2047], 4096, 16), ([2049], 4096, 16), ([1500, 1200, 1], 4096, 16),
                                             ([2400], 1100, 24), ([4000, 350], 8192, 16)])
def test_chunk(hidden, heads, inter, lens, chunk, bits):
    import nano_vllm_candle_amd as pkg

    cfg = pkg.Qwen3Config.tiny(vocab_size=2048, hidden_size=hidden, head_dim=128, num_hidden_layers=LAYERS, num_attention_heads=heads, num_key_value_heads=8, intermediate_size=inter)
    rng = np.random.default_rng(sum(lens))
    seqs = [rng.integers(0, cfg.vocab_size, n + 1).astype(np.uint32) for n in lens]
    ids, out = list(range(len(lens))), []
    for taps in (False, True):
        m = pkg.Qwen3ForCausalLM.from_synthetic(cfg, 3)
        if bits == 24:
            m.set_option("kv_v_bits", 24)
            m.set_option("kv_k_bits", 24)
        m.kv_alloc(sum(n // 256 + 2 for n in lens), len(lens), chunk)
        if taps:
            m.enable_taps()
        _, prompt = m.step(ids, [s[:-1] for s in seqs], True, want_logits=True)
        assert m.counter("tile_resid_launches") == (0 if taps else expected(hidden, sum(lens), chunk))
        if taps:
            m.enable_taps(False)
        _, after = m.step(ids, seqs, False, want_logits=True)
        out.append(np.concatenate([prompt, after]))
        m.close()
    # sums in another order, two 16-bit planes a product (2^-16), keys whose f16 may round the other way: 2^-11 of the largest logit, 2^-14 with the residuals
    assert np.abs(out[0] - out[1]).max() < 2.0 ** (-11 if bits == 16 else -14) * np.abs(out[1]).max()
